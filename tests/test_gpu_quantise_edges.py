"""The quantisers at the edges of their tiles, bit-exact against the oracle: group sizes around a wave's, a
block's and two passes' capacity, fibers that vectors, tiles and slabs cut unevenly, values that are not finite."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("na,pia,q,fps", [
    # rows (q fastest): a wave (<= 512 values), 256 and 1024 threads per group, two passes; uneven ends
    ([7, 3], [1, 2], 1, 1), ([512, 5], [1, 2], 1, 1), ([513, 5], [1, 2], 1, 1), ([61, 341], [1, 2], 1, None),
    ([4097, 6], [1, 2], 1, None), ([8193, 3], [1, 2], 1, None), ([32768, 2], [1, 2], 1, None),
    ([32769, 3], [1, 2], 1, None), ([300001, 2], [1, 2], 1, None),
    # columns: several vectors per thread (short contractions), one row of lanes, tiles of 1024 threads
    ([1029, 1, 9], [1, 2, 3], 2, None), ([4100, 2, 3], [1, 2, 3], 2, None), ([1023, 3, 5], [1, 2, 3], 2, None),
    ([1364, 3, 7], [1, 2, 3], 2, None), ([64, 7, 33], [1, 2, 3], 2, None), ([50, 129, 21], [1, 2, 3], 2, None),
    ([2, 9, 500], [1, 2, 3], 2, None), ([3, 200, 40], [1, 2, 3], 2, None), ([36, 1000, 3], [1, 2, 3], 2, None),
    ([48, 2, 3], [1, 2, 3], 2, 1), ([48, 5, 7], [1, 2, 3], 2, 3), ([12, 5, 7], [1, 2, 3], 2, 1000),
    # slabs narrower than a cache line, cut by groups and blocks
    ([2, 2, 5000], [1, 2, 3], 2, None), ([7, 100, 61], [1, 2, 3], 2, None), ([5, 3, 4001], [1, 2, 3], 2, None),
    ([31, 130, 9], [1, 2, 3], 2, None), ([6, 4, 900], [1, 2, 3], 2, 1), ([4, 1024, 11], [1, 2, 3], 2, None),
    # columns in two passes: long contractions over wide, narrow and odd rows
    ([68, 4096, 2], [1, 2, 3], 2, None), ([67, 2100, 2], [1, 2, 3], 2, None), ([3, 20001, 2], [1, 2, 3], 2, None),
])
def test_fp8_groups(ttvx, device, na, pia, q, fps):
    import torch
    rng = np.random.default_rng(5)
    wa = O.strides(na, pia)
    a = rng.standard_normal(O.span(na, wa)).astype(np.float32)
    a[rng.uniform(size=a.size) < 0.01] *= 100.0
    a[:: max(1, a.size // 7)] = 0.0
    A = torch.from_numpy(a).to(device).as_strided(na, wa)
    codes, scales, f = ttvx.quantize_fp8(q, A, fps)
    oc, osc = O.quantize_fp8(q, a, na, wa, pia, f)
    assert np.array_equal(scales.cpu().numpy(), osc)
    assert np.array_equal(codes.as_strided([a.size], [1]).cpu().numpy(), oc)


def test_fp8_zeros_infinities_and_nan(ttvx, device):
    """A zero group has scale 1; NaN codes keep their sign and do not reach the scale; an infinity's group
    scales to infinity, its finite values to zero."""
    import torch
    for na, q in (([8, 600], 2), ([600, 8], 1)):
        a = np.ones(na, np.float32)
        fibers = a if q == 2 else a.T
        fibers[0, :] = 0.0
        fibers[1, 5], fibers[1, 6] = np.array([0x7FC00001, 0xFFC00001], np.uint32).view(np.float32)
        fibers[2, 3] = -np.inf
        fibers[3, 1], fibers[3, 2] = -448.0, -0.0
        A = torch.from_numpy(np.ascontiguousarray(a)).to(device)
        codes, scales, _ = ttvx.quantize_fp8(q, A, 1)
        c = codes.cpu().numpy() if q == 2 else codes.cpu().numpy().T
        s = scales.cpu().numpy()
        assert s[0] == 1.0 and s[1] == np.float32(1.0) / np.float32(448.0) and np.isinf(s[2]) and s[3] == 1.0
        assert not c[0].any()
        assert c[1, 5] == 0x7F and c[1, 6] == 0xFF and c[1, 0] == 0x7E
        assert (c[2, 3] & 0x7F) == 0x7F and c[2, 0] == 0
        assert c[3, 1] == 0xFE and c[3, 2] == 0x80 and c[3, 0] == 0x38


@pytest.mark.parametrize("n", [1, 7, 8, 9, 2047, 2048, 2051])
def test_bf16_tails(ttvx, device, n):
    import torch
    x = np.random.default_rng(n).standard_normal(n + 1).astype(np.float32)
    x[:1] = np.nan
    for off in (0, 1):
        q = ttvx.quantize_bf16(torch.from_numpy(x).to(device)[off:off + n])
        assert np.array_equal(q.cpu().numpy().view(np.uint16), O.bf16_rne(x[off:off + n]))
