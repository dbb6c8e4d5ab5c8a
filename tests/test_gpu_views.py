"""Products on blocks of a larger tensor (free modes that do not fold to three dimensions) against the FP64
oracle: the unit-stride kernels at the edges of their vectors, waves and contraction groups, every storage
type, outputs with gaps, and the general kernel where nothing has unit stride."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

# (extents of the block, layout, modes)
SHAPES = [
    ([5, 3, 2, 4], [1, 2, 3, 4], (1, 2, 3, 4)),               # the smallest: rows and columns of a few elements
    ([16, 17, 3, 9], [4, 3, 2, 1], (1, 2, 3, 4)),
    ([33, 8, 7, 65], [2, 4, 1, 3], (1, 2, 3, 4)),             # contractions of 7 to 65: every remainder of the rounds
    ([2, 3, 5, 1031], [4, 3, 2, 1], (1, 4)),                  # rows of more than 64 vectors in FP32
    ([3, 2, 2, 40000], [4, 3, 2, 1], (4,)),                   # few long rows: a block each
    ([129, 2, 3000, 3], [1, 2, 3, 4], (3,)),                  # few columns, long contraction: groups along k
    ([64, 12, 70, 40], [1, 2, 3, 4], (1, 2, 3, 4)),           # enough outputs for several row sets per wave
    ([32, 40, 36, 40], [4, 3, 2, 1], (4, 1)),
]
EPS = 2.0 ** -24


def _block(a, na, pia, halo, device, dtype):
    """The values `a` (shape na) as the interior of a tensor `halo` larger on every side, in layout pia."""
    import torch
    outer = [n + 2 * halo for n in na]
    buf = torch.full((int(np.prod(outer)),), float("nan") if dtype.is_floating_point else 255, dtype=dtype, device=device)
    view = buf.as_strided(outer, O.strides(outer, pia))
    for m, n in enumerate(na):
        view = view.narrow(m, halo, n)
    view.copy_(a)
    return view


def _check(got, exact, magnitude, eps):
    """|error| <= (K + 2) eps sum |a b|: the bound of any order of summation, one rounding for each term."""
    k, mag = magnitude
    assert np.all(np.abs(got.astype(np.float64) - exact) <= (k + 2) * eps * mag + 1e-300)


@pytest.mark.parametrize("na,pia,modes", SHAPES)
@pytest.mark.parametrize("dt", ["f32", "f64", "bf16", "fp8"])
def test_block_of_a_larger_tensor(ttvx, device, na, pia, modes, dt):
    import torch
    rng = np.random.default_rng(7)
    x = rng.uniform(-1, 1, na)
    for q in modes:
        b = rng.uniform(-1, 1, na[q - 1])
        if dt == "f64":
            a = torch.from_numpy(x).to(device)
            A, bd = _block(a, na, pia, 1, device, torch.float64), torch.from_numpy(b).to(device)
            C = ttvx.ttv(q, A, bd)
            xs = x
        else:
            bd = torch.from_numpy(b.astype(np.float32)).to(device)
            b = b.astype(np.float32).astype(np.float64)
            xf = x.astype(np.float32)
            if dt == "f32":
                A = _block(torch.from_numpy(xf).to(device), na, pia, 1, device, torch.float32)
                C = ttvx.ttv(q, A, bd)
                xs = xf.astype(np.float64)
            elif dt == "bf16":
                bits = O.bf16_rne(xf.ravel()).reshape(na)
                A = _block(torch.from_numpy(bits.view(np.int16)).to(device), na, pia, 3, device, torch.int16).view(torch.uint16)
                C = ttvx.ttv_bf16(q, A, bd, flags=ttvx.FLAG_KAHAN if q == modes[0] else 0)
                xs = O.bf16_to_f32(bits.ravel()).reshape(na).astype(np.float64)
            else:
                codes = rng.integers(0, 120, na).astype(np.uint8)
                A = _block(torch.from_numpy(codes).to(device), na, pia, 3, device, torch.uint8)
                fps, outputs = 3, int(np.prod(na)) // na[q - 1]
                scales = rng.uniform(0.5, 2, -(-outputs // fps)).astype(np.float32)
                C = ttvx.ttv_fp8(q, A, torch.from_numpy(scales).to(device), fps, bd)
                xs = O.e4m3_decode(codes.ravel()).reshape(na).astype(np.float64)
        shape = [1] * len(na)
        shape[q - 1] = -1
        terms = xs * b.reshape(shape)
        exact, mag = terms.sum(q - 1), np.abs(terms).sum(q - 1)
        if dt == "fp8":
            # fibers are numbered in C's layout order
            pic = O.output_layout(pia, q)
            order = [m - 1 for m in reversed(pic)]
            spread = np.repeat(scales.astype(np.float64), fps)[:outputs].reshape([exact.shape[m] for m in order])
            spread = spread.transpose(np.argsort(order))
            exact, mag = exact * spread, mag * spread
        torch.cuda.synchronize()
        _check(C.cpu().numpy(), exact, (na[q - 1], mag), 2.0 ** -53 if dt == "f64" else EPS)


def test_output_with_gaps_and_no_unit_stride(ttvx, device):
    import torch
    rng = np.random.default_rng(8)
    na = [6, 5, 7, 9]
    x = rng.uniform(-1, 1, na).astype(np.float32)
    b = rng.uniform(-1, 1, 5).astype(np.float32)
    A = _block(torch.from_numpy(x).to(device), na, [4, 3, 2, 1], 2, device, torch.float32)
    buf = torch.full((6, 7, 20), -3.0, device=device)
    ttvx.ttv(2, A, torch.from_numpy(b).to(device), out=buf[:, :, 1:10])
    torch.cuda.synchronize()
    terms = x.astype(np.float64) * b.astype(np.float64).reshape(1, 5, 1, 1)
    _check(buf[:, :, 1:10].cpu().numpy(), terms.sum(1), (5, np.abs(terms).sum(1)), EPS)
    rest = buf.clone()
    rest[:, :, 1:10] = -3.0
    assert bool((rest == -3.0).all())
    # every other element of each mode: the general kernel
    y = rng.uniform(-1, 1, [12, 10, 14]).astype(np.float32)
    Y = torch.from_numpy(y).to(device)[::2, ::2, ::2]
    C = ttvx.ttv(2, Y, torch.from_numpy(b).to(device))
    torch.cuda.synchronize()
    terms = y[::2, ::2, ::2].astype(np.float64) * b.astype(np.float64).reshape(1, 5, 1)
    _check(C.cpu().numpy(), terms.sum(1), (5, np.abs(terms).sum(1)), EPS)
