"""The LDS-staged column and row products at the edges of their tiles against the FP64 oracle: one and many slabs per
block, slabs of odd and even numbers of 16-byte vectors, ends that no vector fills, one and several rounds of
outputs and contraction groups, unaligned bases, every storage type."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu
NARROW, K_LANES = 8, 10          # variants col_narrow, col_k_lanes

# I, K, O
SHAPES = [(2, 1, 1), (2, 2, 5), (3, 2, 4099), (3, 5, 1), (4, 16, 2049), (5, 7, 1200), (6, 4, 3001), (7, 129, 33),
          # rows: one and several lanes each, runs that end inside a word, one and many rounds, the longest
          (1, 2, 40000), (1, 3, 7), (1, 5, 9001), (1, 16, 3000), (1, 31, 1030), (1, 129, 700), (1, 255, 300), (1, 512, 64),
          (1, 1001, 37), (1, 1024, 9), (1, 2048, 6), (1, 4097, 5), (1, 8192, 4),
          (8, 2, 10000), (12, 341, 9), (16, 512, 3), (45, 13, 300), (64, 31, 40), (130, 63, 2), (1024, 8, 2), (4096, 2, 3)]


@pytest.mark.parametrize("I,K,Ox", SHAPES)
@pytest.mark.parametrize("dt", ["f32", "f64", "bf16", "fp8"])
def test_staged_products(ttvx, device, I, K, Ox, dt):
    import torch
    rng = np.random.default_rng(I * 1000 + K)
    x = rng.uniform(-1, 1, (Ox, K, I))
    b = rng.uniform(-1, 1, K)
    real = np.float64 if dt == "f64" else np.float32
    b = b.astype(real)
    bd = torch.from_numpy(b).to(device)
    scale = np.ones((Ox, I))
    ttvx.set_selection(ttvx.SELECT_FORCED, NARROW if I > 1 else K_LANES)
    try:
        for off in (0, 1):          # elements past a 16-byte boundary
            def place(values):
                buf = torch.empty(values.size + off, dtype=torch.from_numpy(values[:0].ravel()).dtype, device=device)
                buf[off:] = torch.from_numpy(values.ravel()).to(device)
                return buf[off:].view(Ox, K, I)
            if dt in ("f32", "f64"):
                v = x.astype(real)
                C = ttvx.ttv(2, place(v), bd)
                v = v.astype(np.float64)
            elif dt == "bf16":
                bits = O.bf16_rne(x.astype(np.float32).ravel())
                v = O.bf16_to_f32(bits).reshape(x.shape).astype(np.float64)
                C = ttvx.ttv_bf16(2, place(bits.view(np.int16).reshape(x.shape)).view(torch.uint16), bd,
                                  flags=ttvx.FLAG_KAHAN if off else 0)
            else:
                codes = rng.integers(0, 120, x.shape).astype(np.uint8)
                v = O.e4m3_decode(codes.ravel()).reshape(x.shape).astype(np.float64)
                fps = 3 if off else 1 + I // 2
                s = rng.uniform(0.5, 2, -(-Ox * I // fps)).astype(np.float32)
                scale = np.repeat(s.astype(np.float64), fps)[:Ox * I].reshape(Ox, I)
                C = ttvx.ttv_fp8(2, place(codes), torch.from_numpy(s).to(device), fps, bd)
            torch.cuda.synchronize()
            terms = v * b.astype(np.float64)[None, :, None]
            exact, mag = terms.sum(1) * scale, np.abs(terms).sum(1) * scale
            # any order of K products and sums, then one scaling: (K + 2) roundings of the magnitudes
            eps = 2.0 ** -53 if dt == "f64" else 2.0 ** -24
            assert np.all(np.abs(C.cpu().numpy().astype(np.float64) - exact) <= (K + 2) * eps * mag + 1e-300)
    finally:
        ttvx.restore_default_selection()


SPLIT_COL, SPLIT_DOT = 9, 4          # variants col_split, dot_split

# I, K, O: FP64 chunks of rows (one and several per block, split and unsplit, odd rows, few and many lane vectors);
# long rows (2 and 4 vectors per lane, 1, 2 and 4 waves along the row, odd numbers of rows, several pieces per wave)
LONG = [(2, 20000, 3), (3, 11003, 5), (16, 4100, 1), (45, 900, 7), (64, 2100, 2), (255, 131, 9), (100, 3000, 2),
        (1024, 67, 3), (513, 300, 1), (7, 1 << 20, 1),
        (1, 1025, 3), (1, 2049, 6), (1, 2500, 1001), (1, 4096, 37), (1, 5003, 258), (1, 16385, 5), (1, 100003, 3),
        (1, 300001, 64)]


@pytest.mark.parametrize("I,K,Ox", LONG)
@pytest.mark.parametrize("dt", ["f32", "f64", "bf16", "fp8"])
def test_long_contractions(ttvx, device, I, K, Ox, dt):
    import torch
    rng = np.random.default_rng(I * 7 + K)
    x = rng.uniform(-1, 1, (Ox, K, I)).astype(np.float64 if dt == "f64" else np.float32)
    b = rng.uniform(-1, 1, K).astype(x.dtype)
    bd = torch.from_numpy(b).to(device)
    scale = np.ones((Ox, I))
    ttvx.set_selection(ttvx.SELECT_FORCED, SPLIT_COL if I > 1 else SPLIT_DOT)
    try:
        for off, flags in ((0, 0), (1, 0), (0, ttvx.FLAG_FP64_FINAL)):
            if flags and I > 1:
                continue        # not every one of these shapes splits, and the rule's FP8 pick has no FP64 partial sums
            def place(values):
                buf = torch.empty(values.size + off, dtype=torch.from_numpy(values[:0].ravel()).dtype, device=device)
                buf[off:] = torch.from_numpy(values.ravel()).to(device)
                return buf[off:].view(Ox, K, I)
            if dt in ("f32", "f64"):
                v = x.astype(np.float64)
                C = ttvx.ttv(2, place(x), bd, flags=flags)
            elif dt == "bf16":
                bits = O.bf16_rne(x.ravel())
                v = O.bf16_to_f32(bits).reshape(x.shape).astype(np.float64)
                C = ttvx.ttv_bf16(2, place(bits.view(np.int16).reshape(x.shape)).view(torch.uint16), bd,
                                  flags=flags | (ttvx.FLAG_KAHAN if off else 0))
            else:
                codes = rng.integers(0, 120, x.shape).astype(np.uint8)
                v = O.e4m3_decode(codes.ravel()).reshape(x.shape).astype(np.float64)
                fps = 1 + I // 2
                s = rng.uniform(0.5, 2, -(-Ox * I // fps)).astype(np.float32)
                scale = np.repeat(s.astype(np.float64), fps)[:Ox * I].reshape(Ox, I)
                C = ttvx.ttv_fp8(2, place(codes), torch.from_numpy(s).to(device), fps, bd, flags=flags)
            torch.cuda.synchronize()
            terms = v * b.astype(np.float64)[None, :, None]
            exact, mag = terms.sum(1) * scale, np.abs(terms).sum(1) * scale
            # no output sums more than K / 64 terms in one chain: far inside (K / 8 + 64) roundings of the magnitudes
            eps = 2.0 ** -53 if dt == "f64" else 2.0 ** -24
            assert np.all(np.abs(C.cpu().numpy().astype(np.float64) - exact) <= (K / 8 + 64) * eps * mag + 1e-300)
    finally:
        ttvx.restore_default_selection()


@pytest.mark.parametrize("I,K,Ox,variant", [(1, 50001, 40, SPLIT_DOT), (5, 1 << 18, 1, SPLIT_COL)])
def test_split_under_capture_without_a_buffer(ttvx, device, I, K, Ox, variant):
    """A capture on a stream that has no buffer for partial sums takes the unsplit kernel; every replay is right."""
    import torch
    A = torch.empty((Ox, K, I), device=device).uniform_(-1, 1)
    b = torch.empty(K, device=device).uniform_(-1, 1)
    exact = (A.double() * b.double().view(1, -1, 1)).sum(1)
    mag = (A.double() * b.double().view(1, -1, 1)).abs().sum(1)
    C = torch.empty((Ox, I), device=device)
    ttvx.set_selection(ttvx.SELECT_FORCED, variant)
    try:
        s = torch.cuda.Stream()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            ttvx.ttv(2, A, b, out=C)
        for _ in range(3):
            C.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            assert bool(((C.double() - exact).abs() <= (K / 8 + 64) * 2.0 ** -24 * mag).all())
    finally:
        ttvx.restore_default_selection()
