"""The work that users of this library give it, as cases that can be timed and compared.

A case is a dict of plain values.  Its "kind" says which public entry points a pass goes through:

* ``product``  -- ``ttv`` / ``ttv_bf16`` / ``ttv_fp8`` on a dense tensor, over one mode, or over every mode
                  in turn (``q`` 0, as the power method and the Tucker sweeps do)
* ``view``     -- ``ttv`` on a tensor that is a block inside a larger one (the interior of a grid with
                  ghost cells, a window of a longer series), so that its strides have gaps
* ``quantise`` -- ``quantize_fp8`` / ``quantize_bf16``: FP32 to the reduced storage that products read
* ``chain``    -- ``ttvs``: every mode but q contracted
* ``batch``    -- ``Batch``: many products of different shapes in a few launches

Extents are texts like "128x128x64", layouts list the modes from the fastest to the slowest ("1,2,3" is
first-order).  Every value is made from the seed on the GPU.
"""
import math
import random

import torch

import ttv_amd
from ttv_amd.batch import Batch

_DEVICE = "cuda"
_BYTES = {"f32": 4, "f64": 8, "bf16": 2, "fp8": 1}


# ---- cases ------------------------------------------------------------------------------------

def _shape(na):
    return "x".join(str(n) for n in na)


def _order(pia):
    return ",".join(str(m) for m in pia)


def _product(na, q, pia, dtype, kahan=False):
    return {"kind": "product", "na": _shape(na), "q": q, "pia": _order(pia), "dtype": dtype, "kahan": kahan}


def _view(na, halo, q, pia, dtype):
    return {"kind": "view", "na": _shape(na), "halo": halo, "q": q, "pia": _order(pia), "dtype": dtype}


def _quantise(na, q, pia, dtype):
    return {"kind": "quantise", "na": _shape(na), "q": q, "pia": _order(pia), "dtype": dtype}


def _chain(na, q, pia, dtype, order):
    return {"kind": "chain", "na": _shape(na), "q": q, "pia": _order(pia), "dtype": dtype, "order": order}


def _batch(count, cap_log2, shapes):
    return {"kind": "batch", "count": count, "cap_log2": cap_log2, "shapes": shapes}


def listed():
    return [
        # a small dense product inside somebody's loop: what a call costs
        dict(_product([24, 36, 30], 2, [1, 2, 3], "f32"), name="small_f32"),
        # the reference's plain double-precision product (order 3, first-order, the middle mode)
        dict(_product([256, 256, 256], 2, [1, 2, 3], "f64"), name="cube_f64"),
        # the headline tensor, every mode in turn: rows, narrow columns and wide columns
        dict(_product([128] * 4, 0, [1, 2, 3, 4], "f32"), name="order4_all_modes_f32"),
        # high order with small extents: an output of a sixteenth of the input, short contractions
        dict(_product([16] * 7, 6, [7, 6, 5, 4, 3, 2, 1], "f32"), name="order7_f32"),
        # measured data with extents as they come (odd rows, some layout), every mode in turn
        dict(_product([101, 67, 95, 149], 0, [3, 1, 4, 2], "f32"), name="ragged_all_modes_f32"),
        # a few very long contractions (a long series against a handful of channels)
        dict(_product([7, 3, 4000037], 3, [3, 2, 1], "f32"), name="long_rows_f32"),
        # the interior of a grid with ghost cells, every mode in turn
        dict(_view([96, 90, 84, 80], 2, 0, [4, 3, 2, 1], "f32"), name="interior_all_modes_f32"),
        # bfloat16 storage with odd extents, every mode in turn
        dict(_product([255, 129, 131, 61], 0, [1, 2, 3, 4], "bf16"), name="ragged_all_modes_bf16"),
        # FP8 storage of a large tensor of high order, contracted over its long mode
        dict(_product([4096, 4, 8, 4, 8, 4, 2, 64], 1, [5, 2, 8, 1, 7, 3, 6, 4], "fp8"), name="order8_fp8"),
        # a large tensor on its way into FP8 storage
        dict(_quantise([128] * 4, 2, [1, 2, 3, 4], "fp8"), name="quantise_fp8"),
        # all modes but one contracted (one step of a rank-one approximation)
        dict(_chain([44, 40, 36, 38, 42], 3, [5, 4, 3, 2, 1], "f32", "optimal"), name="chain_order5_f32"),
        # many products of uneven shape in one call
        dict(_batch(48, 26, 7), name="batch_f32"),
    ]


def _extents(rng, p, size):
    """p extents of at least 2 whose product is about `size`, uneven and seldom round."""
    w = [rng.gammavariate(2.0, 1.0) + 0.05 for _ in range(p)]
    na = [max(2, round(size ** (x / sum(w)))) for x in w]
    while math.prod(na) > size:
        m = max(range(p), key=lambda r: na[r])
        if na[m] == 2:
            break
        na[m] = max(2, int(na[m] * size / math.prod(na)))
    return na


def _layout(rng, p):
    r = rng.random()
    if r < 0.35:
        return list(range(1, p + 1))
    if r < 0.7:
        return list(range(p, 0, -1))
    return rng.sample(range(1, p + 1), p)


def draw(rng):
    """One more case: sizes spread over the logarithm of 2^14 .. 2^28 elements."""
    size = int(2.0 ** rng.uniform(14, 28))
    r = rng.random()
    if r < 0.50:
        p = rng.randint(2, 7)
        na = _extents(rng, p, size) if rng.random() < 0.7 else [max(2, round(size ** (1 / p) - 0.5))] * p
        dtype = rng.choice(["f32", "f32", "bf16", "fp8", "f64"])
        q = rng.randint(1, p) if size > 1 << 25 else rng.choice([0, rng.randint(1, p)])
        return _product(na, q, _layout(rng, p), dtype, dtype in ("bf16", "fp8") and rng.random() < 0.2)
    if r < 0.60:
        # a long mode against a few free elements
        p = rng.randint(2, 3)
        na = [rng.randint(2, 12) for _ in range(p)]
        q = rng.randint(1, p)
        na[q - 1] = max(1 << 12, size // math.prod(n for m, n in enumerate(na, 1) if m != q))
        return _product(na, q, _layout(rng, p), rng.choice(["f32", "f32", "bf16", "fp8", "f64"]))
    if r < 0.72:
        p = rng.randint(2, 5)
        na = [n + 2 for n in _extents(rng, p, max(1 << 14, size >> 2))]
        q = rng.randint(1, p) if size > 1 << 25 else rng.choice([0, rng.randint(1, p)])
        return _view(na, rng.randint(1, 3), q, _layout(rng, p),
                     rng.choice(["f32", "f32", "f64"]))
    if r < 0.84:
        p = rng.randint(2, 7)
        return _quantise(_extents(rng, p, size), rng.randint(1, p), _layout(rng, p), rng.choice(["fp8", "bf16"]))
    if r < 0.95:
        p = rng.randint(3, 6)
        return _chain(_extents(rng, p, size), rng.randint(1, p), _layout(rng, p), rng.choice(["f32", "f32", "f64"]),
                      rng.choice(["optimal", "optimal", "fused"]))
    return _batch(rng.randint(6, 40), rng.randint(20, 25), rng.randint(1, 1 << 20))


# ---- inputs -------------------------------------------------------------------------------------

def _numbers(text, sep):
    return [int(x) for x in text.split(sep)]


def _strides(na, pia):
    wa, step = [0] * len(na), 1
    for m in pia:
        wa[m - 1] = step
        step *= na[m - 1]
    return wa


def _modes(case):
    p = len(_numbers(case["na"], "x"))
    return list(range(1, p + 1)) if case["q"] == 0 else [case["q"]]


def _generator(seed):
    return torch.Generator(device=_DEVICE).manual_seed(seed)


def _uniform(g, n, dtype):
    return torch.empty(n, dtype=dtype, device=_DEVICE).uniform_(-1, 1, generator=g)


def _with_outliers(g, n):
    """N(0, 1) values, one in a hundred of them 100 times larger: what reduced storage meets."""
    x = torch.empty(n, dtype=torch.float32, device=_DEVICE).normal_(generator=g)
    at = torch.randint(0, n, (n // 100,), generator=g, device=_DEVICE)
    x[at] = x[at] * 100
    return x


def _real(case):
    return torch.float64 if case["dtype"] == "f64" else torch.float32


def _inputs(case, seed):
    """(A, {mode: vector}): A in FP64 or FP32 with its layout's strides, a vector for each mode."""
    g = _generator(seed)
    na, pia, dt = _numbers(case["na"], "x"), _numbers(case["pia"], ","), _real(case)
    if case["kind"] == "view":
        h = case["halo"]
        outer = [n + 2 * h for n in na]
        a = _uniform(g, math.prod(outer), dt).as_strided(outer, _strides(outer, pia))
        for m, n in enumerate(na):
            a = a.narrow(m, h, n)
    else:
        n = math.prod(na)
        a = _with_outliers(g, n) if case["dtype"] in ("bf16", "fp8") else _uniform(g, n, dt)
        a = a.as_strided(na, _strides(na, pia))
    return a, {m: _uniform(g, n, dt) for m, n in enumerate(na, 1)}


def _batch_shapes(case):
    """Order 3 or 4, extents 16 .. 512, at most 2^cap_log2 elements, any mode, any layout."""
    rng = random.Random(case["shapes"])
    out = []
    for _ in range(case["count"]):
        p = rng.choice([3, 4])
        while True:
            na = [rng.randint(16, 512) for _ in range(p)]
            if math.prod(na) <= 1 << case["cap_log2"]:
                break
        out.append((na, rng.randint(1, p), rng.sample(range(1, p + 1), p)))
    return out


def _batch_inputs(case, seed):
    g = _generator(seed)
    out = []
    for na, q, pia in _batch_shapes(case):
        a = _uniform(g, math.prod(na), torch.float32).as_strided(na, _strides(na, pia))
        out.append((q, a, _uniform(g, na[q - 1], torch.float32)))
    return out


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        return kind, Batch(_batch_inputs(case, seed)), None, None
    a, bs = _inputs(case, seed)
    if kind == "quantise":
        return kind, a, case["q"], case["dtype"]
    if kind == "chain":
        return kind, a, (case["q"], [b for m, b in bs.items() if m != case["q"]]), case["order"]
    calls = [(q, bs[q]) for q in _modes(case)]
    if case["dtype"] == "bf16":
        return "bf16", ttv_amd.quantize_bf16(a), calls, ttv_amd.FLAG_KAHAN if case["kahan"] else 0
    if case["dtype"] == "fp8":
        # the scales run along the contracted fibers, so every mode has its own codes
        return ("fp8", [ttv_amd.quantize_fp8(q, a) for q, _ in calls], calls,
                ttv_amd.FLAG_KAHAN if case["kahan"] else 0)
    return "plain", a, calls, None


def run(state):
    kind, a, calls, option = state
    if kind == "plain":
        return [ttv_amd.ttv(q, a, b) for q, b in calls]
    if kind == "bf16":
        return [ttv_amd.ttv_bf16(q, a, b, flags=option) for q, b in calls]
    if kind == "fp8":
        return [ttv_amd.ttv_fp8(q, codes, scales, fps, b, flags=option)
                for (codes, scales, fps), (q, b) in zip(a, calls)]
    if kind == "quantise":
        if option == "bf16":
            return ttv_amd.quantize_bf16(a).view(torch.int16)
        return list(ttv_amd.quantize_fp8(calls, a)[:2])
    if kind == "chain":
        return ttv_amd.ttvs(calls[0], a, calls[1], option)
    a.launch()
    return a.outputs


# ---- what a pass cannot do without, and its results in 64 bits -----------------------------------

def work(case):
    if case["kind"] == "batch":
        nbytes = flops = 0
        for na, q, _ in _batch_shapes(case):
            n = math.prod(na)
            nbytes += 4 * (n + n // na[q - 1] + na[q - 1])
            flops += 2 * n
        return {"bytes": nbytes, "flops": flops}
    na = _numbers(case["na"], "x")
    n, s = math.prod(na), _BYTES[case["dtype"]]
    if case["kind"] == "quantise":
        scales = -(-(n // na[case["q"] - 1]) // _fibers_per_scale(na[case["q"] - 1])) if s == 1 else 0
        return {"bytes": 4 * n + s * n + 4 * scales, "flops": 2 * n}
    acc = 8 if case["dtype"] == "f64" else 4
    if case["kind"] == "chain":
        return {"bytes": s * n + acc * sum(na), "flops": 2 * n}
    nbytes = flops = 0
    for q in _modes(case):
        k = na[q - 1]
        nbytes += s * n + acc * (n // k + k)
        if s == 1:
            nbytes += 4 * -(-(n // k) // _fibers_per_scale(k))
        flops += 2 * n
    return {"bytes": nbytes, "flops": flops}


def _fibers_per_scale(k):
    return max(1, -(-4096 // k))


def _contract(a, q, b, chunk=1 << 27):
    """A x_q b in 64 bits, in pieces along mode q (of at most `chunk` elements where a piece can be cut)."""
    k = a.shape[q - 1]
    per = max(1, chunk // max(1, a.numel() // k))
    shape = [1] * a.dim()
    shape[q - 1] = -1
    out = 0
    for k0 in range(0, k, per):
        kk = min(per, k - k0)
        out = out + (a.narrow(q - 1, k0, kk).double() * b[k0:k0 + kk].double().view(shape)).sum(q - 1)
    return out


def _fp8_scales(a, q, pia):
    """Largest magnitude of each scale group / 448, and the same spread over C's elements (C in its
    layout: the fastest free mode last)."""
    c = a.abs().amax(q - 1).permute([m - 1 if m < q else m - 2 for m in reversed(pia) if m != q])
    fps = _fibers_per_scale(a.shape[q - 1])
    flat = c.reshape(-1)
    groups = -(-flat.numel() // fps)
    flat = torch.nn.functional.pad(flat, (0, groups * fps - flat.numel())).view(groups, fps).amax(1)
    return flat, fps, c.shape


def _fp8_contract(a, q, pia, b):
    """The product of the e4m3 codes that A has (absolute maximum of each group at 448), in 64 bits."""
    top, fps, shape = _fp8_scales(a, q, pia)
    order = [m - 1 if m < q else m - 2 for m in reversed(pia) if m != q]
    back = sorted(range(len(order)), key=lambda r: order[r])
    spread = lambda x: x.repeat_interleave(fps)[:math.prod(shape)].view(shape).permute(back)
    ones, most = torch.ones_like(top), torch.full_like(top, 448.0)
    inv = spread(torch.where(top > 0, most / top, ones))          # divisions, not products with a reciprocal
    scale = spread(torch.where(top > 0, top / most, ones))
    out = 0
    step = max(1, (1 << 28) // inv.numel())
    for k0 in range(0, a.shape[q - 1], step):
        kk = min(step, a.shape[q - 1] - k0)
        x = (a.narrow(q - 1, k0, kk) * inv.unsqueeze(q - 1)).clamp_(-448, 448).to(torch.float8_e4m3fn)
        out = out + _contract(x.to(torch.float32), q, b[k0:k0 + kk])
    return out * scale.double()


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        return [_contract(a, q, b) for q, a, b in _batch_inputs(case, seed)]
    a, bs = _inputs(case, seed)
    if kind == "quantise":
        if case["dtype"] == "bf16":
            return None                       # whole numbers (the bits)
        top = _fp8_scales(a, case["q"], _numbers(case["pia"], ","))[0].double()
        return [None, torch.where(top > 0, top / 448.0, torch.ones_like(top))]
    if kind == "chain":
        left = sorted((m for m in bs if m != case["q"]), reverse=True)
        for m in left:                        # from the highest mode down: lower modes keep their numbers
            a = _contract(a, m, bs[m])
        return a
    if case["dtype"] == "bf16":
        a = a.to(torch.bfloat16).to(torch.float32)
    if case["dtype"] == "fp8":
        return [_fp8_contract(a, q, _numbers(case["pia"], ","), bs[q]) for q in _modes(case)]
    return [_contract(a, q, bs[q]) for q in _modes(case)]
