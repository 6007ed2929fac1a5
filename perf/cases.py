"""The work that users of this library have it do, as measurable cases through its public entry points.

Every case is one call (or one layer step) on data that is already in HBM.  Kinds:

  gemm    `Runtime.gemm` with the configuration `auto_select_layout` picks: a bf16 matrix product
  tile    `Runtime.tile_gemm` with `tile_auto_select`'s spec and a fused epilogue: an activation layer
  w4a16   `Runtime.w4a16_gemm`: int4 weights, bf16 activations (decode, batched decode, prefill)
  wt      `Runtime.matmul_with_wt_bf16`: an f32 program's inference layer on its cached bf16 weight
  linear  `Runtime.matmul` + `matmul_backward_data` + `matmul_backward_weight`: one f32 training step
          of a linear layer
  matmul  `Runtime.matmul`: the forward alone, on an f32 weight
  gptq    `Runtime.gptq_convert`: a GPTQ container's sections to the W4A16 layouts (model load)
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "rust-gpu_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)
import t0mi  # noqa: E402

_rt = None


def _runtime():
    """One runtime for the whole program, on torch's stream."""
    global _rt
    if _rt is None:
        torch.cuda.init()
        _rt = t0mi.Runtime.on_torch_stream(0)
    return _rt


def listed():
    return [
        # A small product, off the tile grid: launch latency and host time count.
        dict(name="gemm_100x1000x1032", kind="gemm", m=100, n=1000, k=1032, nn=False, bf16=False),
        # A small prompt (128 tokens) through a 4096-wide projection: bound by the weight's bytes.
        dict(name="gemm_128x4096x4096", kind="gemm", m=128, n=4096, k=4096, nn=True, bf16=True),
        # The large square product: bound by the matrix cores.
        dict(name="gemm_4096", kind="gemm", m=4096, n=4096, k=4096, nn=True, bf16=True),
        # An MLP layer with its bias and activation fused, rows and widths off the tile grid.
        dict(name="tile_1000x2752x2056", kind="tile", m=1000, n=2752, k=2056, nn=False, bf16=True, act="gelu"),
        # Token generation for 16 sequences on a 4-bit weight: bound by the packed bytes.
        dict(name="w4a16_decode_16", kind="w4a16", m=16, n=11008, k=4096, group=128, zeros=False, bf16=True),
        # Batched generation / a short prompt on the same weight, per-group zero points.
        dict(name="w4a16_rows_100", kind="w4a16", m=100, n=11008, k=4096, group=128, zeros=True, bf16=True),
        # A long prompt on a 4-bit weight: bound by the matrix cores.
        dict(name="w4a16_prefill_4096", kind="w4a16", m=4096, n=14336, k=4096, group=128, zeros=True, bf16=True),
        # f32 inference of a few sequences on a cached bf16 weight.
        dict(name="wt_7x11008x2048", kind="wt", m=7, n=11008, k=2048),
        # One training step (forward, data gradient, weight gradient) of a mid-sized layer.
        dict(name="linear_512x4096x1024", kind="linear", m=512, n=4096, k=1024),
        # The same step at sizes that are not multiples of anything.
        dict(name="linear_333x770x1100", kind="linear", m=333, n=770, k=1100),
        # f32 inference without a cached weight: the f32 weight is read and rounded on each call.
        dict(name="matmul_16x4096x4096", kind="matmul", m=16, n=4096, k=4096),
        # Loading a 4-bit checkpoint.
        dict(name="gptq_11008x4096", kind="gptq", n=11008, k=4096, group=128),
    ]


_MOST_FLOPS = 2.0 * 4096 * 4096 * 14336  # the largest listed case


def _spread(rng, lo, hi, step=1):
    """A multiple of `step` in [lo, hi], spread over its logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    while True:
        kind = rng.choice(["gemm", "tile", "w4a16", "w4a16", "wt", "linear", "matmul", "gptq"])
        if kind == "gemm":
            c = dict(kind=kind, m=_spread(rng, 1, 4096), n=_spread(rng, 64, 14336, 8), k=_spread(rng, 64, 14336, 8),
                     nn=rng.random() < 0.5, bf16=rng.random() < 0.6)
        elif kind == "tile":
            c = dict(kind=kind, m=_spread(rng, 1, 4096), n=_spread(rng, 64, 11008, 8), k=_spread(rng, 64, 8192, 8),
                     nn=rng.random() < 0.3, bf16=rng.random() < 0.6, act=rng.choice(["gelu", "silu", "relu", "none"]))
        elif kind == "w4a16":
            group = rng.choice([128, 128, 128, 64, 32, 256])
            c = dict(kind=kind, m=_spread(rng, 1, 4096), n=_spread(rng, 256, 14336, 8),
                     k=_spread(rng, max(512, group), 14336, group), group=group, zeros=rng.random() < 0.7,
                     bf16=rng.random() < 0.8)
        elif kind == "wt":
            c = dict(kind=kind, m=_spread(rng, 1, 64), n=_spread(rng, 256, 14336, 8), k=_spread(rng, 256, 8192, 8))
        elif kind == "linear":
            step = rng.choice([1, 2, 8, 64])
            c = dict(kind=kind, m=_spread(rng, 8, 2048), n=_spread(rng, 64, 8192, step), k=_spread(rng, 64, 8192, step))
        elif kind == "matmul":
            step = rng.choice([1, 8, 64])
            c = dict(kind=kind, m=_spread(rng, 1, 128), n=_spread(rng, 64, 11008, step), k=_spread(rng, 64, 8192, step))
        else:
            group = rng.choice([128, 128, 64, 32])
            c = dict(kind=kind, n=_spread(rng, 256, 14336, 8), k=_spread(rng, 512, 14336, group), group=group)
        w = work(c)
        if w["flops"] <= _MOST_FLOPS and w["bytes"] >= 1.5e6:  # below, a call is the host's enqueue alone
            return c


def _inputs(case, seed):
    """The case's operands, from the seed alone: activations ~ N(0, 1), weights ~ N(0, 1/K), scales and
    zero points as 4-bit checkpoints have them."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    kind = case["kind"]
    n, k = case["n"], case["k"]
    m = case.get("m", 0)

    def normal(*shape, std=1.0):
        return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32) * std

    def words(*shape):
        return torch.randint(-2**31, 2**31, shape, generator=g, device="cuda", dtype=torch.int32)

    w_std = 1.0 / math.sqrt(k)
    t = {}
    if kind in ("gemm", "tile"):
        t["x"] = normal(m, k).bfloat16()
        t["w"] = (normal(k, n, std=w_std) if case["nn"] else normal(n, k, std=w_std)).bfloat16()
        if kind == "tile":
            t["bias"] = normal(n, std=0.1)
    elif kind == "w4a16":
        groups = k // case["group"]
        t["x"] = normal(m, k).bfloat16()
        t["q"] = words(k // 8, n)
        t["s"] = (torch.rand(groups, n, generator=g, device="cuda") * 0.015 + 0.005).bfloat16()
        t["z"] = words(groups, n // 8) if case["zeros"] else None
    elif kind == "wt":
        t["x"] = normal(m, k)
        t["w"] = normal(n, k, std=w_std).bfloat16()
    elif kind == "gptq":
        groups = k // case["group"]
        t["q"] = words(n, k // 8)
        t["s"] = (torch.rand(n, groups, generator=g, device="cuda") * 0.015 + 0.005).bfloat16().float()
        t["z"] = torch.randint(0, 16, (n, groups), generator=g, device="cuda", dtype=torch.int32)
    else:
        t["x"] = normal(m, k)
        t["w"] = normal(k, n, std=w_std)
        if kind == "linear":
            t["dy"] = normal(m, n)
    return t


def prepare(case, seed):
    kind = case["kind"]
    n, k = case["n"], case["k"]
    m = case.get("m", 0)
    s = _inputs(case, seed)
    s["rt"] = _runtime()
    s["kind"] = kind
    s["dims"] = (m, n, k)
    out = torch.bfloat16 if case.get("bf16") else torch.float32
    od = t0mi.OUT_BF16 if case.get("bf16") else t0mi.OUT_F32
    if kind != "gptq":
        s["y"] = torch.empty(m, n, dtype=out, device="cuda")
    if kind == "gemm":
        s["cfg"] = t0mi.auto_select_layout(m, k, n, t0mi.NN if case["nn"] else t0mi.NT, od)
    elif kind == "tile":
        spec = t0mi.tile_auto_select(m, k, n, t0mi.NN if case["nn"] else t0mi.NT)
        ops = {"gelu": [t0mi.GELU], "silu": [t0mi.SILU], "relu": [t0mi.RELU], "none": []}[case["act"]]
        s["spec"] = spec.copy(out_dtype=od, epilogue=[t0mi.BIAS_ADD] + ops)
    elif kind == "w4a16":
        s["group"], s["od"] = case["group"], od
    elif kind == "linear":
        s["dx"] = torch.empty(m, k, device="cuda")
        s["dw"] = torch.empty(k, n, device="cuda")
    elif kind == "gptq":
        groups = k // case["group"]
        s["group"] = case["group"]
        s["qweight"] = torch.empty(k // 8, n, dtype=torch.int32, device="cuda")
        s["scales"] = torch.empty(groups, n, dtype=torch.bfloat16, device="cuda")
        s["qzeros"] = torch.empty(groups, n // 8, dtype=torch.int32, device="cuda")
    return s


def run(s):
    rt, kind = s["rt"], s["kind"]
    m, n, k = s["dims"]
    if kind == "gemm":
        rt.gemm(s["cfg"], s["x"].data_ptr(), s["w"].data_ptr(), s["y"].data_ptr(), m, n, k)
    elif kind == "tile":
        rt.tile_gemm(s["spec"], s["x"].data_ptr(), s["w"].data_ptr(), s["y"].data_ptr(), m, n, k,
                     bias=s["bias"].data_ptr())
    elif kind == "w4a16":
        z = s["z"]
        rt.w4a16_gemm(s["x"].data_ptr(), s["q"].data_ptr(), s["s"].data_ptr(), 0 if z is None else z.data_ptr(), 8,
                      s["y"].data_ptr(), m, k, n, s["group"], s["od"])
    elif kind == "wt":
        rt.matmul_with_wt_bf16(s["x"].data_ptr(), s["w"].data_ptr(), s["y"].data_ptr(), m, k, n)
    elif kind == "linear":
        x, w, dy = s["x"].data_ptr(), s["w"].data_ptr(), s["dy"].data_ptr()
        rt.matmul(x, w, s["y"].data_ptr(), m, k, n)
        rt.matmul_backward_data(dy, w, s["dx"].data_ptr(), m, k, n)
        rt.matmul_backward_weight(x, dy, s["dw"].data_ptr(), m, k, n)
        return {"y": s["y"], "dx": s["dx"], "dw": s["dw"]}
    elif kind == "matmul":
        rt.matmul(s["x"].data_ptr(), s["w"].data_ptr(), s["y"].data_ptr(), m, k, n)
    else:
        rt.gptq_convert(s["q"].data_ptr(), s["s"].data_ptr(), s["z"].data_ptr(), n, k, s["group"],
                        s["qweight"].data_ptr(), s["scales"].data_ptr(), s["qzeros"].data_ptr())
        return {"qweight": s["qweight"], "scales": s["scales"], "qzeros": s["qzeros"]}
    return s["y"]


def work(case):
    kind = case["kind"]
    n, k = case["n"], case["k"]
    m = case.get("m", 0)
    out = 2 if case.get("bf16") else 4
    if kind == "gptq":
        groups = k // case["group"]
        return {"bytes": 2 * (n * k // 2) + groups * n * (8 + 2) + groups * n // 2, "flops": 0}
    flops = 2.0 * m * n * k
    if kind in ("gemm", "tile"):
        b = 2 * m * k + 2 * k * n + out * m * n + (4 * n if kind == "tile" else 0)
    elif kind == "w4a16":
        groups = k // case["group"]
        b = 2 * m * k + k * n // 2 + 2 * groups * n + (groups * n // 2 if case["zeros"] else 0) + out * m * n
    elif kind == "wt":
        b = 4 * m * k + 2 * k * n + 4 * m * n
    elif kind == "matmul":
        b = 4 * (m * k + k * n + m * n)
    else:  # x, w and dy read, y, dx and dw written
        b = 2 * 4 * (m * k + k * n + m * n)
        flops *= 3
    return {"bytes": b, "flops": flops}


def tolerance(case):
    """Four times what each kind's error against 64 bits measures (or a sum in another order differs by)."""
    kind = case["kind"]
    if kind == "gptq":
        return "exact"
    if case.get("bf16"):
        # The result's own rounding to bf16 (1.7e-3 in the 2-norm); the prefill routes of w4a16 round
        # the weights to bf16 too (2.3e-3).  Two bf16 units in the last place for a single value.
        return {"rel": 9e-3 if kind == "w4a16" else 7e-3, "max": 0.04 if kind == "w4a16" else 2.0**-6}
    if kind == "w4a16":  # f32 results, of exact or of bf16-rounded weights (1.6e-3) by row count
        return {"rel": 7e-3, "max": 0.03}
    if kind == "tile":  # the epilogue's exp2 and rcp are the hardware's, about 1 unit in the last place each
        return {"rel": 8e-6, "max": 8e-5}
    # f32 sums of exact bf16 products: 0.4e-7 to 2e-7 at the listed sizes, up to 1e-6 over 14336 terms in order.
    return {"rel": 4e-6, "max": 4e-5}


def exact(case, seed):
    kind = case["kind"]
    t = _inputs(case, seed)
    shifts = torch.arange(0, 32, 4, device="cuda", dtype=torch.int32)
    if kind == "gptq":
        z = t["z"].t().reshape(t["z"].shape[1], -1, 8)
        packed = (z.long() << shifts.long()).sum(-1)
        packed = torch.where(packed >= 2**31, packed - 2**32, packed).int()
        return {"qweight": t["q"].t().contiguous(), "scales": t["s"].t().contiguous().bfloat16(), "qzeros": packed}
    x = t["x"].bfloat16().double()  # the f32 entry points round their operands to bf16 by definition
    if kind == "w4a16":
        q = ((t["q"].unsqueeze(1) >> shifts.view(1, 8, 1)) & 15).reshape(case["k"], case["n"])
        z = 8 if t["z"] is None else ((t["z"].unsqueeze(2) >> shifts) & 15).reshape(-1, case["n"])
        grp = torch.arange(case["k"], device="cuda") // case["group"]
        w = (q - (z if t["z"] is None else z[grp])).double() * t["s"].double()[grp]
        return x @ w
    w = t["w"].bfloat16().double()
    if kind in ("gemm", "tile"):
        y = x @ (w if case["nn"] else w.t().contiguous())
        if kind == "tile":
            y = y + t["bias"].double()
            if case["act"] == "relu":
                y = y.clamp(min=0)
            elif case["act"] != "none":  # silu, and the sigmoid form of gelu
                y = y * torch.sigmoid(y * (1.702 if case["act"] == "gelu" else 1.0))
        return y
    if kind == "wt":
        return x @ w.t().contiguous()
    if kind == "matmul":
        return x @ w
    dy = t["dy"].bfloat16().double()
    return {"y": x @ w, "dx": dy @ w.t().contiguous(), "dw": x.t().contiguous() @ dy}
