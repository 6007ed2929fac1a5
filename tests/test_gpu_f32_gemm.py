"""GPU parity of the one-launch f32 GEMM behind Ignis matmul forward / backward
(rust-gpu_amd/csrc/gemm_f32.h; src/ignis/ops/bf16_matmul.rs:33-316): every tile, with and without the
K cut over workgroups, at sizes off every tile edge.

Bars: integer operands (|v| <= 8, sums below 2^24) are exact in f32, so the result equals the 64-bit
product bit for bit.  N(0,1) operands: the error of a sum of k exact products added in any order is at
most k * 2^-24 * sum |a b| per output; the bound below uses the root of k times 4, far above a random
walk's.  Operands sit between NaNs, so a value read from outside them shows.
"""
import numpy as np
import pytest

import oracle
import t0mi
from gpu_helpers import runtime, torch

pytestmark = pytest.mark.gpu

# (m, n, k): the product's own sizes.  The tile (and the K pieces) the plan takes for the forward
# product; the other two products take the same or a neighbouring one.
SHAPES = [
    (5, 4, 3),          # 64x64, one cut K tile
    (33, 68, 31),       # 64x64 / 32x32
    (16, 512, 704),     # 32x32
    (13, 260, 7235),    # 32x32, 8 pieces, K % 4 != 0
    (129, 65, 514),     # 64x64, 8 pieces, rows of no multiple of 4
    (40, 300, 1000),    # 64x32, 8 pieces
    (333, 770, 1100),   # 64x32
    (200, 400, 33),     # 64x64
    (130, 3000, 2001),  # 64x64
    (16, 4096, 4096),   # 64x64, 4 pieces
    (512, 1024, 4096),  # 128x64, 4 pieces
    (2048, 517, 129),   # 128x64
    (700, 3001, 101),   # 128x128
    (290, 2168, 3100),  # 128x128, 4 pieces
]
MODES = ["forward", "data", "weight"]


@pytest.fixture(scope="module")
def rt():
    r = runtime()
    yield r
    r.close()


def in_nans(t):
    """A copy of `t` on the GPU with 256 NaNs before and after it."""
    th = torch()
    buf = th.full((t.numel() + 512,), float("nan"), device="cuda:0")
    v = buf[256:256 + t.numel()].view(t.shape)
    v.copy_(t)
    return v


def product(rt, mode, a, b, y, m, n, k):
    """Y[m,n] over K = k: the entry point's own argument order for each product."""
    if mode == "forward":
        rt.matmul(a.data_ptr(), b.data_ptr(), y.data_ptr(), m, k, n)
    elif mode == "data":
        rt.matmul_backward_data(a.data_ptr(), b.data_ptr(), y.data_ptr(), m, n, k)
    else:
        rt.matmul_backward_weight(a.data_ptr(), b.data_ptr(), y.data_ptr(), k, m, n)


def operands(mode, m, n, k, ints):
    th = torch()
    g = th.Generator(device="cuda:0").manual_seed(m * 7 + n * 3 + k)
    a = th.randn(m, k, generator=g, device="cuda:0")
    b = th.randn(k, n, generator=g, device="cuda:0")
    if ints:
        a, b = (a * 3).round().clamp(-8, 8), (b * 3).round().clamp(-8, 8)
    exact = a.bfloat16().double() @ b.bfloat16().double()
    mag = a.bfloat16().double().abs() @ b.bfloat16().double().abs()
    fa = in_nans(a.t().contiguous() if mode == "weight" else a)
    fb = in_nans(b.t().contiguous() if mode == "data" else b)
    return fa, fb, exact, mag


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_f32_product(rt, mode, m, n, k):
    th = torch()
    for ints in (True, False):
        a, b, exact, mag = operands(mode, m, n, k, ints)
        buf = th.full((m * n + 1024,), 7.5, device="cuda:0")
        y = buf[:m * n].view(m, n)
        y.fill_(float("nan"))
        product(rt, mode, a, b, y, m, n, k)
        th.cuda.synchronize()
        assert bool((buf[m * n:] == 7.5).all()), "wrote past Y"
        if ints:
            assert float(mag.max()) < 2**24
            assert th.equal(y.double(), exact)
        else:
            assert bool(((y.double() - exact).abs() <= 4 * k**0.5 * 2.0**-24 * mag + 1e-30).all())
        z = th.empty_like(y)
        product(rt, mode, a, b, z, m, n, k)
        th.cuda.synchronize()
        assert th.equal(y, z), "a second call differs"


# (m, n, k), on the 32x64 tile but for the last three
WT_SHAPES = [
    (1, 8, 8), (3, 200, 40),   # one cut K tile, columns short of the tile
    (7, 11008, 2048),
    (17, 520, 3000),           # K pieces, K % 32 != 0
    (16, 512, 8192),           # 8 pieces
    (33, 1000, 264), (64, 4096, 1032),  # two row tiles
    (64, 72, 4096),
    (44, 9960, 264),           # 64x64, K % 32 != 0
    (64, 13000, 72),           # 64x64, three K tiles, the last one cut
    (62, 3672, 7288),          # 64x64, 4 pieces, K % 32 != 0
]


@pytest.mark.parametrize("m,n,k", WT_SHAPES)
def test_bf16_weight(rt, m, n, k):
    """matmul_with_wt_bf16 (bf16_matmul.rs:99-134): X f32, WT bf16 in place; same bars."""
    th = torch()
    for ints in (True, False):
        a, _, exact, mag = operands("forward", m, n, k, ints)
        g = th.Generator(device="cuda:0").manual_seed(m * 7 + n * 3 + k)
        th.randn(m, k, generator=g, device="cuda:0")
        b = th.randn(k, n, generator=g, device="cuda:0")  # operands()' second draw
        if ints:
            b = (b * 3).round().clamp(-8, 8)
        wt = th.full((n * k + 512,), float("nan"), device="cuda:0", dtype=th.bfloat16)
        w = wt[256:256 + n * k].view(n, k)
        w.copy_(b.t())
        buf = th.full((m * n + 1024,), 7.5, device="cuda:0")
        y = buf[:m * n].view(m, n)
        y.fill_(float("nan"))
        rt.matmul_with_wt_bf16(a.data_ptr(), w.data_ptr(), y.data_ptr(), m, k, n)
        th.cuda.synchronize()
        assert bool((buf[m * n:] == 7.5).all()), "wrote past Y"
        if ints:
            assert th.equal(y.double(), exact)
        else:
            assert bool(((y.double() - exact).abs() <= 4 * k**0.5 * 2.0**-24 * mag + 1e-30).all())


def test_f32_product_against_oracle(rt):
    m, n, k = 333, 770, 1100
    th = torch()
    a, b, _, _ = operands("forward", m, n, k, False)
    y = th.empty(m, n, device="cuda:0")
    product(rt, "forward", a, b, y, m, n, k)
    ab, bb = oracle.bf16_rne(a.cpu().numpy()), oracle.bf16_rne(b.cpu().numpy())
    err, rel = oracle.compare(y.cpu().numpy(), oracle.gemm_bf16(ab, bb, "nn"))
    assert err <= oracle.gemm_tolerance(k, oracle.bf16_to_f32(ab), oracle.bf16_to_f32(bb)) and rel < 1e-5


def test_output_over_an_operand(rt):
    """Y in X's place (square W): both operands are read before Y is written, as ever."""
    th = torch()
    m = n = k = 96
    a, b, exact, _ = operands("forward", m, n, k, True)
    x = a.clone()
    rt.matmul(x.data_ptr(), b.data_ptr(), x.data_ptr(), m, k, n)
    th.cuda.synchronize()
    assert th.equal(x.double(), exact)


def test_special_values(rt):
    """Infinities and NaN reach their own outputs and no others (one K row of zeros against them)."""
    th = torch()
    m, n, k = 70, 132, 75
    a, b, _, _ = operands("forward", m, n, k, True)
    a[3, 10], a[4, 20], a[5, 74] = float("inf"), float("nan"), -float("inf")
    b[10, :], b[74, :] = 1.0, 2.0
    y = th.empty(m, n, device="cuda:0")
    product(rt, "forward", a, b, y, m, n, k)
    th.cuda.synchronize()
    assert bool((y[3] == float("inf")).all()) and bool(y[4].isnan().all()) and bool((y[5] == -float("inf")).all())
    rest = th.cat([y[:3], y[6:]])
    assert bool(rest.isfinite().all())


def test_graph_replay_of_split_calls(rt):
    """The in-launch exchange (counters, slots) recorded into a graph with other calls on either side:
    every replay equals the eager result."""
    th = torch()
    shapes = [(16, 4096, 4096), (40, 300, 1000), (512, 1024, 4096)]
    st = th.cuda.Stream()
    with th.cuda.stream(st):
        r = t0mi.Runtime(device=0, stream=st.cuda_stream)
        data = [operands("forward", *s, False)[:2] for s in shapes]
        want = []
        for (a, b), (m, n, k) in zip(data, shapes):
            y = th.empty(m, n, device="cuda:0")
            product(r, "forward", a, b, y, m, n, k)
            want.append(y)
        st.synchronize()
        outs = [th.empty_like(w) for w in want]
        r.capture_begin()
        for (a, b), y, (m, n, k) in zip(data, outs, shapes):
            product(r, "forward", a, b, y, m, n, k)
        g = r.capture_end()
        for _ in range(4):
            for y in outs:
                y.fill_(float("nan"))
            g.launch()
            st.synchronize()
            for y, w in zip(outs, want):
                assert th.equal(y, w)
            product(r, "forward", *data[1], outs[1], *shapes[1])  # eager work between the replays
        st.synchronize()
        g.destroy()
        r.close()
    assert np.all([bool(w.isfinite().all()) for w in want])
