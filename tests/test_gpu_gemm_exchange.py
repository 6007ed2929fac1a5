"""GPU parity of bf16 GEMMs that sum their two K partitions inside the launch (csrc/gemm_bf16_kernel.h,
exchange_partitions): 64x64 tiles.  `gemm_noalloc` keeps its partial planes in the fixed scratch and sums
them in a launch of their own; a sum of two f32 values has one result, so both must agree bit for bit.
Cases: row and column tails of one, a last K partition that is empty or partial, one tile and several
hundred, f32 and bf16 outputs, bias + ReLU, repeated calls (the arrival counters are left at zero), and a
captured call replayed with eager work between the replays."""
import numpy as np
import pytest

import oracle
import t0mi
from gpu_helpers import empty_dev, from_dev, runtime, to_dev, torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rt():
    r = runtime()
    yield r
    r.close()


def config(nn, od, stages, epilogue=0):
    return t0mi.GemmConfig(tile_m=64, tile_n=64, tile_k=64, wg_size=256, use_lds=1, double_buffer=1, n_col_passes=1,
                           swap_grid=1, transpose=t0mi.NN if nn else t0mi.NT, wave_m=2, wave_n=2, stages=stages,
                           split_k=2, out_dtype=od, epilogue=epilogue)


@pytest.mark.parametrize("m,n,k", [(1, 8, 64), (1, 64, 72), (33, 72, 128), (64, 64, 1032), (65, 136, 200),
                                   (100, 1000, 1032), (97, 4096, 520), (700, 1032, 264)])
@pytest.mark.parametrize("nn,od,epilogue,stages", [
    (False, t0mi.OUT_F32, 0, 4), (True, t0mi.OUT_BF16, 0, 4),
    (True, t0mi.OUT_F32, t0mi.EPI_BIAS_ADD_RELU, 3), (False, t0mi.OUT_BF16, 0, 0),
])
def test_equals_planes(rt, m, n, k, nn, od, epilogue, stages):
    a = oracle.normal_bf16((m, k), m + k, 0.0, 1.0)
    b = oracle.normal_bf16((k, n) if nn else (n, k), n + k, 0.0, 1.0)
    bias = np.linspace(-1, 1, n, dtype=np.float32)
    (da, pa), (db, pb), (dc, pc) = to_dev(a), to_dev(b), to_dev(bias)
    dt = np.uint16 if od == t0mi.OUT_BF16 else np.float32
    cfg = config(nn, od, stages, epilogue)

    def call(f):
        dy, py = empty_dev(m * n * np.dtype(dt).itemsize, fill=0xCD)
        f(cfg, pa, pb, py, m, n, k, pc if epilogue else 0)
        return from_dev(dy, dt, (m, n))

    want = call(rt.gemm_noalloc)
    for _ in range(3):
        assert np.array_equal(call(rt.gemm), want)
    af = oracle.bf16_to_f32(a).astype(np.float64)
    bf = oracle.bf16_to_f32(b).astype(np.float64)
    bf = bf if nn else bf.T
    exact, mag = af @ bf, np.abs(af) @ np.abs(bf)
    if epilogue:
        exact, mag = np.maximum(exact + bias, 0), mag + np.abs(bias)
    got = oracle.bf16_to_f32(want) if od == t0mi.OUT_BF16 else want
    # f32 sums of k + 1 terms, then (bf16) one rounding of 2^-9
    lim = 2 * (k + 1) * 2.0**-24 * mag + (2.0**-8 * np.abs(exact) if od == t0mi.OUT_BF16 else 0)
    assert (np.abs(got - exact) <= lim).all()


@pytest.mark.parametrize("m,n,k", [(128, 1024, 1024), (100, 1032, 1032)])
@pytest.mark.parametrize("over", ["x", "b"])
@pytest.mark.parametrize("nn", [False, True])
def test_output_over_an_operand(rt, m, n, k, over, nn):
    """Y (bf16) in an operand's place, with the configuration the ranking picks: the planes route, whose
    reduce runs after the last read of the operands, as gemm_noalloc."""
    cfg = t0mi.auto_select_layout(m, k, n, t0mi.NN if nn else t0mi.NT, t0mi.OUT_BF16)
    assert (cfg.tile_m, cfg.tile_n, cfg.split_k) == (64, 64, 2)
    cfg = cfg.copy(epilogue=t0mi.EPI_BIAS_ADD)
    a = oracle.normal_bf16((m, k), m + k, 0.0, 1.0)
    b = oracle.normal_bf16((k, n) if nn else (n, k), n + k, 0.0, 1.0)
    bias = np.linspace(-1, 1, n, dtype=np.float32)

    def call(f, y):
        ops = {"x": a, "b": b, "bias": bias}
        dev = {o: to_dev(v) for o, v in ops.items()}
        dy, py = dev[y] if y else empty_dev(m * n * 2, fill=0xCD)
        f(cfg, dev["x"][1], dev["b"][1], py, m, n, k, dev["bias"][1])
        return from_dev(dy, np.uint16, (m, n))

    want = call(rt.gemm_noalloc, None)
    for _ in range(3):
        assert np.array_equal(call(rt.gemm, over), want)


def test_capture(rt):
    th = torch()
    st = th.cuda.Stream()
    m, n, k = 100, 1000, 1032
    with th.cuda.stream(st):
        r = t0mi.Runtime(device=0, stream=st.cuda_stream)
        x = th.randn(m, k, device="cuda:0").bfloat16()
        w = th.randn(n, k, device="cuda:0").bfloat16()
        want, y = th.empty(m, n, device="cuda:0"), th.empty(m, n, device="cuda:0")
        cfg = config(False, t0mi.OUT_F32, 4)
        r.gemm(cfg, x.data_ptr(), w.data_ptr(), want.data_ptr(), m, n, k)
        st.synchronize()
        r.capture_begin()
        r.gemm(cfg, x.data_ptr(), w.data_ptr(), y.data_ptr(), m, n, k)
        g = r.capture_end()
        for _ in range(4):
            y.fill_(float("nan"))
            g.launch()
            st.synchronize()
            assert th.equal(y, want)
            r.gemm(cfg, x.data_ptr(), w.data_ptr(), y.data_ptr(), m, n, k)  # eager work between the replays
        st.synchronize()
        g.destroy()
        r.close()
