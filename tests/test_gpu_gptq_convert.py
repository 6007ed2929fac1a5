"""GPU parity of the GPTQ conversion at the edges of its tiles (rust-gpu_amd/csrc/t0mi_ignis.hip,
src/t0/quant_kernels.rs:177-294): 64 x 64 word blocks, 4 x 4 words a thread, 64 columns x 32 groups of
parameters; sections and outputs at 4-byte (bf16: 2-byte) offsets.  Whole numbers: exact."""
import numpy as np
import pytest

import oracle
from gpu_helpers import check_guard, empty_dev, runtime, to_dev, torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rt():
    r = runtime()
    yield r
    r.close()


def case(rows, cols, group, seed):
    q = oracle.nibbles((cols, rows), seed)
    ng = cols // group
    g = np.random.default_rng(seed)
    scales = (g.standard_normal((rows, ng)) * 0.01).astype(np.float32)  # not bf16-exact: the rounding shows
    zeros = oracle.nibbles((ng, rows), seed + 1)
    return q, scales, zeros


@pytest.mark.parametrize("off", [0, 4])
@pytest.mark.parametrize("rows,cols,group", [
    (8, 8, 8),         # one word row, one group
    (8, 40, 40),       # 5 words per row: a thread's 4 x 4 block cut in K
    (72, 520, 8),      # 65 words, 65 groups: one past the tiles in every direction
    (56, 504, 56),     # 63 words: one short
    (136, 1024, 32),   # 32 groups exactly
    (1000, 264, 24),   # 33 words, 11 groups
])
def test_gptq_convert(rt, rows, cols, group, off):
    q, scales, zeros = case(rows, cols, group, rows + cols)
    ng = cols // group
    pad = np.zeros(off, np.uint8)
    raw = [np.concatenate([pad, a.reshape(-1).view(np.uint8)]) for a in (
        np.ascontiguousarray(oracle.pack_gptq_bytes(q)), scales,
        np.ascontiguousarray(zeros.T.astype(np.int32)))]
    dev = [to_dev(a) for a in raw]
    sizes = [cols // 8 * rows * 4, ng * rows * 2, ng * rows // 8 * 4]
    offs = [off, off // 2, off]
    outs = [empty_dev(n + o, fill=0xAA) for n, o in zip(sizes, offs)]
    rt.gptq_convert(*[p + off for _, p in dev], rows, cols, group, *[p + o for (_, p), o in zip(outs, offs)])
    torch().cuda.synchronize()
    got = []
    for (d, _), n, o in zip(outs, sizes, offs):
        check_guard(d)
        b = d[:n + o].cpu().numpy()
        assert (b[:o] == 0xAA).all()
        got.append(b[o:].copy())
    assert np.array_equal(got[0].view(np.uint32).reshape(cols // 8, rows), oracle.pack_qweight(q))
    assert np.array_equal(got[1].view(np.uint16).reshape(ng, rows), oracle.bf16_rne(np.ascontiguousarray(scales.T)))
    assert np.array_equal(got[2].view(np.uint32).reshape(ng, rows // 8), oracle.pack_qzeros(zeros))


@pytest.mark.parametrize("rows,cols,group", [(72, 520, 8), (4096, 2048, 128)])
def test_parameters_over_the_packed_weights(rt, rows, cols, group):
    """scales_bf16 and qzeros in the packed buffer, whose words are no longer needed."""
    q, scales, zeros = case(rows, cols, group, rows + cols)
    ng = cols // group
    dp, pp = to_dev(np.ascontiguousarray(oracle.pack_gptq_bytes(q)))
    ds, ps = to_dev(scales)
    dz, pz = to_dev(np.ascontiguousarray(zeros.T.astype(np.int32)))
    dq, pq = empty_dev(cols // 8 * rows * 4, fill=0xAA)
    sb, zb = ng * rows * 2, ng * rows // 2
    rt.gptq_convert(pp, ps, pz, rows, cols, group, pq, pp, pp + sb)
    torch().cuda.synchronize()
    check_guard(dq)
    b = dp[:sb + zb].cpu().numpy()
    assert np.array_equal(dq[:cols // 8 * rows * 4].cpu().numpy().view(np.uint32).reshape(cols // 8, rows),
                          oracle.pack_qweight(q))
    assert np.array_equal(b[:sb].view(np.uint16).reshape(ng, rows), oracle.bf16_rne(np.ascontiguousarray(scales.T)))
    assert np.array_equal(b[sb:].view(np.uint32).reshape(ng, rows // 8), oracle.pack_qzeros(zeros))
