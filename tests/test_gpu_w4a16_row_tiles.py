"""GPU parity of the W4A16 decode kernel's row tiles in one launch (csrc/w4a16.hip, decode_row_tiles): a
narrow weight's 64-column strips leave CUs idle, so the slabs of a call run as several tiles of 1 to 4
slabs side by side.  Every row goes through the operations of a 16-row slab whatever the tile, so the
f32 results equal, bit for bit, those of the same rows inside a call that tiles them differently; and
they are within the fp32 bound k * 2^-24 * sum |a w| (times 2) of the exact product.
Cases: a last tile of one row, of one slab, tiles of 1, 2, 3 and 4 slabs, planes over K (K > 4096) with
tiles of one slab and of three, groups 32 to 256, widths off the strip (test_host_routes.py holds them to it)."""
import numpy as np
import pytest

import oracle
import t0mi
from gpu_helpers import empty_dev, from_dev, runtime, to_dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rt():
    r = runtime()
    yield r
    r.close()


CASES = [
    (17, 1024, 520, 128, True),     # two tiles of one slab, the last one row
    (33, 512, 4096, 64, False),     # three of one
    (100, 4096, 1376, 128, True),   # seven of one
    (129, 512, 1000, 32, True),     # nine of one, one row past eight slabs
    (191, 1024, 4096, 128, False),  # four of three
    (96, 2048, 520, 256, True),     # group 256: six of one
    (112, 8192, 520, 128, True),    # seven of one, planes over K
    (150, 512, 6000, 128, False),   # five of two, 94 strips
    (128, 512, 6000, 128, True),    # two of four
    (100, 1024, 4096, 64, True),    # group 64: four of two
    (112, 512, 5000, 32, False),    # group 32: three of three, the last one slab
    (96, 512, 6000, 256, True),     # group 256: three of two
    (185, 8192, 2048, 128, False),  # four of three, planes over K
]


@pytest.mark.parametrize("m,k,n,group,zeros", CASES)
def test_row_tiles(rt, m, k, n, group, zeros):
    a = oracle.normal_bf16((m, k), 3 * m + n, 0.0, 1.0)
    w = oracle.pack_qweight(oracle.nibbles((k, n), m + 1))
    s = oracle.uniform_bf16((k // group, n), m + 2, 0.005, 0.02)
    z = oracle.pack_qzeros(oracle.nibbles((k // group, n), m + 3)) if zeros else None
    da, pa = to_dev(a)
    dw, pw = to_dev(w)
    ds, ps = to_dev(s)
    pz = 0
    if zeros:
        dz, pz = to_dev(z)

    def call(r0, rows):
        dy, py = empty_dev(rows * n * 4, fill=0xCD)
        rt.w4a16_gemm(pa + r0 * k * 2, pw, ps, pz, 8, py, rows, k, n, group, t0mi.OUT_F32)
        return from_dev(dy, np.float32, (rows, n))

    y = call(0, m)
    wf = oracle.dequant_qweight_f32(w, s, z, group, 8).astype(np.float64)
    af = oracle.bf16_to_f32(a).astype(np.float64)
    lim = 2 * k * 2.0**-24 * (np.abs(af) @ np.abs(wf))
    assert (np.abs(y - af @ wf) <= lim).all()
    for r0, rows in ((0, min(m, 48)), (16, m - 16)):  # other tilings of the same rows, over 16 rows each
        if rows > 16:
            assert np.array_equal(call(r0, rows), y[r0:r0 + rows]), (r0, rows)


def test_output_over_the_activations(rt):
    """One strip and one launch of four slabs: Y (f32, the size of A) in A's place."""
    m, k, n, group = 64, 128, 64, 128
    a = oracle.normal_bf16((m, k), 5, 0.0, 1.0)
    w = oracle.pack_qweight(oracle.nibbles((k, n), 6))
    s = oracle.uniform_bf16((k // group, n), 7, 0.005, 0.02)
    (da, pa), (dw, pw), (ds, ps) = to_dev(a), to_dev(w), to_dev(s)
    dy, py = empty_dev(m * n * 4, fill=0xCD)
    rt.w4a16_gemm(pa, pw, ps, 0, 8, py, m, k, n, group, t0mi.OUT_F32)
    want = from_dev(dy, np.float32, (m, n))
    rt.w4a16_gemm(pa, pw, ps, 0, 8, pa, m, k, n, group, t0mi.OUT_F32)
    assert np.array_equal(from_dev(da, np.float32, (m, n)), want)
