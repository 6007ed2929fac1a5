"""Which kernels libt0mi launches for a call, and that a call which returned no error launched what it
needs: the host side alone, with a stand-in for the HIP runtime (host_runtime.py).  The kernels'
results are the GPU tests' matter."""
import pytest

from host_runtime import host  # noqa: F401

PLANES = ["gemm_bf16_planes_kernel", "t0mi_splitk_reduce"]


@pytest.mark.parametrize("layout", ["NT", "NN"])
@pytest.mark.parametrize("m,k,n", [(128, 1024, 1024), (256, 1024, 1024), (100, 1032, 1032)])
def test_split_two_writes_y_after_the_operands_are_read(host, m, k, n, layout):
    """64x64 tiles in two K partitions: summed inside the launch, which stores a tile of Y while others
    read X and B; so planes and a reduce where Y meets X, B or the bias by so much as one row's end."""
    r = host(f"""
m, k, n = {m}, {k}, {n}
cfg = t0mi.auto_select_layout(m, k, n, t0mi.{layout}, t0mi.OUT_BF16)
assert (cfg.tile_m, cfg.tile_n, cfg.split_k) == (64, 64, 2)
bias = cfg.copy(epilogue=t0mi.EPI_BIAS_ADD)
rt.gemm(cfg, X, B, Y, m, n, k)  # the buffers are made
xb, bb, yb = m * k * 2, n * k * 2, m * n * 2
done(dict(
    apart=[names(rt.gemm, c, x, b, y, m, n, k, z) for c, x, b, y, z in [
        (cfg, X, B, Y, 0), (bias, X, B, Y, BIAS), (cfg, X, B, X + xb, 0), (cfg, X, B, X - yb, 0),
        (cfg, X, B, B + bb, 0), (bias, X, B, BIAS + 4 * n, BIAS)]],
    over=[names(rt.gemm, c, x, b, y, m, n, k, z) for c, x, b, y, z in [
        (cfg, X, B, X, 0), (cfg, X, B, B, 0), (bias, X, B, BIAS, BIAS), (cfg, X, B, X + xb - 16, 0),
        (cfg, X, B, X - yb + 16, 0), (cfg, X, B, B + bb - 16, 0), (bias, X, B, BIAS + 4 * n - 16, BIAS)]],
))
""")
    assert all(c == ["gemm_bf16_exchange_kernel"] for c in r["apart"]), r["apart"]
    assert all(c == PLANES for c in r["over"]), r["over"]


def test_gptq_parameters_over_the_packed_weights(host):
    """The weights are read whole before scales or zero points are written into their place."""
    r = host("""
rows, cols, group = 72, 520, 8
pk, pr = rows * cols // 2, cols // group * rows
S, Z, Q, S2, Z2 = [i << 40 for i in range(2, 7)]
hip.fake_launches()
def grids(s2, z2):
    rt.gptq_convert(X, S, Z, rows, cols, group, Q, s2, z2)
    return [l[1] for l in launches()]
done(dict(apart=[grids(S2, Z2), grids(X + pk, Z2), grids(S2, X + pk), grids(X - pr * 2, Z2), grids(S2, X - pr // 2)],
          over=[grids(X, Z2), grids(S2, X), grids(X + pk - 2, Z2), grids(X - pr * 2 + 2, Z2), grids(S2, X + pk - 4),
                grids(S2, X - pr // 2 + 4), grids(X, X + pr * 2)]))
""")
    weights, params = 2 * 2, 3 * 2  # 65 words and 72 rows in 64s; 65 groups in 32s and 72 rows in 64s
    assert r["apart"] == [[weights + params]] * 5
    assert r["over"] == [[weights, params]] * 7
