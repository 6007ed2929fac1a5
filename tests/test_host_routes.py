"""Which kernels libt0mi launches for a call, and that a call which returned no error launched what it
needs: the host side alone, with a stand-in for the HIP runtime (host_runtime.py).  The kernels'
results are the GPU tests' matter; the last tests here hold the cases of those to the kernels that they
name."""
import re

import pytest

import test_gpu_f32_gemm
import test_gpu_w4a16_row_tiles
import test_gpu_w4a16_slabs
from host_runtime import host  # noqa: F401

PLANES = ["gemm_bf16_plain_kernel", "t0mi_splitk_reduce"]


@pytest.mark.parametrize("layout", ["NT", "NN"])
@pytest.mark.parametrize("m,k,n", [(128, 1024, 1024), (256, 1024, 1024), (100, 1032, 1032)])
def test_split_two_writes_y_after_the_operands_are_read(host, m, k, n, layout):
    """64x64 tiles in two K partitions: summed inside the launch, which stores a tile of Y while others
    read X and B; so planes and a reduce where Y meets X or B by so much as one row's end."""
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
        (cfg, X, B, B + bb, 0)]],
    over=[names(rt.gemm, c, x, b, y, m, n, k, z) for c, x, b, y, z in [
        (cfg, X, B, X, 0), (bias, X, B, B, BIAS), (cfg, X, B, X + xb - 16, 0), (cfg, X, B, X - yb + 16, 0),
        (cfg, X, B, B + bb - 16, 0)]],
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


MEMORY = """
def call(f, *args):
    "The kernels of a call, its error text (None: it returned OK) and the library's text after it."
    hip.fake_launches()
    try:
        f(*args)
        e = None
    except t0mi.T0miError as x:
        e = str(x)
    return [[l[0].split("<")[0] for l in launches()], e, t0mi.last_error()]
cfg = t0mi.auto_select_layout(128, 1024, 1024, t0mi.NT, t0mi.OUT_BF16)
spec = t0mi.tile_auto_select(128, 1024, 1024, t0mi.NT)
calls = dict(
    f32=lambda: call(rt.matmul, X, B, Y, 512, 1024, 517),        # one piece: needs no slots
    f32_pieces=lambda: call(rt.matmul, X, B, Y, 40, 1000, 300),  # K pieces
    gemm=lambda: call(rt.gemm, cfg, X, B, Y, 128, 1024, 1024),   # two K partitions
    tile=lambda: call(rt.tile_gemm, spec, X, B, Y, 128, 1024, 1024),
    w4=lambda: call(rt.w4a16_gemm, X, B, 5 << 40, 0, 8, Y, 100, 8192, 520, 128),  # K planes, row tiles
)
try:
    rt.matmul(X + 4, B, Y, 8, 8, 8)
except t0mi.T0miError:
    pass
before = t0mi.last_error()
assert "aligned" in before
"""


def test_routes_with_memory(host):
    r = host(MEMORY + "done({n: f() for n, f in calls.items()})")
    assert {n: c[0] for n, c in r.items()} == {
        "f32": ["t0mi_fill_kernel", "gemm_f32_kernel"],  # the exchange's counters are made by the first call
        "f32_pieces": ["gemm_f32_kernel"],
        "gemm": ["gemm_bf16_exchange_kernel"],
        "tile": ["gemm_bf16_exchange_kernel"],
        "w4": ["w4a16_decode_v2", "t0mi_splitk_reduce"],
    }
    assert all(c[1] is None for c in r.values())


@pytest.mark.parametrize("limit", [8 << 20, 400 << 10])
def test_no_memory_for_an_optional_buffer(host, limit):
    """Out of memory for buffers that a call can do without: it takes its other route, or the same one if it
    does not use them, returns OK, and leaves the library's error text as it was.  (HIP's last error, if
    the failed allocation stayed in it, would fail the launch check.)"""
    r = host(MEMORY + f"""
rt.matmul(X, B, Y, 4096, 1024, 4096)  # makes the conversion passes' buffer
if {limit} < 1 << 20:
    del calls["gemm"]  # its partial planes have to fit
hip.fake_set_malloc_limit({limit})
out = {{n: f() for n, f in calls.items()}}
done([before, out])
""")
    before, out = r
    assert all(c[1] is None and c[2] == before for c in out.values()), out
    assert out["f32"][0][-1] == "gemm_f32_kernel"
    assert out["f32_pieces"][0] == ["cvt_bf16_kernel"] * 2 + out["f32_pieces"][0][2:]
    if limit < 1 << 20:  # no workspace for planes either
        assert out["tile"][0] == ["gemm_bf16_plain_kernel"]
        assert out["w4"][0] == ["w4a16_decode_v2", "t0mi_splitk_reduce"] * 2
    else:
        assert out["gemm"][0] == out["tile"][0] == PLANES


def test_first_call_under_capture(host):
    """Buffers that may not grow now: as above, and the captured calls return OK."""
    r = host(MEMORY + """
calls = {n: calls[n] for n in ("f32", "tile")}
rt.capture_begin()
out = {n: f() for n, f in calls.items()}
rt.capture_end()
done([before, out])
""")
    before, out = r
    assert all(c[1] is None and c[2] == before for c in out.values()), out
    assert out["f32"][0] == ["gemm_f32_kernel"] and out["tile"][0] == ["gemm_bf16_plain_kernel"]


@pytest.mark.parametrize("call,warm,then", [
    ("lambda m: rt.matmul(X, B, Y, m, 4230, 522)", 1659, 1004),            # passes below the one launch
    ("lambda m: rt.matmul_with_wt_bf16(X, B, Y, m, 4096, 4096)", 16, 1),   # the persistent decode
    ("lambda m: rt.matmul_with_wt_bf16(X, B, Y, m, 4376, 2912)", 38, 37),  # the scheduled GEMM's planes
    ("lambda m: rt.matmul_backward_data(X, B, Y, m, 688, 1529)", 1037, 933),
    ("lambda k: rt.matmul_backward_weight(X, B, Y, 6350, k, 522)", 1257, 1052),  # the layer's width
])
def test_smaller_batches_captured_after_the_largest(host, call, warm, then):
    """A call runs once at its largest batch, in one launch; at a smaller batch, captured, it takes the
    conversion passes, whose buffers the first call made as well."""
    r = host(f"""
call = {call}
a = names(call, {warm})
rt.capture_begin()
b = names(call, {then})
rt.capture_end()
done([a, b])
""")
    assert r[0][-1] == "gemm_f32_kernel" and r[1][0].startswith("cvt_bf16"), r


def test_split_k_planes_run_the_kernel_without_the_epilogue(host):
    """Every prebuilt tile but single waves of up to 64x64 writes its planes with gemm_bf16_plain_kernel (the
    256x256 ping-pong kernel has its own); the chain then runs in the reduce."""
    r = host("""
import re
out, buf = [], ctypes.create_string_buffer(1 << 16)
t0mi.lib().t0mi_gemm_variants(buf, len(buf))
for name in buf.value.decode().split(","):
    v = [int(x) for x in re.findall("[0-9]+", name)] + [int(name.endswith("_nn"))]
    cfg = t0mi.GemmConfig(tile_m=v[0], tile_n=v[1], tile_k=v[2], wave_m=v[3], wave_n=v[4], stages=v[5], transpose=v[6],
                          wg_size=64 * v[3] * v[4], use_lds=1, double_buffer=1, n_col_passes=1, swap_grid=1, split_k=4,
                          epilogue=t0mi.EPI_BIAS_ADD_RELU)
    rt.gemm(cfg, X, B, Y, 256, 512, 2048, BIAS)
    out.append([v, [l[0].split("<")[0] for l in launches() if "fill" not in l[0]]])
done(out)
""")
    assert len(r) > 60
    for (bm, bn, bk, wm, wn, st, nn), k in r:
        pingpong = (bm, bn, bk, wm, wn, st) == (256, 256, 64, 2, 4, 2)
        one = wm * wn == 1 and bm * bn <= 64 * 64
        want = "gemm_bf16_pingpong_kernel" if pingpong else "gemm_bf16_kernel" if one else "gemm_bf16_plain_kernel"
        assert k == [want, "t0mi_splitk_reduce"], (bm, bn, bk, wm, wn, st, nn)


def test_dispatch_with_y_of_less_alignment(host):
    """A raw dispatch does not ask for a Y aligned to 16 bytes: bf16 there takes the kernel that asks itself."""
    r = host("""
out = []
for o in (t0mi.OUT_F32, t0mi.OUT_BF16):
    c = t0mi.preset("tile_128x64_k32").copy(out_dtype=o)
    for y in (Y, Y + 8):
        hip.fake_launches()
        rt.dispatch(rt.kernel(c), t0mi.compute_grid_auto(c, 256, 128), t0mi.build_kernargs(X, B, y, 64, 128, 256, c), False)
        out.append([l[0].split("<")[0] for l in launches()])
done(out)
""")
    plain, both = ["gemm_bf16_plain_kernel"], ["gemm_bf16_kernel"]
    assert r == [plain, plain, plain, both]


@pytest.mark.parametrize("m,n,k", [(9, 2584, 320), (16, 240, 4736), (1, 4096, 512)])
def test_tile_spec_of_few_rows_runs_the_schedule(host, m, n, k):
    """NT of up to 16 rows: the ranked schedule, not the decode kernel that run_gemm_auto has for them."""
    r = host(f"""
spec = t0mi.tile_preset("tile_64x64_k16")
rt.tile_gemm(spec, X, B, Y, {m}, {n}, {k})  # buffers are made
done(names(rt.tile_gemm, spec, X, B, Y, {m}, {n}, {k}))
""")
    assert r and all(x in ("gemm_bf16_plain_kernel", "gemm_bf16_exchange_kernel", "t0mi_splitk_reduce") for x in r), r


def test_tile_spec_keeps_its_tile_for_short_k(host):
    """Short K, where the ranking picks tiles of 128 and 256 rows, too few to fill the chip."""
    r = host("""
spec = t0mi.tile_preset("tile_64x64_k16")
out = []
for m, n, k, nn in [(1527, 672, 32, 1), (277, 4240, 16, 1), (1998, 2432, 136, 1), (2314, 1736, 200, 1),
                    (321, 2896, 48, 1), (1423, 1760, 88, 1), (100, 1000, 40, 1)]:
    head = t0mi.auto_gemm_plan(m, n, k, nn, t0mi.OUT_F32)[0]
    hip.fake_launches()
    rt.tile_gemm(spec.copy(transpose=nn), X, B, Y, m, n, k)
    out.append([head.tile_m, k, [l[0] for l in launches() if "fill" not in l[0]]])
done(out)
""")
    assert [x[0] for x in r] == [256, 256, 256, 256, 128, 128, 64], r
    for tile_m, k, names in r:
        own = k <= {256: 160, 128: 64}.get(tile_m, 0)
        assert (names[0].split("<")[1].split(",")[:3] == ["64", "64", "16"]) == own, (tile_m, k, names)


def test_outputs_without_a_chain_run_the_kernels_without_its_code(host):
    """Every prebuilt tile (but the ping-pong kernel's) and the persistent tile loops: with the epilogue's code
    and registers a chainless call lost up to half its waves."""
    r = host("""
def run(f, *args):
    f(*args)
    return [l[0] for l in launches()]
out = []
for v in t0mi.variants():
    for o in (t0mi.OUT_F32, t0mi.OUT_BF16):
        for e in (t0mi.EPI_STORE_F32, t0mi.EPI_BIAS_ADD_RELU):
            c = v.copy(out_dtype=o, epilogue=e)
            out.append([(v.tile_m, v.tile_n, v.tile_k, v.wave_m, v.wave_n) == (256, 256, 64, 2, 4) and v.stages == 0,
                        o, e, run(rt.gemm, c, X, B, Y, 256, 512, 2048, BIAS)])
loops = []
for p in ("tile_persistent_decode", "tile_persistent_128x64_k32", "tile_persistent_256x128_k32"):
    for o in (t0mi.OUT_F32, t0mi.OUT_BF16):
        for e in ([], [t0mi.BIAS_ADD]):
            s = t0mi.tile_preset(p).copy(out_dtype=o, epilogue=e)
            loops.append([o, bool(e), run(rt.tile_gemm, s, X, B, Y, 256, 512, 2048, BIAS)])
done([out, loops])
""")
    assert len(r[0]) > 240
    for pingpong, o, e, k in r[0]:
        want = "gemm_bf16_pingpong_kernel" if pingpong else "gemm_bf16_kernel" if e else "gemm_bf16_plain_kernel"
        assert len(k) == 1 and k[0].split("<")[0] == want, k
        assert e or pingpong or k[0].endswith(f",(TileSums){1 + o}>"), k
    for o, e, k in r[1]:
        assert len(k) == 1 and k[0].startswith("gemm_bf16_persistent_kernel<"), k
        assert k[0].endswith(f",(TileSums){0 if e else 1 + o}>"), k


@pytest.mark.parametrize("layout", ["NT", "NN"])
def test_tile_spec_writes_y_after_the_operands_are_read(host, layout):
    """Y over X or B, all of it inside the spec's one tile: that tile's kernel, which stores Y after its
    last read; the ranked schedule would cut it into several."""
    r = host(f"""
spec = t0mi.tile_preset("tile_128x128_k32").copy(transpose=t0mi.{layout}, out_dtype=t0mi.OUT_BF16)
def run(y):
    rt.tile_gemm(spec, X, B, y, 128, 128, 128)
    return [l[0] + " %d" % (l[1] * l[2]) for l in launches()]
rt.tile_gemm(spec, X, B, Y, 128, 128, 128)
hip.fake_launches()
done([run(Y), run(X), run(B), run(X + 128 * 128 * 2 - 16), run(X + 128 * 128 * 2)])
""")
    own = f"gemm_bf16_plain_kernel<128,128,32,2,2,2,{str(layout == 'NN').lower()},(TileSums)2> 1"
    assert r[0] == r[4] != [own]
    assert r[1] == r[2] == r[3] == [own]


def test_w4a16_row_tiles_apart_from_the_operands(host):
    """A weight of one 64-column strip, up to 64 rows: one workgroup reads everything and then stores Y, which
    may lie over an operand; side by side, one row tile's Y would lie over another's activations."""
    r = host("""
m, k, n, group = 64, 128, 64, 128  # four slabs in one launch
S, Z = 5 << 40, 6 << 40
def grid(y, z=Z):
    rt.w4a16_gemm(X, B, S, z, 8, y, m, k, n, group, t0mi.OUT_F32)
    return launches()[-1][1:4]
grid(Y)
done(dict(apart=[grid(Y), grid(X + m * k * 2), grid(Y, 0)],
          over=[grid(y) for y in (X, X + m * k * 2 - 16, B, S, Z)]))
""")
    assert r["apart"] == [[1, 1, 4]] * 3
    assert r["over"] == [[1, 1, 1]] * 5


def test_every_preset_has_its_own_tile_under_capture(host):
    r = host("""
out = []
for p in t0mi.tile_preset_names():
    for nn in range(2):
        spec = t0mi.tile_preset(p).copy(transpose=nn)
        if spec.persistent:
            continue
        rt.capture_begin()
        rt.tile_gemm(spec, X, B, Y, 128, 1032, 1032)
        rt.capture_end()
        out.append([[spec.tile_m, spec.tile_n, spec.tile_k, nn], [l[0] for l in launches()]])
done(out)
""")
    assert len(r) == 46
    for (m, n, k, nn), names in r:
        bk = 64 if k % 64 == 0 else 32 if k % 32 == 0 else 16
        assert len(names) == 1
        assert names[0].startswith(f"gemm_bf16_plain_kernel<{m},{max(n, 64) if nn else n},{bk},"), (m, n, k, nn, names)


def test_w4a16_cases_run_the_kernels_they_name(host):
    cases = [c[:4] for c in test_gpu_w4a16_slabs.CASES + test_gpu_w4a16_row_tiles.CASES]
    r = host(f"""
out = []
for m, k, n, group in {[list(c) for c in cases]}:
    hip.fake_launches()
    rt.w4a16_gemm(X, B, 5 << 40, 6 << 40, 8, Y, m, k, n, group, t0mi.OUT_F32)
    out.append([l for l in launches() if l[0].startswith("w4a16")])
done(out)
""")
    after, side, planes = {}, {}, set()
    for (m, k, n, group), ls in zip(cases, r):
        for name, _, gy, gz, _ in ls:
            t = re.fullmatch(r"w4a16_decode_v2<(.*)>", name).group(1).split(",")
            slabs, tiles = int(t[5]), t[7] == "true"
            assert int(t[2]) * 32 == group and tiles == (gz > 1)
            (side if tiles else after).setdefault(group, set()).add(slabs)
            if gy > 1:
                planes.add((slabs > 1, tiles))
    assert after == {32: {3}, 64: {3}, 128: {2, 3, 4}, 256: {1, 2}}
    assert side == {32: {1, 3}, 64: {1, 2}, 128: {1, 2, 3, 4}, 256: {1, 2}}
    assert planes == {(True, False), (False, True), (True, True)}


def test_f32_cases_run_the_tiles_they_name(host):
    r = host(f"""
def kernel(f):
    hip.fake_launches()
    f()
    l = launches()[-1]
    return l[:2] if l[0].startswith("gemm_f32") else None
out = []
for m, n, k in {[list(c) for c in test_gpu_f32_gemm.SHAPES]}:
    out += [kernel(lambda: rt.matmul(X, B, Y, m, k, n)), kernel(lambda: rt.matmul_backward_data(X, B, Y, m, n, k)),
            kernel(lambda: rt.matmul_backward_weight(X, B, Y, k, m, n))]
done([out, [kernel(lambda: rt.matmul_with_wt_bf16(X, B, Y, m, k, n)) + [m, n]
            for m, n, k in {[list(c) for c in test_gpu_f32_gemm.WT_SHAPES]}]])
""")
    products, wt = r
    seen = {p[0] for p in products if p}
    tiles = ["32,32", "64,32", "64,64", "128,64", "128,128"]
    for t in tiles:
        for mode in ("false,true", "false,false", "true,true"):  # forward, data, weight
            assert any(s.startswith(f"gemm_f32_kernel<{t},") and s.endswith(f",{mode},false>") for s in seen), (t, mode)
    got = set()
    for name, grid, m, n in wt:
        bm, bn = [int(v) for v in re.match(r"gemm_f32_kernel<(\d+),(\d+),", name).groups()]
        got.add((bm, grid > -(-m // bm) * -(-n // bn)))
    assert got == {(32, False), (32, True), (64, False), (64, True)}  # one piece, several
