"""The persistent four-wave kernel on tiles of 128, 160, 192 and 224 rows x 256 columns, of 288 x 224 and of 128 and 160 x 192: exact results at the
edges of the tiles (GPU), and what the plan takes them for (CPU).  Bar: 16-bit outputs bit-exact against the oracle."""
import numpy as np
import pytest

from ms_custom_ops_amd import cabi
from oracle import gmm_oracle as O

ROWS = {cabi.OV_W4_128: 128, cabi.OV_W4_160: 160, cabi.OV_W4_192: 192, cabi.OV_W4_224: 224, cabi.OV_W4_288: 288,
        cabi.OV_W4_128x192: 128, cabi.OV_W4_160x192: 160}
LAYOUTS = ["packed", "nk", "kn"]


def _run(seed, rows, k, n, override, layout, *, out="bf16", act=0):
    from gpu_utils import run_w8a8
    rng = np.random.default_rng(seed)
    e, m = len(rows), sum(rows)
    x, w = rng.integers(-128, 128, (m, k), dtype=np.int8), rng.integers(-128, 128, (e, k, n), dtype=np.int8)
    bias = rng.integers(-1000, 1001, (e, n)).astype(np.int32)
    scale, pt = rng.uniform(1e-3, 1e-2, (e, n)).astype(np.float32), rng.uniform(1e-3, 1e-2, m).astype(np.float32)
    ends = np.cumsum(rows)
    got, info = run_w8a8(x, w, ends, bias, scale, pt, out=out, override=override, transpose_b=layout == "nk", packed=layout == "packed",
                         act_type=act, launches=2)
    return got, info, (x, w, ends, bias, scale, pt)


@pytest.mark.gpu
@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("override", list(ROWS))
@pytest.mark.parametrize("k,n", [(512, 80), (656, 464), (1040, 1008)])   # fewest K slabs; K and N tails: columns of one wave, of both, several tiles
def test_exact_at_the_edges(device, override, layout, k, n):
    h = ROWS[override]
    rows = [h, 0, 1, h + 1, h - 1, 17, 2 * h, h // 2, h // 2 + 1]
    got, info, args = _run(k + n, rows, k, n, override, layout)
    want = O.grouped_matmul_w8a8(*args)
    assert "256x256x128_w4" in info and (("tile_rows=%d" % h) in info) == (h != 288 or layout != "kn"), info
    assert np.array_equal(got, np.asarray(want).view(np.uint16)), info


@pytest.mark.gpu
@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("override", list(ROWS))
def test_more_tiles_than_compute_units(device, override, layout):
    # the operand stream of a tile's last slabs runs into the next tile, in another group or panel; float16
    got, info, args = _run(7, [700, 300, 90, 2050], 576, 5200, override, layout, out="f16")
    want = O.grouped_matmul_w8a8(*args, out_dtype="f16")
    assert np.array_equal(got, np.asarray(want).view(np.uint16)), info


@pytest.mark.gpu
@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("override", list(ROWS))
def test_silu_equals_the_256_row_tile(device, override, layout):
    a, _, _ = _run(11, [150, 320], 640, 528, override, layout, act=cabi.ACT_SILU)
    b, info, _ = _run(11, [150, 320], 640, 528, cabi.OV_TILE_256_W4, layout, act=cabi.ACT_SILU)
    assert "tile_rows" not in info and np.array_equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("override", list(ROWS))
@pytest.mark.parametrize("form", ["bf16", "u64", "shared", "scalar", "bare"])
def test_forms_of_the_epilogue_operands(device, form, override, layout):
    # the tables of a tile: bfloat16 scales are widened in place, 64-bit ones read every other word, one row or one value for all
    # groups, no scale per token (288 rows: the second pass of the first wave writes the ones); two tiles per workgroup's table or more
    from gpu_utils import run_w8a8
    h, k, n = ROWS[override], 528, 2320
    rows = [h, 0, h - 1, 2 * h + 1, 16, 700]
    rng = np.random.default_rng(h + len(form))
    e, m = len(rows), sum(rows)
    x, w = rng.integers(-128, 128, (m, k), dtype=np.int8), rng.integers(-128, 128, (e, k, n), dtype=np.int8)
    scale, pt = rng.uniform(1e-3, 1e-2, (e, n)).astype(np.float32), rng.uniform(1e-3, 1e-2, m).astype(np.float32)
    bias = rng.integers(-1000, 1001, (e, n)).astype(np.int32) if form in ("bf16", "u64") else None
    given, kw = scale, {}
    if form == "bf16":
        given = O.f32_to_bf16_bits(scale)
        scale, kw = O.bf16_bits_to_f32(given), dict(scale_dtype=cabi.DT_BF16)
    elif form == "u64":
        given, kw = O.encode_scale_int64(scale), dict(scale_dtype=cabi.DT_U64)
    elif form in ("shared", "scalar"):
        given, kw = (scale[0], dict(scale_per_group=0)) if form == "shared" else (scale[0, :1], dict(scale_per_group=0, scale_is_scalar=1))
        scale = np.broadcast_to(given, (e, n))
    if form in ("bf16", "scalar", "bare"):
        pt = None
    ends = np.cumsum(rows)
    got, info = run_w8a8(x, w, ends, bias, given, pt, override=override, transpose_b=layout == "nk", packed=layout == "packed", launches=2, **kw)
    want = O.grouped_matmul_w8a8(x, w, ends, bias, scale, pt)
    assert "256x256x128_w4" in info and np.array_equal(got, np.asarray(want).view(np.uint16)), info


@pytest.mark.gpu
@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("override", list(ROWS))
def test_fast_gelu_equals_the_256_row_tile(device, override, layout):
    a, _, _ = _run(12, [150, 320], 640, 528, override, layout, act=cabi.ACT_FAST_GELU, out="f16")
    b, info, _ = _run(12, [150, 320], 640, 528, cabi.OV_TILE_256_W4, layout, act=cabi.ACT_FAST_GELU, out="f16")
    assert "tile_rows" not in info and np.array_equal(a, b)


def _plan(m, k, n, e, layout, *, out=cabi.DT_BF16, act=0):
    op = cabi.GmmOp(x_dtype=cabi.DT_I8, out_dtype=out, scale_dtype=cabi.DT_NONE if out == cabi.DT_I32 else cabi.DT_F32, transpose_b=int(layout == "nk"), act_type=act,
                    weight_layout=int(layout == "packed"), **({} if e == 1 else dict(group_list_dtype=cabi.DT_I64)))
    op.plan(m, k, n, e)
    info = op.plan_info()
    op.close()
    return info


@pytest.mark.gpu
@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("rows", [[256] * 4, [288, 280, 270, 186], [128, 128, 128, 640], [1024, 0, 0, 0], [0, 161, 383, 470], [1, 1, 1, 1]])
def test_shape_picked_from_the_groups(device, layout, rows):
    # one plan, group lists that the device gives different tiles; rows past the last boundary stay untouched
    from gpu_utils import run_w8a8
    rng = np.random.default_rng(5)
    m, k, n, e = 1024, 512, 14336, 4
    x, w = rng.integers(-128, 128, (m, k), dtype=np.int8), rng.integers(-128, 128, (e, k, n), dtype=np.int8)
    scale, pt = rng.uniform(1e-3, 1e-2, (e, n)).astype(np.float32), rng.uniform(1e-3, 1e-2, m).astype(np.float32)
    got, info = run_w8a8(x, w, rows, None, scale, pt, transpose_b=layout == "nk", packed=layout == "packed", group_list_type=1, launches=2)
    assert "tile_rows=by_groups" in info, info
    ends = np.cumsum(rows)
    want = np.asarray(O.grouped_matmul_w8a8(x, w, ends, None, scale, pt)).view(np.uint16)
    assert np.array_equal(got[:ends[-1]], want[:ends[-1]]) and (got[ends[-1]:] == 0x7FC0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("bad,good,kind", [([300, 200, 5000, 1024], [300, 300, 1024, 1024], 0), ([-5, 512, 100, 700], [0, 512, 512, 700], 0),
                                           ([300, 2000, 5, 7], [300, 1024, 1024, 1024], 1), ([-3, 10, 2 ** 40, 1], [0, 10, 1024, 1024], 1)])
def test_shape_picked_from_malformed_groups(device, layout, bad, good, kind):
    # decreasing boundaries, negative ones, ones past the last row: the tiles are counted from the clamped ranges that the kernel walks
    from gpu_utils import run_w8a8
    rng = np.random.default_rng(8)
    m, k, n, e = 1024, 512, 14336, 4
    x, w = rng.integers(-128, 128, (m, k), dtype=np.int8), rng.integers(-128, 128, (e, k, n), dtype=np.int8)
    scale = rng.uniform(1e-3, 1e-2, (e, n)).astype(np.float32)
    kw = dict(transpose_b=layout == "nk", packed=layout == "packed")
    got, info = run_w8a8(x, w, bad, None, scale, None, group_list_type=kind, **kw)
    assert "tile_rows=by_groups" in info, info
    want = np.asarray(O.grouped_matmul_w8a8(x, w, good, None, scale, None)).view(np.uint16)
    assert np.array_equal(got[:good[-1]], want[:good[-1]]) and (got[good[-1]:] == 0x7FC0).all()


@pytest.mark.gpu
def test_shape_picked_over_more_than_64_groups(device):
    from gpu_utils import run_w8a8
    rng = np.random.default_rng(6)
    e, k, n = 70, 512, 2064
    rows = rng.integers(0, 500, e)
    rows[3], rows[68] = 0, 900
    m = int(rows.sum())
    x, w = rng.integers(-128, 128, (m, k), dtype=np.int8), rng.integers(-128, 128, (e, k, n), dtype=np.int8)
    scale, pt = rng.uniform(1e-3, 1e-2, (e, n)).astype(np.float32), rng.uniform(1e-3, 1e-2, m).astype(np.float32)
    got, info = run_w8a8(x, w, np.cumsum(rows), None, scale, pt, packed=True, launches=2)
    assert "tile_rows=by_groups" in info, info
    assert np.array_equal(got, np.asarray(O.grouped_matmul_w8a8(x, w, np.cumsum(rows), None, scale, pt)).view(np.uint16))


@pytest.mark.gpu
def test_shape_picked_over_hundreds_of_groups(device):
    # more than 256 packed groups of just more than 256 rows on average, some of them in the second launch: the bits of 256 x 256 tiles
    from gpu_utils import run_w8a8
    rng = np.random.default_rng(9)
    e, k, n = 300, 2048, 80
    rows = rng.poisson(290, e) * (rng.random(e) < 0.9)
    rows[:5] = [0, 1, 64, 65, 900]
    rows[-1] += e * 270 - rows.sum()
    assert rows[-1] > 0
    m = int(rows.sum())
    x, w = rng.integers(-128, 128, (m, k), dtype=np.int8), rng.integers(-128, 128, (e, k, n), dtype=np.int8)
    scale, pt = rng.uniform(1e-3, 1e-2, (e, n)).astype(np.float32), rng.uniform(1e-3, 1e-2, m).astype(np.float32)
    a, info = run_w8a8(x, w, np.cumsum(rows), None, scale, pt, packed=True, launches=2)
    assert "tile_rows=by_groups" in info and "small_groups=64" in info, info
    b, info = run_w8a8(x, w, np.cumsum(rows), None, scale, pt, packed=True, override=cabi.OV_TILE_256_W4)
    assert "tile_rows" not in info and np.array_equal(a, b)


@pytest.mark.parametrize("m,k,n,e,layout,rows", [
    (2048, 4096, 11008, 1, "nk", "192"), (2048, 4096, 11008, 1, "packed", "192"),    # 344 tiles of 256 rows, 473 of 192: two rounds either way
    (16384, 4096, 14336, 1, "nk", ""),                                               # many rounds: the tile that reads least
    (2029, 3040, 2896, 1, "nk", "128"),                                              # one round of 192 tiles in place of 128 x 256 ones
    (2048, 4096, 14336, 8, "packed", "by_groups"), (4096, 4096, 14336, 8, "kn", "by_groups"),
    (8192, 4096, 14336, 8, "kn", "")])                                               # several groups, many rounds
def test_the_plan(m, k, n, e, layout, rows):
    info = _plan(m, k, n, e, layout)
    assert "tile_256x256x128_w4" in info and (("tile_rows=" + rows) in info if rows else "tile_rows" not in info), info


@pytest.mark.parametrize("kwargs", [dict(out=cabi.DT_I32), dict(act=cabi.ACT_RELU), dict(act=cabi.ACT_GELU_TANH)])
def test_outputs_that_stay_on_256_rows(kwargs):
    assert "tile_rows" not in _plan(2048, 4096, 11008, 1, "nk", **kwargs)


@pytest.mark.parametrize("rows", [257, 296])
def test_groups_just_beyond_256_rows(rows):
    assert "tile_rows=by_groups" in _plan(8 * rows, 4096, 14336, 8, "packed")
    for kwargs in (dict(act=cabi.ACT_RELU), dict(out=cabi.DT_I32)):   # (256 x 256 tiles only: equal chunks of up to 160 rows)
        assert "rows160" in _plan(8 * rows, 4096, 14336, 8, "packed", **kwargs)
    assert "rows160" in _plan(8 * 297, 4096, 14336, 8, "packed")


def test_planning_takes_no_longer_for_many_groups():
    # a server plans anew for every row count: the skewed routings that the plan looks at are not added up group by group (1024 groups took 15 times
    # what 64 take; 4 is far from either side's noise)
    import ctypes
    import time

    plan = cabi.load().msco_gmm_plan
    best = {}
    for e in (64, 1024):
        op = cabi.GmmOp(x_dtype=cabi.DT_I8, out_dtype=cabi.DT_BF16, scale_dtype=cabi.DT_F32, transpose_b=1, group_list_dtype=cabi.DT_I64)
        ws, times = ctypes.c_size_t(0), []
        for step in range(200):
            began = time.perf_counter()
            plan(op._h, 40 * e + step, 4096, 2048, e, ctypes.byref(ws))
            times.append(time.perf_counter() - began)
        assert "by_groups" in op.plan_info()   # (the comparison with smaller tiles was made)
        best[e] = min(times)
        op.close()
    assert best[1024] < 4 * best[64]


@pytest.mark.parametrize("e,rows,k,n,by_groups", [
    (16, 270, 2048, 8192, True), (16, 270, 2048, 8208, False), (16, 296, 2800, 8208, False), (16, 270, 2816, 8208, True),   # four chunk workgroups per CU; a long K
    # 256 x 256 tiles that make more than six rounds
    (64, 270, 2048, 3584, False), (128, 270, 2048, 1792, False), (32, 270, 2048, 7168, False), (256, 270, 2048, 528, False),
    (16, 270, 4096, 14336, True), (64, 270, 4096, 4096, True),
    (257, 270, 2048, 512, True), (1000, 290, 4096, 400, True),                                        # more than 256 groups: shapes, whatever the rounds
    (1100, 270, 2048, 512, False)])
def test_chunks_of_groups_beyond_256_rows(e, rows, k, n, by_groups):
    # (out of the chunk kernels only into shapes that are picked from the groups)
    info = _plan(e * rows, k, n, e, "packed")
    assert ("tile_rows=by_groups" if by_groups else "rows160") in info, info


def test_more_groups_than_the_persistent_kernel_takes():
    assert "256x256x64" in _plan(1100 * 270, 2048, 496, 1100, "packed")


def test_a_forced_k_split_keeps_the_chunks():
    op = cabi.GmmOp(x_dtype=cabi.DT_I8, out_dtype=cabi.DT_BF16, scale_dtype=cabi.DT_F32, weight_layout=cabi.WL_PACKED, group_list_dtype=cabi.DT_I64, force_split_k=1)
    op.plan(8 * 270, 4096, 8192, 8)
    assert "rows160" in op.plan_info()   # (no shape is picked then)
    op.close()


# The shape with the least modelled time: one whole round of the chip where only that shape makes one.  (columns, rows of the groups, groups of up to so
# many rows left out, index into the shapes)
ONE_ROUND = [(4096, [256] * 16, 0, 0), (4096, [224] * 16, 0, 1), (4096, [192] * 16, 0, 2), (4096, [160] * 16, 0, 3), (4096, [128] * 16, 0, 4),
             (14336, [288] * 8, 0, 5), (14336, [257] * 8, 0, 5), (3072, [128] * 16, 0, 6), (3072, [160] * 16, 0, 7),
             (512, [128] * 128, 0, 4), (512, [0] * 70 + [224] * 128, 0, 1),                                     # more than 64 groups
             (4096, [224] * 16 + [64] * 100, 64, 1), (4096, [224] * 16 + [64] * 100, 0, 4), (4096, [0] * 8, 0, 0)]   # a second launch's groups do not count


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("n,rows,rows_lo,index", ONE_ROUND)
def test_the_pick(layout, n, rows, rows_lo, index):
    got = cabi.probe_tile_pick_host(["kn", "nk", "packed"].index(layout), 4096, n, rows, rows_lo)
    assert got == index if index != 5 or layout != "kn" else got == 3   # (no 288 x 224 on [E,K,N])


@pytest.mark.gpu
@pytest.mark.parametrize("layout", [0, 1, 2])
def test_the_device_picks_as_the_host(device, layout):
    # outputs do not show the shape; the kernel's counting (two counts to a sum, 64 groups at a time, clamped boundaries) and its rule do, on one wavefront
    import torch
    rng = np.random.default_rng(layout)
    cases = [(n, rows, lo, np.cumsum(rows), 0, sum(rows)) for n, rows, lo, _ in ONE_ROUND]
    for _ in range(60):
        e, n = int(rng.choice([1, 2, 8, 63, 64, 65, 128, 300, 1024])), 16 * int(rng.integers(32, 900))
        rows = (rng.gamma(rng.choice([0.3, 2.0, 20.0]), 1.0, e) * rng.choice([2, 15, 60])).astype(np.int64)
        kind = int(rng.integers(2))
        cases.append((n, rows, int(rng.choice([0, 64])), rows if kind else np.cumsum(rows), kind, int(rows.sum()) + int(rng.integers(3))))
    cases += [(14336, [300, 0, 724, 0], 0, [300, 200, 5000, 1024], 0, 1024), (14336, [300, 724, 0, 0], 0, [300, 2000, 5, 7], 1, 1024)]
    st, seen = torch.cuda.current_stream().cuda_stream, set()
    for n, rows, lo, given, kind, m in cases:
        choice, gl = torch.full((1,), -1, dtype=torch.int32, device="cuda:0"), torch.from_numpy(np.asarray(given, dtype=np.int64)).to("cuda:0")
        cabi.probe_tile_pick(layout, m, 512, n, len(rows), lo, gl.data_ptr(), kind, choice.data_ptr(), st)
        want = cabi.probe_tile_pick_host(layout, 512, n, rows, lo)
        assert int(choice.item()) == want, (n, list(rows)[:8], lo, kind)
        seen.add(want)
    assert seen == set(range(8)) - ({5} if layout == 0 else set())
    with pytest.raises(cabi.BackendError):
        cabi.probe_tile_pick(layout, 128, 512, 512, 1025, 0, gl.data_ptr(), 0, choice.data_ptr(), st)
