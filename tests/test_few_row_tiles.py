"""32-row tiles of int8 activations (kernel_override 17, 18, and what the plan sends there): bit-exact against the oracle at the edges of
a tile's rows and columns, with K inside one ring of slabs, at its end and in its tail, with a K split, and over groups without rows."""
import numpy as np
import pytest

from ms_custom_ops_amd import cabi
from oracle import gmm_oracle as O

# (rows per group, K, N); two more rows of x lie behind the last group
SHAPES = [([1], 16, 16), ([32], 128, 128), ([33, 0, 31], 400, 144), ([5, 1, 0, 64, 65], 512, 272), ([0, 3] * 70, 656, 256), ([17], 2064, 1040)]


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["kn", "nk", "packed"])
@pytest.mark.parametrize("override", [cabi.OV_TILE_32x128, cabi.OV_TILE_32x256])
@pytest.mark.parametrize("split", [1, 3])
@pytest.mark.parametrize("counts,k,n", SHAPES)
def test_bit_exact(device, counts, k, n, split, override, layout):
    from gpu_utils import run_w8a8
    rng = np.random.default_rng(k + n)
    e, rows = len(counts), sum(counts)
    m = rows + 2
    x, w = rng.integers(-128, 128, (m, k), dtype=np.int8), rng.integers(-128, 128, (e, k, n), dtype=np.int8)
    bias = rng.integers(-1000, 1001, (e, n)).astype(np.int32)
    scale, pt = rng.uniform(1e-3, 1e-2, (e, n)).astype(np.float32), rng.uniform(1e-3, 1e-2, m).astype(np.float32)
    ends = np.cumsum(counts)
    form = dict(transpose_b=layout == "nk", packed=layout == "packed", override=override, force_split_k=split, launches=3)
    for out, untouched in (("bf16", 0x7FC0), ("f16", 0x7FC0), ("i32", -7777)):
        got, info = run_w8a8(x, w, ends, bias, scale, pt, out=out, **form)
        want = O.grouped_matmul_w8a8(x, w, ends, bias, *((scale, pt) if out != "i32" else ()), out_dtype=out)
        assert ("32x" in info) == (layout != "packed") and ("32x256" in info) == (layout == "kn" and override == cabi.OV_TILE_32x256), info
        assert np.array_equal(got[:rows], want[:rows].view(got.dtype)), (out, info)
        assert (got[rows:] == untouched).all(), info


def _plan(m, k, n, e, transpose_b=False, packed=False):
    op = cabi.GmmOp(x_dtype=cabi.DT_I8, weight_dtype=cabi.DT_I8, out_dtype=cabi.DT_BF16, group_list_dtype=cabi.DT_I64, scale_dtype=cabi.DT_F32,
                    scale_per_group=1, transpose_b=int(transpose_b), weight_layout=cabi.WL_PACKED if packed else cabi.WL_ROW_MAJOR)
    op.plan(m, k, n, e)
    info = op.plan_info()
    op.close()
    return info


# (m, k, n, e, transpose_b, packed, what the plan names); shapes whose K is not split, so that no device is needed
@pytest.mark.parametrize("m,k,n,e,nk,packed,must", [
    (8, 640, 36864, 1, False, False, "skinny_tile_32x128"), (8, 640, 36992, 1, False, False, "tile_64x128"), (8, 1024, 36992, 1, False, False, "skinny_tile_32x256"),
    (32, 1024, 36864, 1, True, False, "skinny_tile_32x128"), (33, 1024, 36864, 1, True, False, "tile_64x128"), (128, 2048, 7168, 8, False, False, "skinny_tile_32x256"),
    (129, 2048, 7168, 8, False, False, "tile_64x128"), (6, 1024, 8192, 64, False, False, "skinny_tile_32x256"), (5, 1024, 32768, 64, False, False, "w8a8_skinny layout"),
    (64, 1024, 8192, 64, True, False, "tile_64x128"), (8, 496, 131072, 1, False, False, "w8a8_skinny layout"), (8, 640, 36864, 1, False, True, "stream")])
def test_the_rule(m, k, n, e, nk, packed, must):
    info = _plan(m, k, n, e, nk, packed)
    assert must in info and "split_k=1 " in info, info


def test_a_launch_without_a_workspace_of_the_callers_keeps_what_it_took():
    """No split whose partial tiles do not fit the 32 MiB that such a launch brings (the groups of a malformed list count)."""
    for m, k, n, e in ((40, 8192, 1024, 40), (100, 8192, 512, 100), (2, 8192, 14336, 2)):
        op = cabi.GmmOp(x_dtype=cabi.DT_I8, weight_dtype=cabi.DT_I8, out_dtype=cabi.DT_BF16, group_list_dtype=cabi.DT_I64, scale_dtype=cabi.DT_F32, scale_per_group=1)
        try:
            op.plan(m, k, n, e)
        except cabi.BackendError:
            pass   # (a split plan allocates counters on the device; the plan itself stands)
        assert "skinny_tile_32x128" in op.plan_info() and op.workspace_bytes <= 32 << 20, op.plan_info()
        op.close()
