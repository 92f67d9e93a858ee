"""K slices of the small tiles: which split the plan takes where the tiles of an XCD (an eighth of all, rounded up) with their slices just fit its 32
CUs and where they just do not.  256 CUs."""
import re

import pytest

from ms_custom_ops_amd import cabi


def _plan(m, k, n, e=1, nk=False, packed=False):
    op = cabi.GmmOp(x_dtype=cabi.DT_I8, weight_dtype=cabi.DT_I8, out_dtype=cabi.DT_BF16, scale_dtype=cabi.DT_F32, scale_per_group=1, transpose_b=int(nk),
                    weight_layout=cabi.WL_PACKED if packed else cabi.WL_ROW_MAJOR, **({} if e == 1 else dict(group_list_dtype=cabi.DT_I64)))
    try:
        op.plan(m, k, n, e)
    except cabi.BackendError:
        pass   # (a split plan allocates counters on the device; the plan itself stands)
    info = op.plan_info()
    op.close()
    return info.split("kernel=")[1].split()[0], int(re.search(r"split_k=(\d+)", info)[1])


@pytest.mark.parametrize("m,k,n,nk,packed,kernel,split", [
    (72, 2688, 5120, True, False, "w8a8_tile_64x128", 3), (72, 2688, 5280, True, False, "w8a8_tile_64x128", 2),      # 80 and 84 tiles
    (72, 2688, 5280, False, True, "w8a8_tile_64x128", 2), (244, 2912, 2688, True, False, "w8a8_tile_64x128", 2),
    (40, 16384, 6144, False, True, "w8a8_tile_64x128", 5), (40, 16384, 6272, False, True, "w8a8_tile_64x128", 4),      # 48 and 49
    (19, 4864, 8192, False, False, "w8a8_skinny_tile_32x128", 4), (19, 4864, 8320, False, False, "w8a8_skinny_tile_32x128", 3),   # 64 and 65
    (19, 4800, 8192, False, False, "w8a8_skinny_tile_32x128", 3), (23, 3616, 8048, True, False, "w8a8_skinny_tile_32x128", 3),    # four slices fill an XCD: 75 K blocks and fewer
    (4, 2272, 10240, False, False, "w8a8_skinny_tile_32x128", 3), (4, 2272, 10448, False, False, "w8a8_skinny_tile_32x128", 2)])
def test_one_group(m, k, n, nk, packed, kernel, split):
    assert _plan(m, k, n, nk=nk, packed=packed) == (kernel, split)


@pytest.mark.parametrize("m,k,n,e,split", [
    (353, 3616, 832, 32, 1), (352, 3616, 832, 32, 2),      # more than 11 rows a group and 11, 224 tiles: two to a CU cost 1.6 and 1.2 times one
    (384, 3616, 512, 32, 2), (112, 3680, 3680, 8, 1), (112, 3680, 1920, 8, 2)])
def test_several_groups_on_32_row_tiles(m, k, n, e, split):
    assert _plan(m, k, n, e) == ("w8a8_skinny_tile_32x128", split)


@pytest.mark.parametrize("m,k,n,e,kernel", [
    (6, 5760, 560, 128, "w8a8_skinny_16w"), (6, 5744, 560, 128, "w8a8_skinny_tile_32x128"),      # 30 tiles, 30 times 192 and less
    (2, 7712, 656, 16, "w8a8_skinny_16w"), (2, 4576, 1136, 16, "w8a8_skinny_16w"), (2, 3072, 1136, 16, "w8a8_skinny_tile_32x128"),
    (6, 7712, 656, 16, "w8a8_skinny_16w"), (7, 7712, 656, 16, "w8a8_skinny_tile_32x128"), (63, 7680, 528, 8, "w8a8_skinny_tile_32x128")])      # up to two rows for five experts
def test_few_tiles_and_a_long_k_stay_with_the_decode_kernels(m, k, n, e, kernel):
    assert _plan(m, k, n, e)[0] == kernel


@pytest.mark.parametrize("m,k,n,e", [(16, 8192, 1024, 1), (24, 4096, 512, 4), (8, 4192, 656, 1), (2, 8096, 1024, 1)])
def test_packed_decode_walks_k_in_one_slice(m, k, n, e):
    assert _plan(m, k, n, e, packed=True) == ("w8a8_stream", 1)
