"""The rule that takes the next tile shape where 128 x 128 or 64 x 128 tiles are just too many for one round of the chip: what it
picks at both sides of its lines (CPU), and exact results of those picks (GPU)."""
import numpy as np
import pytest

from ms_custom_ops_amd import cabi

# (rows, K, N, groups, [E,N,K], packed, what the plan names); 256 CUs
PICKS = [(720, 1024, 5632, 1, False, False, "tile_128x256"), (720, 1008, 5632, 1, False, False, "tile_128x128"),
         (640, 4096, 5632, 1, False, False, "tile_128x128"), (720, 4096, 5632, 1, True, False, "tile_128x128"),
         (720, 4096, 5632, 1, False, True, "tile_128x128"),
         (1320, 7168, 3696, 8, False, False, "tile_128x256"), (5744, 1792, 560, 8, False, False, "tile_128x128"),
         (776, 2048, 2368, 8, False, False, "tile_128x128"), (776, 2032, 2368, 8, False, False, "tile_64x128"),
         (776, 2048, 2368, 8, True, False, "tile_128x128"), (4736, 2048, 1248, 32, True, False, "tile_256x256x128_w4"),
         (4736, 2032, 1248, 32, True, False, "tile_128x128"), (4736, 2048, 1248, 32, False, False, "tile_128x256")]


def _op(m, k, n, e, nk, packed):
    op = cabi.GmmOp(x_dtype=cabi.DT_I8, weight_dtype=cabi.DT_I8, out_dtype=cabi.DT_BF16, scale_dtype=cabi.DT_F32, scale_per_group=1, transpose_b=int(nk),
                    weight_layout=cabi.WL_PACKED if packed else cabi.WL_ROW_MAJOR, **({} if e == 1 else dict(group_list_dtype=cabi.DT_I64, group_list_type=1)))
    return op, op.plan(m, k, n, e)


@pytest.mark.parametrize("m,k,n,e,nk,packed,must", PICKS)
def test_the_rule(m, k, n, e, nk, packed, must):
    op, _ = _op(m, k, n, e, nk, packed)
    assert must in op.plan_info(), op.plan_info()
    op.close()


@pytest.mark.gpu
@pytest.mark.parametrize("m,k,n,e,nk,packed,must", [p for p in PICKS if p[3] > 1 or p[1] == 1024 or p[5]])
def test_exact(device, m, k, n, e, nk, packed, must):
    import torch

    from gpu_utils import ptr, to_dev
    from oracle import gmm_oracle as O

    rng = np.random.default_rng(k + n)
    x, w = rng.integers(-128, 128, (m, k), dtype=np.int8), rng.integers(-128, 128, (e, k, n), dtype=np.int8)
    s = rng.uniform(1e-3, 1e-2, (e, n)).astype(np.float32)
    counts = rng.multinomial(m - 3, rng.dirichlet(np.full(e, 4.0))).astype(np.int64) if e > 1 else None
    tx, tw, ts = to_dev(x), to_dev(w.transpose(0, 2, 1) if nk else w), to_dev(s)
    if packed:
        src, tw = tw, torch.empty(e * cabi.packed_weight_bytes(k, n), dtype=torch.int8, device="cuda:0")
        cabi.pack_weight(src.data_ptr(), tw.data_ptr(), e, k, n)
    gl = to_dev(counts) if e > 1 else None
    op, ws = _op(m, k, n, e, nk, packed)
    assert must in op.plan_info()
    buf = torch.empty(max(ws, 1), dtype=torch.uint8, device="cuda:0")
    out = torch.full((m, n), 0x7FC0, dtype=torch.int16, device="cuda:0")
    op.launch([ptr(tx), ptr(tw), None, ptr(ts), ptr(gl) if e > 1 else None, None, None, None], out.data_ptr(), buf.data_ptr(), ws, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    op.close()
    ends = np.cumsum(counts) if e > 1 else np.array([m], dtype=np.int64)
    want = O.grouped_matmul_w8a8(x, w, ends, None, s, None)
    rows = int(ends[-1])
    assert np.array_equal(out.cpu().numpy().view(np.uint16)[:rows], np.asarray(want).view(np.uint16)[:rows])


# several groups, counted with the mean of their row tiles over random routings: both sides of the lines, and a K split that would make two rounds
@pytest.mark.parametrize("m,k,n,e,nk,must,split", [
    (1960, 4032, 1776, 8, False, "tile_128x128", 1), (2120, 4032, 1776, 8, False, "tile_128x256", 1),            # 250 and 302 tiles of 128 x 128 expected
    (920, 6400, 1712, 8, True, "tile_64x128", 1), (1016, 6400, 1712, 8, True, "tile_128x128", 1),                # 236 and 274 of 64 x 128
    (2872, 3168, 592, 16, True, "tile_128x128", 1), (2900, 6688, 544, 8, True, "tile_128x128", 2)])              # 160 and 125 of 128 x 128 instead
def test_the_rule_counts_a_mean_routing(m, k, n, e, nk, must, split):
    op = cabi.GmmOp(x_dtype=cabi.DT_I8, weight_dtype=cabi.DT_I8, out_dtype=cabi.DT_BF16, scale_dtype=cabi.DT_F32, scale_per_group=1, transpose_b=int(nk),
                    group_list_dtype=cabi.DT_I64, group_list_type=1)
    try:
        op.plan(m, k, n, e)
    except cabi.BackendError:
        pass   # (a split plan allocates counters on the device; the plan itself stands)
    info = op.plan_info()
    op.close()
    assert must in info and f"split_k={split} " in info, info
