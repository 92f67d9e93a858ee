"""Partial tiles of the decode kernels' K split, numbered by the launch's chunk slots: how many a plan asks for (CPU), and exact results where
groups have several chunks, some none, with a guard behind the workspace (GPU)."""
import re

import numpy as np
import pytest

from ms_custom_ops_amd import cabi
from oracle import gmm_oracle as O


def _slots(m, e, rows):
    """Chunks of `rows` rows that e groups with m rows in all can have: one started chunk per group that holds rows, and m / rows full ones."""
    return max(1, min(e * max(1, -(-m // rows)), min(m, e) + m // rows))


# (16-bit x, packed, m, k, n, e, rows per chunk, columns of a partial tile, bytes of one)
@pytest.mark.parametrize("half,packed,m,k,n,e,rows,cols,tile", [
    (True, True, 294, 5120, 13200, 64, 16, 256, 17408), (True, True, 600, 5120, 1456, 64, 16, 256, 17408), (False, True, 100, 16384, 1024, 50, 16, 256, 16384),
    (False, False, 40, 400, 4096, 8, 16, 128, 8192)])
def test_what_a_plan_asks_for(half, packed, m, k, n, e, rows, cols, tile):
    dt = dict(x_dtype=cabi.DT_BF16, out_dtype=cabi.DT_BF16, antiquant_dtype=cabi.DT_BF16) if half else dict(x_dtype=cabi.DT_I8, out_dtype=cabi.DT_BF16, scale_dtype=cabi.DT_F32)
    op = cabi.GmmOp(group_list_dtype=cabi.DT_I64, weight_layout=cabi.WL_PACKED if packed else cabi.WL_ROW_MAJOR, kernel_override=cabi.OV_SKINNY,
                    force_split_k=2, **dt)
    try:
        op.plan(m, k, n, e)
    except cabi.BackendError:
        pass   # (a split plan allocates counters on the device; the plan itself stands)
    info = op.plan_info()
    op.close()
    split, strips, size = (int(re.search(f"{f}=(\\d+)", info)[1]) for f in ("split_k", "strips", "workspace"))
    if not packed:
        strips = -(-n // cols)   # (the 16-wave kernel has strips of its own)
    assert split > 1 and size == _slots(m, e, rows) * strips * split * tile, info
    assert size < 200 << 20, info


@pytest.mark.gpu
@pytest.mark.parametrize("counts", [[33, 0, 5, 17, 64], [0, 1, 0, 16, 2], [100], [3] * 40])
@pytest.mark.parametrize("layout,k,n,split", [("kn", 1040, 272, 3), ("nk", 4112, 272, 3), ("kn", 2064, 4112, 2), ("packed", 2064, 272, 3)])
def test_int8_bit_exact(device, counts, layout, k, n, split):
    from gpu_utils import run_w8a8
    rng = np.random.default_rng(k + n + len(counts))
    e, rows = len(counts), sum(counts)
    m = rows + 2
    x, w = rng.integers(-128, 128, (m, k), dtype=np.int8), rng.integers(-128, 128, (e, k, n), dtype=np.int8)
    scale, pt = rng.uniform(1e-3, 1e-2, (e, n)).astype(np.float32), rng.uniform(1e-3, 1e-2, m).astype(np.float32)
    ends = np.cumsum(counts)
    got, info = run_w8a8(x, w, ends, None, scale, pt, transpose_b=layout == "nk", packed=layout == "packed", override=cabi.OV_SKINNY, force_split_k=split, launches=3)
    want = O.grouped_matmul_w8a8(x, w, ends, None, scale, pt)
    assert "split_k=1 " not in info and ("skinny" in info or "stream" in info), info
    assert np.array_equal(got[:rows], want[:rows].view(got.dtype)) and (got[rows:] == 0x7FC0).all(), info


@pytest.mark.gpu
@pytest.mark.parametrize("counts", [[33, 0, 5, 17, 64], [0, 1, 0, 16, 2], [3] * 40])
def test_weight_only_within_the_workspace(device, counts):
    """bfloat16 x on packed weights, three slices: within one rounding and float32 noise of float64, the same bits every time, nothing behind the
    workspace written."""
    import torch
    from gpu_utils import pack_on_device, ptr, to_dev
    k, n = 4368, 272
    rng = np.random.default_rng(len(counts))
    e, rows = len(counts), sum(counts)
    x = O.f32_to_bf16_bits(rng.standard_normal((rows, k)).astype(np.float32))
    s = O.f32_to_bf16_bits(rng.uniform(1e-3, 1e-2, (e, n)).astype(np.float32))
    w = rng.integers(-128, 128, (e, k, n), dtype=np.int8)
    tx, ts, gl = to_dev(x), to_dev(s), to_dev(np.asarray(counts, dtype=np.int64))
    tw = pack_on_device(to_dev(w), e, k, n)
    op = cabi.GmmOp(x_dtype=cabi.DT_BF16, out_dtype=cabi.DT_BF16, group_list_dtype=cabi.DT_I64, group_list_type=1, antiquant_dtype=cabi.DT_BF16,
                    weight_layout=cabi.WL_PACKED, kernel_override=cabi.OV_SKINNY, force_split_k=3)
    ws = op.plan(rows, k, n, e)
    info = op.plan_info()
    assert "split_k=1 " not in info or "stream_rows" in info, info
    buf = torch.full((ws + (1 << 20),), 0x7F, dtype=torch.uint8, device="cuda:0")
    got = []
    for _ in range(3):
        out = torch.full((rows, n), 0x7FC0, dtype=torch.int16, device="cuda:0")
        op.launch([ptr(tx), ptr(tw), None, None, ptr(gl), None, ptr(ts), None], out.data_ptr(), buf.data_ptr(), ws, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        got.append(out.cpu().numpy().view(np.uint16))
    op.close()
    assert all(np.array_equal(got[0], q) for q in got[1:]) and bool((buf[ws:] == 0x7F).all())
    xf, sf = O.bf16_bits_to_f32(x), O.bf16_bits_to_f32(s)
    ends, starts = np.cumsum(counts), np.cumsum(counts) - counts
    exact = O.a16w8_grouped_f64(xf, w, sf, np.zeros((e, n), np.float32), ends)[:rows]
    # (the kernel sums x (w + 128) and takes 128 sum x out again: the noise is that of the larger sum)
    mag = np.concatenate([np.abs(xf[a:b]) @ ((np.abs(w[g].astype(np.float64)) + 256) * sf[g]) for g, (a, b) in enumerate(zip(starts, ends))])
    assert (np.abs(O.bf16_bits_to_f32(got[0]).astype(np.float64) - exact) <= 2.0 ** -7 * np.abs(exact) + 2e-5 * mag).all()
