"""Weight-only decode on packed weights: the K slices that the plan makes beyond 64 blocks of 64, at the edges of a slice's 32 blocks and
with a K tail, against float64; and what the plan does where their partial tiles are too large."""
import numpy as np
import pytest
import torch

from gpu_utils import ptr, to_dev
from ms_custom_ops_amd import cabi
from oracle import gmm_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("counts,k,n,split", [([3], 4096, 1040, 1), ([1], 4112, 528, 3), ([16, 0, 1, 5], 6144, 272, 3), ([2, 0, 0, 7], 6160, 48, 4), ([9], 8192, 16, 4),
                                              ([1, 1], 16384, 32, 8), ([2], 16400, 32, 5)])
def test_within_one_rounding(device, counts, k, n, split, dtype):
    """One rounding of the output plus float32 accumulation noise (2e-5 of the sum of the terms' magnitudes: 16 x 4 lanes' partial sums of
    at most 300 additions each of relative error 2^-24, and their sums) against float64; every launch the same bits, whichever slice
    arrives last."""
    rng = np.random.default_rng(k + n)
    e, rows = len(counts), sum(counts)
    m = rows + 2
    to_bits = O.f32_to_bf16_bits if dtype == "bf16" else (lambda a: a.astype(np.float16).view(np.uint16))
    to_f = O.bf16_bits_to_f32 if dtype == "bf16" else (lambda b: b.view(np.float16).astype(np.float32))
    x = to_bits(rng.standard_normal((m, k)).astype(np.float32))
    x[rows:] = 0x7F80 if dtype == "bf16" else 0x7C00         # infinities behind the last group reach no output
    s, o = to_bits(rng.uniform(1e-3, 1e-2, (e, n)).astype(np.float32)), to_bits(rng.integers(-8, 9, (e, n)).astype(np.float32))
    w = rng.integers(-128, 128, (e, k, n), dtype=np.int8)
    dt = cabi.DT_BF16 if dtype == "bf16" else cabi.DT_F16
    tx, tw, gl, ts, to = to_dev(x), to_dev(w), to_dev(np.asarray(counts, dtype=np.int64)), to_dev(s), to_dev(o)
    src, tw = tw, torch.empty(e * cabi.packed_weight_bytes(k, n), dtype=torch.int8, device="cuda:0")
    cabi.pack_weight(src.data_ptr(), tw.data_ptr(), e, k, n)
    op = cabi.GmmOp(x_dtype=dt, weight_dtype=cabi.DT_I8, out_dtype=dt, group_list_dtype=cabi.DT_I64, group_list_type=1, antiquant_dtype=dt,
                    has_antiquant_offset=1, weight_layout=cabi.WL_PACKED)
    ws = op.plan(m, k, n, e)
    assert "a16w8_stream " in op.plan_info() and f"split_k={split} " in op.plan_info()
    buf = torch.full((max(ws, 1),), 0x7F, dtype=torch.uint8, device="cuda:0")
    got = []
    for _ in range(3):
        out = torch.full((m, n), 0x7FC0, dtype=torch.int16, device="cuda:0")
        op.launch([ptr(tx), ptr(tw), None, None, ptr(gl), None, ptr(ts), ptr(to)], out.data_ptr(), buf.data_ptr(), ws, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        got.append(out.cpu().numpy().view(np.uint16))
    op.close()
    assert (got[0] == got[1]).all() and (got[0] == got[2]).all()
    xf, of = to_f(x)[:rows], to_f(o)
    ends, starts = np.cumsum(counts), np.cumsum(counts) - counts
    exact = O.a16w8_grouped_f64(xf, w, to_f(s), of, ends)[:rows]
    mag = np.concatenate([np.abs(xf[a:b]) @ (np.abs(w[g].astype(np.float64)) * to_f(s)[g]) + np.abs(xf[a:b]).sum(1, keepdims=True) * np.abs(of[g] * to_f(s)[g])
                          for g, (a, b) in enumerate(zip(starts, ends))])
    ulp = 2.0 ** -7 if dtype == "bf16" else 2.0 ** -10
    assert (np.abs(to_f(got[0][:rows]).astype(np.float64) - exact) <= ulp * np.abs(exact) + 2e-5 * mag).all()
    assert (got[0][rows:] == 0x7FC0).all()                  # rows behind the last group are left alone


def test_short_slices_only_within_the_static_workspace(device):
    def plan(m, k, n, e):
        op = cabi.GmmOp(x_dtype=cabi.DT_BF16, out_dtype=cabi.DT_BF16, group_list_dtype=cabi.DT_I64, antiquant_dtype=cabi.DT_BF16, weight_layout=cabi.WL_PACKED)
        return op.plan(m, k, n, e), op.plan_info()

    size, info = plan(18, 4288, 2320, 16)
    assert "split_k=3 " in info and size <= cabi.STATIC_WORKSPACE_BYTES
    size, info = plan(32, 8192, 14336, 8)      # four slices: 62 MB
    assert "split_k=2 " in info and size <= cabi.STATIC_WORKSPACE_BYTES
