"""Row-chunk kernel (kernel_override 11) with groups of several equal chunks, on every XCD's share of (group, strip) pairs, against
the oracle: bit-exact accumulators and outputs, with and without non-temporal weight loads (one chunk per group expected or more)."""
import numpy as np
import pytest
import torch

from gpu_utils import ptr, to_dev
from ms_custom_ops_amd import cabi
from oracle import gmm_oracle as O

pytestmark = pytest.mark.gpu


# rows per group, K, N; two more rows of x lie behind the last group
@pytest.mark.parametrize("counts,k,n", [([161, 0, 320, 321], 1040, 272), ([700, 257], 512, 2320), ([5, 0] * 35 + [333], 64, 48),
                                        ([1, 160, 17, 0, 129], 144, 4624)])
def test_several_chunks_per_group_bit_exact(device, counts, k, n):
    rng = np.random.default_rng(k + n)
    e, rows = len(counts), sum(counts)
    m = rows + 2
    x = rng.integers(-128, 128, (m, k), dtype=np.int8)
    w = rng.integers(-128, 128, (e, k, n), dtype=np.int8)
    scale = rng.uniform(1e-3, 1e-2, (e, n)).astype(np.float32)
    pt = rng.uniform(1e-3, 1e-2, m).astype(np.float32)
    want = O.grouped_matmul_w8a8(x, w, np.cumsum(counts), None, scale, pt)
    src, tx, gl, ts, tp = to_dev(w), to_dev(x), to_dev(np.asarray(counts, dtype=np.int64)), to_dev(scale), to_dev(pt)
    tw = torch.empty(e * cabi.packed_weight_bytes(k, n), dtype=torch.int8, device="cuda:0")
    cabi.pack_weight(src.data_ptr(), tw.data_ptr(), e, k, n)
    op = cabi.GmmOp(x_dtype=cabi.DT_I8, weight_dtype=cabi.DT_I8, out_dtype=cabi.DT_BF16, group_list_dtype=cabi.DT_I64, group_list_type=1,
                    scale_dtype=cabi.DT_F32, per_token_dtype=cabi.DT_F32, scale_per_group=1, kernel_override=cabi.OV_ROWS160,
                    weight_layout=cabi.WL_PACKED)
    assert op.plan(m, k, n, e) == 0 and "rows160" in op.plan_info(), op.plan_info()
    out = torch.full((m, n), 0x7FC0, dtype=torch.int16, device="cuda:0")
    op.launch([ptr(tx), ptr(tw), None, ptr(ts), ptr(gl), ptr(tp), None, None], out.data_ptr(), None, 0, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    op.close()
    got = out.cpu().numpy().view(np.uint16)
    assert np.array_equal(got[:rows], want[:rows])
    assert (got[rows:] == 0x7FC0).all()
