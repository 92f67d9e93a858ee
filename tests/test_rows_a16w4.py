"""The weight-only 128-row kernel on 4-bit [E,K,N] weights (kernel_override 14, 15, 16): bit for bit what it gives on int8 weights of
the same values, whose own tests compare them with float64; at the ends of the range of float32 too."""
import numpy as np
import pytest
import torch

from gpu_utils import ptr, to_dev
from ms_custom_ops_amd import cabi
from oracle import gmm_oracle as O

# (rows per group, K, N): every number of row blocks, K tails, strips that end inside a wave's 64 columns, empty groups
SHAPES = [([1, 0, 16, 17, 40, 50, 65, 90, 97, 128], 80, 272), ([129, 0, 257, 1], 336, 528), ([0, 5] * 40, 48, 64), ([300, 20], 1040, 16)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("override,split", [(cabi.OV_ROWS16, 0), (cabi.OV_ROWS16_256, 1), (cabi.OV_ROWS16_256, 3), (cabi.OV_ROWS16_256X2, 1), (cabi.OV_ROWS16_256X2, 2)])
@pytest.mark.parametrize("counts,k,n", SHAPES)
def test_equals_the_kernel_on_int8_weights(device, counts, k, n, override, split, dtype):
    rng = np.random.default_rng(k + n)
    e, rows = len(counts), sum(counts)
    m = rows + 2
    to_bits = O.f32_to_bf16_bits if dtype == "bf16" else (lambda a: a.astype(np.float16).view(np.uint16))
    x = to_bits(rng.standard_normal((m, k)).astype(np.float32))
    x[rows:] = 0x7F80 if dtype == "bf16" else 0x7C00         # infinities behind the last group reach no output
    s, o = to_bits(rng.uniform(1e-3, 1e-2, (e, n)).astype(np.float32)), to_bits(rng.integers(-8, 9, (e, n)).astype(np.float32))
    w = rng.integers(-8, 8, (e, k, n), dtype=np.int8)
    dt = cabi.DT_BF16 if dtype == "bf16" else cabi.DT_F16
    tx, gl, ts, to = to_dev(x), to_dev(np.asarray(counts, dtype=np.int64)), to_dev(s), to_dev(o)
    outs = []
    for bits in (4, 8):
        tw = to_dev(O.pack_int4(w) if bits == 4 else w)
        op = cabi.GmmOp(x_dtype=dt, weight_dtype=cabi.DT_I4 if bits == 4 else cabi.DT_I8, out_dtype=dt, group_list_dtype=cabi.DT_I64, group_list_type=1,
                        antiquant_dtype=dt, has_antiquant_offset=1, kernel_override=override, force_split_k=split)
        ws = op.plan(m, k, n, e)
        assert "rows128" in op.plan_info() and "widened" not in op.plan_info()
        buf = torch.full((max(ws, 1),), 0x7F, dtype=torch.uint8, device="cuda:0")
        for _ in range(2):
            out = torch.full((m, n), 0x7FC0, dtype=torch.int16, device="cuda:0")
            op.launch([ptr(tx), ptr(tw), None, None, ptr(gl), None, ptr(ts), ptr(to)], out.data_ptr(), buf.data_ptr(), ws, torch.cuda.current_stream().cuda_stream)
            torch.cuda.synchronize()
            outs.append(out.cpu().numpy().view(np.uint16))
        op.close()
    assert all(np.array_equal(outs[0], q) for q in outs[1:])
    assert outs[0][:rows].any() and (outs[0][rows:] == 0x7FC0).all()      # rows behind the last group are left alone


@pytest.mark.gpu
@pytest.mark.parametrize("exponent", [121, -124, -130])
@pytest.mark.parametrize("override,split", [(cabi.OV_ROWS16, 0), (cabi.OV_ROWS16_256, 1), (cabi.OV_ROWS16_256, 3), (cabi.OV_ROWS16_256X2, 2)])
def test_sums_at_the_ends_of_float32(device, override, split, exponent):
    """bfloat16 x around 2^exponent: what is finite on int8 weights is the same on 4-bit ones (sums up to 2^128, brought back by
    the scales), and subnormal x, products and sums lose nothing."""
    rng = np.random.default_rng(3)
    counts, k, n = [100, 33], 256, 272
    m = sum(counts)
    x = O.f32_to_bf16_bits(np.ldexp(rng.standard_normal((m, k)), exponent).astype(np.float32))
    s = O.f32_to_bf16_bits(np.full((2, n), 2.0 ** -6 if exponent > 0 else 1.0, np.float32))
    w = rng.integers(-8, 8, (2, k, n), dtype=np.int8)
    tx, gl, ts = to_dev(x), to_dev(np.asarray(counts, dtype=np.int64)), to_dev(s)
    outs = {}
    for bits in (4, 8):
        tw = to_dev(O.pack_int4(w) if bits == 4 else w)
        op = cabi.GmmOp(x_dtype=cabi.DT_BF16, weight_dtype=cabi.DT_I4 if bits == 4 else cabi.DT_I8, out_dtype=cabi.DT_BF16, group_list_dtype=cabi.DT_I64,
                        group_list_type=1, antiquant_dtype=cabi.DT_BF16, kernel_override=override, force_split_k=split)
        ws = op.plan(m, k, n, 2)
        buf = torch.zeros(max(ws, 1), dtype=torch.uint8, device="cuda:0")
        out = torch.zeros((m, n), dtype=torch.int16, device="cuda:0")
        op.launch([ptr(tx), ptr(tw), None, None, ptr(gl), None, ptr(ts), None], out.data_ptr(), buf.data_ptr(), ws, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        op.close()
        outs[bits] = out.cpu().numpy().view(np.uint16)
    finite = (outs[8] & 0x7F80) != 0x7F80
    assert np.array_equal(outs[4][finite], outs[8][finite])
    if exponent > 0:
        assert O.bf16_bits_to_f32(outs[8][finite]).max() > 2.0 ** (124 - 6)   # sums that sixteen times their value would have made infinite
    else:
        assert finite.all() and (outs[8] & 0x7FFF).any()
