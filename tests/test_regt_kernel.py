"""Kernels on row-major [E,K,N] weights of 4 and 8 bits, at the edges of their chunks, strips, K steps and K splits, against
the oracle: the ones that transpose and convert in registers (kernel_override 12: chunks of 16 / 32 rows, strips of 256 / 512
columns, steps of 64 / 32 K) and the tiles that read 4-bit weights through LDS (13: 64 or 128 x 256, slabs of 64 K)."""
import numpy as np
import pytest
import torch

from gpu_utils import ptr, to_dev
from ms_custom_ops_amd import cabi
from oracle import gmm_oracle as O

pytestmark = pytest.mark.gpu

# (rows per group, K, N, forced K split); the last list entry is where the rows end, M is two more
SHAPES = [([1], 16, 16, 0), ([16, 0, 17], 48, 256, 0), ([3, 33, 1], 2064, 272, 3), ([5] * 24, 80, 528, 0), ([31, 2], 4096, 512, 8),
          ([0, 0, 64, 7], 96, 1040, 2), ([2] * 70, 64, 48, 0)]


def _run(x_dtype, bits, x, w, counts, split, operands, out_dtype, override=cabi.OV_REGT, must="", **fields):
    m, (e, k, n) = x.shape[0], w.shape
    wd = to_dev(O.pack_int4(w) if bits == 4 else w)
    gl = to_dev(np.asarray(counts, dtype=np.int64))
    op = cabi.GmmOp(x_dtype=x_dtype, weight_dtype=cabi.DT_I4 if bits == 4 else cabi.DT_I8, out_dtype=out_dtype, group_list_dtype=cabi.DT_I64,
                    group_list_type=1, kernel_override=override, force_split_k=split, **fields)
    ws = op.plan(m, k, n, e)
    assert {cabi.OV_AUTO: must, cabi.OV_REGT: "regt", cabi.OV_TILE_4BIT: "4bit"}[override] in op.plan_info(), op.plan_info()
    assert must in op.plan_info(), op.plan_info()
    tws = torch.empty(max(ws, 1), dtype=torch.uint8, device="cuda:0")
    out = torch.full((m, n), 0x7FC0, dtype=torch.int32 if out_dtype == cabi.DT_I32 else torch.int16, device="cuda:0")
    tx = to_dev(x)
    ins = [ptr(tx), ptr(wd), None, None, ptr(gl), None, None, None]
    for slot, t in operands.items():
        ins[slot] = ptr(t)
    for _ in range(2):   # the arrival counters of a K split reset themselves
        op.launch(ins, out.data_ptr(), tws.data_ptr(), ws, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    op.close()
    return out.cpu().numpy()


def _weights(rng, bits, e, k, n):
    return rng.integers(-8, 8, (e, k, n), dtype=np.int8) if bits == 4 else rng.integers(-128, 128, (e, k, n), dtype=np.int8)


TILE_SHAPES = [([65], 80, 16, 0), ([64, 1, 0, 63], 4096, 272, 4), ([129, 40, 128], 2064, 528, 0), ([100] * 9, 256, 6144, 0)]


@pytest.mark.parametrize("counts,k,n,split,bits,override",
                         [(*s, bits, cabi.OV_REGT) for s in SHAPES for bits in (4, 8)] + [(*s, 4, cabi.OV_TILE_4BIT) for s in SHAPES + TILE_SHAPES])
def test_int8_activations_bit_exact(device, counts, k, n, split, bits, override):
    rng = np.random.default_rng(k + n + bits)
    e, rows = len(counts), sum(counts)
    x = rng.integers(-128, 128, (rows + 2, k), dtype=np.int8)
    w = _weights(rng, bits, e, k, n)
    bias = rng.integers(-1000, 1001, (e, n), dtype=np.int32)
    scale = rng.uniform(1e-3, 1e-2, (e, n)).astype(np.float32)
    pt = rng.uniform(1e-3, 1e-2, rows + 2).astype(np.float32)
    want, acc = O.grouped_matmul_w8a8(x, w, np.cumsum(counts), bias, scale, pt, return_acc=True)
    ops = {cabi.IN_BIAS: to_dev(bias), cabi.IN_SCALE: to_dev(scale), cabi.IN_PER_TOKEN_SCALE: to_dev(pt)}
    got = _run(cabi.DT_I8, bits, x, w, counts, split, ops, cabi.DT_BF16, override, bias_dtype=cabi.DT_I32, scale_dtype=cabi.DT_F32, per_token_dtype=cabi.DT_F32)
    assert np.array_equal(got[:rows].view(np.uint16), want[:rows])
    assert (got[rows:] == 0x7FC0).all()                      # rows behind the last group are left alone
    raw = _run(cabi.DT_I8, bits, x, w, counts, split, {cabi.IN_BIAS: ops[cabi.IN_BIAS]}, cabi.DT_I32, override, bias_dtype=cabi.DT_I32)
    assert np.array_equal(raw[:rows], acc[:rows] + np.repeat(bias, counts, axis=0))


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("counts,k,n,split", SHAPES)
def test_16_bit_activations_within_one_rounding_and_equal_for_both_weight_widths(device, counts, k, n, split, dtype):
    """One rounding of the output plus float32 accumulation noise (1e-5 of the sum of the terms' magnitudes: K <= 4096
    additions of relative error 2^-24 each) against float64; 4-bit weights and 8-bit weights of the same values give the
    same bits where both take 16-row chunks (the 4-bit operands are 16 times the values, a power of two)."""
    rng = np.random.default_rng(k + n)
    e, rows = len(counts), sum(counts)
    to_bits = O.f32_to_bf16_bits if dtype == "bf16" else (lambda a: a.astype(np.float16).view(np.uint16))
    to_f = O.bf16_bits_to_f32 if dtype == "bf16" else (lambda b: b.view(np.float16).astype(np.float32))
    x = to_bits(rng.standard_normal((rows + 2, k)).astype(np.float32))
    s = to_bits(rng.uniform(1e-3, 1e-2, (e, n)).astype(np.float32))
    o = to_bits(rng.integers(-8, 9, (e, n)).astype(np.float32))
    dt = cabi.DT_BF16 if dtype == "bf16" else cabi.DT_F16
    ops = {cabi.IN_ANTIQUANT_SCALE: to_dev(s), cabi.IN_ANTIQUANT_OFFSET: to_dev(o)}
    run = lambda bits, w: _run(dt, bits, x, w, counts, split, ops, dt, antiquant_dtype=dt, has_antiquant_offset=1).view(np.uint16)
    ends, starts = np.cumsum(counts), np.cumsum(counts) - counts
    for w in (_weights(rng, 8, e, k, n), _weights(rng, 4, e, k, n)):
        got = run(8, w)
        exact = O.a16w8_grouped_f64(to_f(x), w, to_f(s), to_f(o), ends)[:rows]
        mag = np.concatenate([np.abs(to_f(x)[a:b]) @ (np.abs(w[g].astype(np.float64) + to_f(o)[g]) * to_f(s)[g]) for g, (a, b) in enumerate(zip(starts, ends))])
        ulp = 2.0 ** -7 if dtype == "bf16" else 2.0 ** -10
        assert (np.abs(to_f(got[:rows]).astype(np.float64) - exact) <= ulp * np.abs(exact) + 1e-5 * mag).all()
        assert (got[rows:] == 0x7FC0).all()
    avg = -(-(rows + 2) // e)
    if (avg if e == 1 else avg + avg // 2) <= 16:   # chunks of 16 rows for both widths: the same order of summation
        assert np.array_equal(got, run(4, w))


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
def test_16_bit_activations_long_k_exact(device, dtype, bits):
    """K beyond 2^17 and beyond what int32 sums of 16 times the products could hold.  x is -1, 0 or 1, so every float32 partial sum
    is exact (|sum| <= 127 K < 2^24; 4-bit weights: multiples of 16 below 2^28) and the output is two roundings of it: the same bits."""
    rng = np.random.default_rng(bits)
    k, n, counts = 131088, 48, [2, 1]
    xv = rng.integers(-1, 2, (5, k)).astype(np.float32)
    x = O.f32_to_bf16_bits(xv) if dtype == "bf16" else xv.astype(np.float16).view(np.uint16)
    w = np.maximum(_weights(rng, bits, 2, k, n), -127)
    sv = (2.0 ** rng.integers(-8, -4, (2, n))).astype(np.float32) if dtype == "bf16" else np.full((2, n), 2.0 ** -10, np.float32)
    s = O.f32_to_bf16_bits(sv) if dtype == "bf16" else sv.astype(np.float16).view(np.uint16)
    dt = cabi.DT_BF16 if dtype == "bf16" else cabi.DT_F16
    got = _run(dt, bits, x, w, counts, 0, {cabi.IN_ANTIQUANT_SCALE: to_dev(s)}, dt, antiquant_dtype=dt).view(np.uint16)
    acc = np.concatenate([xv[:2].astype(np.int64) @ w[0].astype(np.int64), xv[2:3].astype(np.int64) @ w[1].astype(np.int64)])
    want = acc.astype(np.float32) * np.repeat(sv, counts, axis=0)
    assert np.array_equal(got[:3], O.f32_to_bf16_bits(want) if dtype == "bf16" else want.astype(np.float16).view(np.uint16))
    assert (got[3:] == 0x7FC0).all()


# (rows per group, K, N, what the plan names): the form with one K step in flight per wave, planned from 256 workgroups on, in
# strips of 256 columns without and with a K split and in strips of 512; groups of up to 17 rows, the last strip cut at 16 columns
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("counts,k,n,must", [([1, 16, 0, 17, 3, 2, 0, 1] * 4, 80, 4112, "split_k=1 strips=17 "), ([3, 0, 1, 2] * 8, 2064, 1040, "split_k=3 strips=5 "),
                                             ([1, 16, 0, 17, 3, 2, 0, 1] * 4, 48, 3088, "split_k=1 strips=7 "), ([1] * 32, 16, 3072 + 16, "split_k=1 strips=7 ")])
def test_shallow_form_within_one_rounding(device, counts, k, n, must, dtype):
    """Tolerance as above; the same values given as 4-bit weights take the other form and give the same bits."""
    rng = np.random.default_rng(k + n)
    e, rows = len(counts), sum(counts)
    to_bits = O.f32_to_bf16_bits if dtype == "bf16" else (lambda a: a.astype(np.float16).view(np.uint16))
    to_f = O.bf16_bits_to_f32 if dtype == "bf16" else (lambda b: b.view(np.float16).astype(np.float32))
    x = to_bits(rng.standard_normal((rows + 2, k)).astype(np.float32))
    s = to_bits(rng.uniform(1e-3, 1e-2, (e, n)).astype(np.float32))
    o = to_bits(rng.integers(-8, 9, (e, n)).astype(np.float32))
    dt = cabi.DT_BF16 if dtype == "bf16" else cabi.DT_F16
    ops = {cabi.IN_ANTIQUANT_SCALE: to_dev(s), cabi.IN_ANTIQUANT_OFFSET: to_dev(o)}
    run = lambda bits, w, name, split=0: _run(dt, bits, x, w, counts, split, ops, dt, cabi.OV_AUTO, name, antiquant_dtype=dt, has_antiquant_offset=1).view(np.uint16)
    ends, starts = np.cumsum(counts), np.cumsum(counts) - counts
    for bits in (8, 4):
        w = _weights(rng, bits, e, k, n)
        got = run(8, w, "regt_shallow layout=[E,K,N] m=%d k=%d n=%d e=%d %s" % (rows + 2, k, n, e, must))
        exact = O.a16w8_grouped_f64(to_f(x), w, to_f(s), to_f(o), ends)[:rows]
        mag = np.concatenate([np.abs(to_f(x)[a:b]) @ (np.abs(w[g].astype(np.float64) + to_f(o)[g]) * to_f(s)[g]) for g, (a, b) in enumerate(zip(starts, ends))])
        ulp = 2.0 ** -7 if dtype == "bf16" else 2.0 ** -10
        assert (np.abs(to_f(got[:rows]).astype(np.float64) - exact) <= ulp * np.abs(exact) + 1e-5 * mag).all()
        assert (got[rows:] == 0x7FC0).all()
    assert np.array_equal(got, run(4, w, "skinny_regt ", int(must[8])))   # (the same K slices)


def test_large_a8w4_call_widens_first(device):
    """A call large enough for the persistent kernel: the int8 copy at the front of the workspace gives the bits that int8
    weights of the same values give, and those of the oracle on the first and last rows of every group."""
    rng = np.random.default_rng(0)
    counts, k, n = [40000, 26001], 512, 1040
    e, rows = len(counts), sum(counts)
    x, w = rng.integers(-128, 128, (rows + 2, k), dtype=np.int8), _weights(rng, 4, e, k, n)
    scale = rng.uniform(1e-3, 1e-2, (e, n)).astype(np.float32)
    ops = {cabi.IN_SCALE: to_dev(scale)}
    run = lambda bits, name: _run(cabi.DT_I8, bits, x, w, counts, 0, ops, cabi.DT_BF16, cabi.OV_AUTO, name, scale_dtype=cabi.DT_F32, scale_per_group=1)
    got = run(4, "a8w4_widened_tile_256x256x128_w4")
    assert np.array_equal(got, run(8, "w8a8_tile_256x256x128_w4"))
    for g, (a, b) in enumerate(((0, 40000), (40000, rows))):
        pick = np.r_[a:a + 8, b - 8:b]
        want = O.grouped_matmul_w8a8(x[pick], w[g:g + 1], np.array([16]), None, scale[g:g + 1], None)
        assert np.array_equal(got[pick].view(np.uint16), want)
    assert (got[rows:] == 0x7FC0).all()


# (weight bits, override, groups x rows, what the plan names): register transpose with three and one K steps in flight, 4-bit weights,
# the kernel of up to 128-row chunks
@pytest.mark.parametrize("bits,override,counts,must", [(8, cabi.OV_AUTO, [5, 16], "skinny_regt layout"), (8, cabi.OV_AUTO, [3] * 40, "regt_shallow"),
                                                       (4, cabi.OV_AUTO, [5, 16], "skinny_regt layout"), (8, cabi.OV_ROWS16, [100, 30], "rows128")])
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
def test_16_bit_operands_may_start_at_any_element(device, dtype, bits, override, counts, must):
    """x, scale and offset one element behind a 16-byte boundary: the same bits as on one."""
    rng = np.random.default_rng(bits)
    e, m, k, n = len(counts), sum(counts), 80, 1808
    dt, t16 = (cabi.DT_BF16, torch.bfloat16) if dtype == "bf16" else (cabi.DT_F16, torch.float16)
    half = lambda a: torch.from_numpy(a.astype(np.float32)).cuda().to(t16)
    x, s, o = half(rng.standard_normal((m, k))), half(rng.uniform(1e-3, 1e-2, (e, n))), half(rng.integers(-8, 9, (e, n)))
    w = _weights(rng, bits, e, k, n)
    wd, gl = to_dev(O.pack_int4(w) if bits == 4 else w), to_dev(np.asarray(counts, dtype=np.int64))

    def shifted(t):
        whole = torch.zeros(t.numel() + 16, dtype=t16, device="cuda")
        assert whole.data_ptr() % 16 == 0
        view = whole[1:1 + t.numel()].view(t.shape)
        return view.copy_(t)

    op = cabi.GmmOp(x_dtype=dt, weight_dtype=cabi.DT_I4 if bits == 4 else cabi.DT_I8, out_dtype=dt, group_list_dtype=cabi.DT_I64, group_list_type=1,
                    antiquant_dtype=dt, has_antiquant_offset=1, kernel_override=override)
    ws = op.plan(m, k, n, e)
    assert must in op.plan_info(), op.plan_info()
    tws = torch.empty(max(ws, 1), dtype=torch.uint8, device="cuda")
    outs = []
    for ins in ((x, s, o), (shifted(x), s, o), (x, shifted(s), shifted(o))):
        out = torch.zeros((m, n), dtype=t16, device="cuda")
        op.launch([ptr(ins[0]), ptr(wd), None, None, ptr(gl), None, ptr(ins[1]), ptr(ins[2])], out.data_ptr(), tws.data_ptr(), ws,
                  torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        outs.append(out.view(torch.int16))
    op.close()
    assert outs[0].any() and torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


# (x type, rows per group, K, N, forced K split, what the plan names)
WIDENED = [("bf16", [100, 90], 192, 96, 0, "a16w4_widened_"), ("f16", [70, 0, 230], 2048, 1040, 0, "a16w4_widened_"),
           ("bf16", [198], 2048, 272, 4, "a16w4_widened_skinny_rows layout=[E,K,N] m=200 k=2048 n=272 e=1 split_k=4"),
           ("f16", [5, 6], 100, 24, 0, "a16w4_widened_generic"), ("i8", [5, 6], 100, 24, 0, "a8w4_widened_generic"),
           ("i8", [3], 131072, 48, 8, "a8w4_widened_skinny")]


@pytest.mark.parametrize("x_type,counts,k,n,split,must", WIDENED)
def test_widened_by_the_backend_like_8_bit_weights(device, x_type, counts, k, n, split, must):
    """4-bit weights that no kernel reads directly: an int8 copy at the front of the workspace, the partial tiles of a K split
    behind it.  The bits of the same call on int8 weights of the same values, and int8 x against the oracle."""
    rng = np.random.default_rng(k + n)
    e, rows = len(counts), sum(counts)
    w = _weights(rng, 4, e, k, n)
    w[:, ::2, ::3] = -8
    if x_type == "i8":
        x, dt, out = rng.integers(-128, 128, (rows + 2, k), dtype=np.int8), cabi.DT_I8, cabi.DT_BF16
        s = rng.uniform(1e-3, 1e-2, (e, n)).astype(np.float32)
        ops, fields = {cabi.IN_SCALE: to_dev(s)}, dict(scale_dtype=cabi.DT_F32, scale_per_group=1)
    else:
        to_bits = O.f32_to_bf16_bits if x_type == "bf16" else (lambda a: a.astype(np.float16).view(np.uint16))
        x, dt = to_bits(rng.standard_normal((rows + 2, k)).astype(np.float32)), cabi.DT_BF16 if x_type == "bf16" else cabi.DT_F16
        out = dt
        s, o = to_bits(rng.uniform(1e-3, 1e-2, (e, n)).astype(np.float32)), to_bits(rng.integers(-8, 9, (e, n)).astype(np.float32))
        ops, fields = {cabi.IN_ANTIQUANT_SCALE: to_dev(s), cabi.IN_ANTIQUANT_OFFSET: to_dev(o)}, dict(antiquant_dtype=dt, has_antiquant_offset=1)
    run = lambda bits, name: _run(dt, bits, x, w, counts, split, ops, out, cabi.OV_AUTO, name, **fields).view(np.uint16)
    got, wide = run(4, must), run(8, "8_")
    assert np.array_equal(got[:rows], wide[:rows])
    if x_type == "i8":
        assert np.array_equal(got[:rows], O.grouped_matmul_w8a8(x, w, np.cumsum(counts), None, s, None)[:rows])
    else:
        to_f = O.bf16_bits_to_f32 if x_type == "bf16" else (lambda b: b.view(np.float16).astype(np.float32))
        exact = O.a16w8_grouped_f64(to_f(x), w, to_f(s), to_f(o), np.cumsum(counts))[:rows]
        assert np.abs(to_f(got[:rows]) - exact).max() <= 2.0 ** (-7 if x_type == "bf16" else -10) * np.abs(exact).max()


# (x type, override, rows per group, K, N, what the plan names)
ACTIVATED = [("i8", cabi.OV_REGT, [3, 33, 1], 272, 272, "a8w4_skinny_regt"), ("i8", cabi.OV_TILE_4BIT, [3, 33, 1], 272, 272, "64x256_4bit"),
             ("i8", cabi.OV_TILE_4BIT, [100] * 9, 256, 6128, "128x256_4bit"), ("bf16", cabi.OV_REGT, [3, 33, 1], 272, 272, "a16w4_skinny_regt")]


@pytest.mark.parametrize("act", [O.ACT_RELU, O.ACT_GELU_TANH, O.ACT_FAST_GELU, O.ACT_SILU])
@pytest.mark.parametrize("x_type,override,counts,k,n,must", ACTIVATED)
def test_activation_on_4_bit_weights(device, x_type, override, counts, k, n, must, act):
    """int8 x: the activation of the exact float32 value within one output ulp (relu: the same bits).  16-bit x: of the
    kernel's own plain output within that ulp and the plain output's (the functions are 1.13-Lipschitz)."""
    rng = np.random.default_rng(n)
    e, rows = len(counts), sum(counts)
    w = _weights(rng, 4, e, k, n)
    if x_type == "i8":
        x = rng.integers(-128, 128, (rows + 2, k), dtype=np.int8)
        s, pt = rng.uniform(1e-3, 1e-2, (e, n)).astype(np.float32), rng.uniform(1e-2, 1e-1, rows + 2).astype(np.float32)
        pre = O.grouped_matmul_w8a8(x, w, np.cumsum(counts), None, s, pt, out_dtype="f32")[:rows]
        ops = {cabi.IN_SCALE: to_dev(s), cabi.IN_PER_TOKEN_SCALE: to_dev(pt)}
        got = _run(cabi.DT_I8, 4, x, w, counts, 0, ops, cabi.DT_BF16, override, must, scale_dtype=cabi.DT_F32, scale_per_group=1, per_token_dtype=cabi.DT_F32,
                   act_type=act)[:rows].view(np.uint16)
        slack = 0.0
    else:
        x, s = O.f32_to_bf16_bits(rng.standard_normal((rows + 2, k)).astype(np.float32)), O.f32_to_bf16_bits(rng.uniform(5e-3, 5e-2, (e, n)).astype(np.float32))
        run = lambda **f: _run(cabi.DT_BF16, 4, x, w, counts, 0, {cabi.IN_ANTIQUANT_SCALE: to_dev(s)}, cabi.DT_BF16, override, must, antiquant_dtype=cabi.DT_BF16, **f)[:rows].view(np.uint16)
        pre, got = O.bf16_bits_to_f32(run()), run(act_type=act)
        slack = 1.13 * 2.0 ** -8
    assert (pre < -1).any() and (pre > 1).any()
    ref = O.activation(pre, act)
    if act == O.ACT_RELU:
        assert np.array_equal(got, O.f32_to_bf16_bits(ref.astype(np.float32)))
    else:
        assert (np.abs(O.bf16_bits_to_f32(got).astype(np.float64) - ref) <= 2.0 ** -7 * np.abs(ref) + slack * np.abs(pre) + 1e-30).all()


@pytest.mark.parametrize("exponent", [119, -124, -130])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("counts,split", [([16, 3], 1), ([31, 2], 2)])
def test_16_bit_activations_at_the_ends_of_float32(device, counts, split, bits, exponent):
    """bfloat16 x around 2^exponent: sums up to 2^127, brought back by the scales, stay finite, and subnormal x and products are kept.
    Bounds: float32 sums of 256 exact products (2^-16 of the terms' magnitudes), one bfloat16 rounding (half a step of 2^-133 where the
    output is subnormal)."""
    rng = np.random.default_rng(13)
    e, m, k, n = len(counts), sum(counts), 256, 272
    x = O.f32_to_bf16_bits(np.ldexp(rng.standard_normal((m, k)), exponent).astype(np.float32))
    w = rng.integers(-8, 8, (e, k, n), dtype=np.int8)
    scale = 2.0 ** -6 if exponent > 0 else 1.0
    s = O.f32_to_bf16_bits(np.full((e, n), scale, np.float32))
    out = _run(cabi.DT_BF16, bits, x, w, counts, split, {cabi.IN_ANTIQUANT_SCALE: to_dev(s)}, cabi.DT_BF16, antiquant_dtype=cabi.DT_BF16)
    got = O.bf16_bits_to_f32(out.view(np.uint16)).astype(np.float64)
    assert np.isfinite(got).all()
    xv, r = O.bf16_bits_to_f32(x).astype(np.float64), 0
    largest = 0.0
    for i, c in enumerate(counts):
        want, mag = xv[r:r + c] @ w[i].astype(np.float64), np.abs(xv[r:r + c]) @ np.abs(w[i].astype(np.float64))
        assert (np.abs(got[r:r + c] - scale * want) <= 2.0 ** -8 * scale * np.abs(want) + 2.0 ** -16 * scale * mag + 2.0 ** -134).all()
        largest, r = max(largest, np.abs(want).max()), r + c
    assert exponent < 0 or 2.0 ** 124 < largest < 2.0 ** 128     # (sixteen times these sums is infinite)
