"""4-bit weights and 16-bit x where the 128-row kernel would have few workgroups: the plan leaves them to the register-transpose kernels,
groups of any number of rows.  What it picks at both sides of its lines (CPU), and its results there against float64 (GPU)."""
import numpy as np
import pytest

from ms_custom_ops_amd import cabi

# (rows, K, N, groups, register-transpose kernels); 256 CUs: 64 workgroups of 128 rows x 256 columns
PICKS = [(944, 3056, 768, 8, True), (930, 3072, 512, 8, True), (930, 3088, 512, 8, False), (464, 2048, 2048, 8, True), (464, 2048, 2064, 8, False),
         (1152, 2080, 512, 32, True), (1152, 2080, 768, 32, False), (2120, 1056, 512, 8, True), (2120, 1056, 768, 8, False)]


def _op(m, k, n, e, dt):
    op = cabi.GmmOp(x_dtype=dt, out_dtype=dt, weight_dtype=cabi.DT_I4, group_list_dtype=cabi.DT_I64, antiquant_dtype=dt, has_antiquant_offset=1)
    try:
        return op, op.plan(m, k, n, e)
    except cabi.BackendError:
        return op, 0   # (no device: a split plan cannot allocate its counters; the plan itself stands)


@pytest.mark.parametrize("m,k,n,e,regt", PICKS)
@pytest.mark.parametrize("dt", [cabi.DT_BF16, cabi.DT_F16])
def test_the_rule(m, k, n, e, regt, dt):
    op, _ = _op(m, k, n, e, dt)
    assert ("a16w4_skinny_regt" if regt else "a16w4_rows128") in op.plan_info(), op.plan_info()
    op.close()


def test_chunks_that_a_random_routing_makes():
    # 32 experts, 54 rows: 64 chunks of an average group's and 71 of a random routing; two strips of those twice are more than 256 workgroups
    op, _ = _op(32 * 54, 3024, 400, 32, cabi.DT_BF16)
    assert "split_k=1 strips=2" in op.plan_info(), op.plan_info()
    op.close()


def test_strips_are_no_wider_than_the_columns():
    # partial tiles of a forced split show the strip: as wide for 256 chunks of 112 columns (strips of 512 "fill" the chip) as for 86
    def bytes_of(rows, e):
        op = cabi.GmmOp(x_dtype=cabi.DT_BF16, out_dtype=cabi.DT_BF16, weight_dtype=cabi.DT_I4, group_list_dtype=cabi.DT_I64, antiquant_dtype=cabi.DT_BF16,
                        has_antiquant_offset=1, force_split_k=2)
        try:
            op.plan(rows * e, 1504, 112, e)
        except cabi.BackendError:
            pass   # (no device for the counters)
        info = op.plan_info()
        op.close()
        assert "skinny_regt" in info and "strips=1" in info, info
        return int(info.split("workspace=")[1].split()[0]) // (e + rows * e // 32)
    assert bytes_of(114, 64) == bytes_of(54, 32)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("counts,k,n", [([130, 0, 33, 257, 1, 64, 32, 200], 1040, 512), ([5, 300, 31, 0, 90, 127, 128, 129], 2064, 272),
                                        ([0, 130, 33, 64, 65, 31, 96, 13] * 4, 720, 400), ([114, 0, 228, 115, 129, 1, 63, 97] * 8, 544, 112)])
def test_against_float64(device, counts, k, n, dtype):
    # bound: one rounding of the output, and 1e-5 of the sum of the terms' magnitudes for K < 4096 float32 additions of 2^-24 each
    import torch

    from gpu_utils import ptr, to_dev
    from oracle import gmm_oracle as O

    rng = np.random.default_rng(k)
    e, rows = len(counts), sum(counts)
    to_bits = O.f32_to_bf16_bits if dtype == "bf16" else (lambda a: a.astype(np.float16).view(np.uint16))
    to_f = O.bf16_bits_to_f32 if dtype == "bf16" else (lambda b: b.view(np.float16).astype(np.float32))
    x = to_bits(rng.standard_normal((rows, k)).astype(np.float32))
    w = rng.integers(-8, 8, (e, k, n), dtype=np.int8)
    s, o = to_bits(rng.uniform(1e-3, 1e-2, (e, n)).astype(np.float32)), to_bits(rng.integers(-8, 9, (e, n)).astype(np.float32))
    ends = np.cumsum(counts)
    op, ws = _op(rows, k, n, e, cabi.DT_BF16 if dtype == "bf16" else cabi.DT_F16)
    assert "a16w4_skinny_regt" in op.plan_info()
    ts = [to_dev(a) for a in (x, O.pack_int4(w), ends.astype(np.int64), s, o)]
    buf = torch.empty(max(ws, 1), dtype=torch.uint8, device="cuda:0")
    out = torch.full((rows, n), 0x7FC0, dtype=torch.int16, device="cuda:0")
    for _ in range(2):
        op.launch([ptr(ts[0]), ptr(ts[1]), None, None, ptr(ts[2]), None, ptr(ts[3]), ptr(ts[4])], out.data_ptr(), buf.data_ptr(), ws, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    op.close()
    got = to_f(out.cpu().numpy().view(np.uint16)).astype(np.float64)
    exact = O.a16w8_grouped_f64(to_f(x), w, to_f(s), to_f(o), ends)
    mag = np.concatenate([np.abs(to_f(x)[b - c:b]) @ (np.abs(w[g].astype(np.float64) + to_f(o)[g]) * to_f(s)[g]) for g, (b, c) in enumerate(zip(ends, counts))])
    assert (np.abs(got - exact) <= (2.0 ** -7 if dtype == "bf16" else 2.0 ** -10) * np.abs(exact) + 1e-5 * mag).all()
