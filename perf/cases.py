"""Timed cases: what a user of this package has it do, through its Python entry points.

Six kinds of work, each with the range of sizes that serving meets:

dense        quant_batch_matmul: one int8 linear layer, 1 row (one token) to 4096 rows (a prefill batch)
grouped      grouped_matmul: the int8 expert matrices of a MoE layer, from a decode step (16 tokens) to prefill (4096 tokens),
             few large experts or many small ones, evenly or unevenly used, weights as stored, transposed or prepacked
weight_only  grouped_matmul_v4_cops with 16-bit activations and 8-bit or 4-bit expert weights
a8w4         grouped_matmul_v4_cops with int8 activations and 4-bit expert weights (per-channel scales)
w4           grouped_matmul_w4: int8 activations, 4-bit weights with K-group scales, a few rows over hundreds of experts
moe_ffn      a whole expert layer: routing with quantisation, int8 up projection with SiLU, weight-only down projection,
             un-permutation

Quantised inputs are uniform over their whole range, scales uniform around the size that gives outputs of order one,
16-bit activations normal; rows go to experts by the top-k of random logits, so groups are as uneven as real ones.
"""
import math

import torch

import ms_custom_ops_amd as ops

_HALF = {"bf16": torch.bfloat16, "f16": torch.float16}
_MAX_OPS = 0.98e12          # multiply-adds x 2 of one pass
_MAX_WEIGHTS = 480e6        # weight elements of one pass


def listed():
    return [
        # a dense layer of one decoded token (the smallest call: latency and launches count), and a prefill batch of it
        {"name": "dense_1_row", "kind": "dense", "m": 1, "k": 4096, "n": 11008, "layout": "kn", "bias": True, "out": "f16"},
        {"name": "dense_2048_rows", "kind": "dense", "m": 2048, "k": 4096, "n": 11008, "layout": "nk", "bias": True, "out": "bf16"},
        # one expert layer, 8 experts of 4096 x 14336: a decode step, a serving batch, a prefill batch
        {"name": "moe_decode_16_tokens", "kind": "grouped", "tokens": 16, "top_k": 2, "e": 8, "k": 4096, "n": 14336,
         "layout": "packed", "zipf": 0.0, "bias": False},
        {"name": "moe_1024_tokens", "kind": "grouped", "tokens": 1024, "top_k": 2, "e": 8, "k": 4096, "n": 14336,
         "layout": "packed", "zipf": 0.0, "bias": False},
        {"name": "moe_prefill_4096_tokens", "kind": "grouped", "tokens": 4096, "top_k": 2, "e": 8, "k": 4096, "n": 14336,
         "layout": "packed", "zipf": 0.0, "bias": False},
        # 64 small experts, unevenly used, weights as they are stored
        {"name": "moe_64_experts_skewed", "kind": "grouped", "tokens": 8192, "top_k": 6, "e": 64, "k": 2048, "n": 2816,
         "layout": "kn", "zipf": 1.2, "bias": False},
        # 16-bit activations: decode on 8-bit weights, prefill on 8-bit weights, decode on 4-bit weights
        {"name": "a16w8_decode_16_tokens", "kind": "weight_only", "tokens": 16, "top_k": 2, "e": 8, "k": 4096, "n": 14336,
         "layout": "kn", "bits": 8, "x": "bf16", "offset": True},
        {"name": "a16w8_2048_tokens", "kind": "weight_only", "tokens": 2048, "top_k": 2, "e": 8, "k": 4096, "n": 14336,
         "layout": "packed", "bits": 8, "x": "bf16", "offset": True},
        {"name": "a16w4_16_tokens", "kind": "weight_only", "tokens": 16, "top_k": 2, "e": 8, "k": 4096, "n": 14336,
         "layout": "kn", "bits": 4, "x": "f16", "offset": True},
        # int8 activations on 4-bit weights, a serving batch
        {"name": "a8w4_128_tokens", "kind": "a8w4", "tokens": 128, "top_k": 2, "e": 8, "k": 4096, "n": 14336, "out": "bf16"},
        # a few rows over 256 experts with K-group scales
        {"name": "w4_32_rows_256_experts", "kind": "w4", "rows": 32, "e": 256, "k": 7168, "n": 256, "group": 256},
        # the operators of an expert layer in a row, serving batch, odd token count
        {"name": "moe_ffn_509_tokens", "kind": "moe_ffn", "tokens": 509, "top_k": 8, "e": 64, "hidden": 2048, "inter": 1408},
    ]


def _log_int(rng, lo, hi, step=1):
    return max(lo, min(hi, step * round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)))


def draw(rng):
    while True:
        c = _draw(rng)
        rows, weights, ops_ = _size(c)
        # few tokens over more weights than the largest listed layer, or more work than its prefill, is not drawn
        if weights <= _MAX_WEIGHTS and ops_ <= (_MAX_OPS / 2 if c["kind"] == "weight_only" else _MAX_OPS):
            return c


def _draw(rng):
    kind = rng.choice(["dense", "dense", "grouped", "grouped", "grouped", "weight_only", "weight_only", "a8w4", "w4", "moe_ffn"])
    if kind == "dense":
        return {"kind": kind, "m": _log_int(rng, 1, 4096), "k": _log_int(rng, 1024, 8192, 32), "n": _log_int(rng, 1024, 14336, 16),
                "layout": rng.choice(["kn", "nk", "packed"]), "bias": rng.random() < 0.5, "out": rng.choice(["bf16", "f16"])}
    if kind == "w4":
        g = rng.choice([128, 256])
        return {"kind": kind, "rows": _log_int(rng, 1, 64), "e": rng.choice([64, 128, 256]), "k": _log_int(rng, 512, 8192, g),
                "n": _log_int(rng, 128, 7168, 16), "group": g}
    e = rng.choice([8, 16, 32, 64, 128])
    top_k = rng.choice([1, 2, 4, 6, 8])
    tokens = _log_int(rng, 1, 4096)
    if kind == "moe_ffn":
        return {"kind": kind, "tokens": tokens, "top_k": rng.choice([1, 2, 4, 8]), "e": e, "hidden": rng.choice([2048, 5120, 7168]),
                "inter": _log_int(rng, 512, 4096, 32)}
    c = {"kind": kind, "tokens": tokens, "top_k": top_k, "e": e, "k": _log_int(rng, 512, 8192, 32), "n": _log_int(rng, 512, 14336, 16)}
    if kind == "grouped":
        c.update(layout=rng.choice(["kn", "nk", "packed", "packed"]), zipf=rng.choice([0.0, 0.0, 0.6, 1.2]), bias=rng.random() < 0.3)
    elif kind == "weight_only":
        bits = rng.choice([8, 8, 4])
        c.update(layout="kn" if bits == 4 else rng.choice(["kn", "packed"]), bits=bits, x=rng.choice(["bf16", "f16"]), offset=rng.random() < 0.7)
    else:
        c.update(out=rng.choice(["bf16", "f16"]))
    return c


def _size(c):
    """(rows, weight elements, operations) of one pass."""
    if c["kind"] == "dense":
        rows, weights, per_row = c["m"], c["k"] * c["n"], c["k"] * c["n"]
    elif c["kind"] == "w4":
        rows, weights, per_row = c["rows"], c["e"] * c["k"] * c["n"], c["k"] * c["n"]
    elif c["kind"] == "moe_ffn":
        rows = c["tokens"] * c["top_k"]
        weights, per_row = 2 * c["e"] * c["hidden"] * c["inter"], 2 * c["hidden"] * c["inter"]
    else:
        rows, weights, per_row = c["tokens"] * c["top_k"], c["e"] * c["k"] * c["n"], c["k"] * c["n"]
    return rows, weights, 2.0 * rows * per_row


def _popularity(e, zipf):
    p = [1.0 / (i + 1) ** zipf for i in range(e)]
    return [v / sum(p) for v in p]


def _experts_hit(tokens, top_k, e, zipf):
    """Experts that hold rows, on average over the routings (what is read of the weights depends on it)."""
    return sum(1.0 - (1.0 - min(1.0, p * top_k)) ** tokens for p in _popularity(e, zipf))


class _Inputs:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def int8(self, *shape):
        return torch.randint(-127, 128, shape, generator=self.g, device="cuda", dtype=torch.int8)

    def nibbles(self, *shape):
        return torch.randint(-128, 128, shape, generator=self.g, device="cuda", dtype=torch.int8)

    def uniform(self, lo, hi, *shape):
        return torch.rand(shape, generator=self.g, device="cuda") * (hi - lo) + lo

    def normal(self, dtype, *shape):
        return torch.randn(shape, generator=self.g, device="cuda").to(dtype)

    def experts(self, tokens, top_k, e, zipf):
        """int32 [tokens, top_k]: the experts of every token, most wanted first."""
        logits = torch.randn((tokens, e), generator=self.g, device="cuda")
        logits += torch.tensor([math.log(p) for p in _popularity(e, zipf)], device="cuda")
        return logits.topk(top_k, dim=1).indices.to(torch.int32)

    def group_list(self, tokens, top_k, e, zipf):
        """int64 [e]: where each expert's rows end once the rows are sorted by expert."""
        counts = torch.bincount(self.experts(tokens, top_k, e, zipf).flatten().long(), minlength=e)
        return counts.cumsum(0)


def _weight(w, layout, n):
    """int8 [..., K, N] bytes in the layout the case asks for."""
    if layout == "nk":
        return w.transpose(-1, -2).contiguous()
    return ops.trans_data(w, transdata_type=1) if layout == "packed" else w


def prepare(case, seed):
    c, r = case, _Inputs(seed)
    s = {"kind": c["kind"]}
    if c["kind"] == "dense":
        s.update(x=r.int8(c["m"], c["k"]), w=_weight(r.int8(c["k"], c["n"]), c["layout"], c["n"]), scale=r.uniform(1e-3, 1e-2, c["n"]),
                 bias=torch.randint(-1000, 1001, (c["n"],), generator=r.g, device="cuda", dtype=torch.int32) if c["bias"] else None,
                 transposed=c["layout"] == "nk", format="FRACTAL_NZ" if c["layout"] == "packed" else "ND", out=_HALF[c["out"]])
    elif c["kind"] == "w4":
        # sorted random boundaries over the rows: most experts hold none
        cuts = torch.randint(0, c["rows"] + 1, (c["e"] - 1,), generator=r.g, device="cuda").sort().values
        ends = torch.cat([cuts, torch.tensor([c["rows"]], device="cuda")]).to(torch.int32)
        s.update(x=r.int8(c["rows"], c["k"]), w=r.nibbles(c["e"], c["n"], c["k"] // 2), group_list=ends,
                 bias=torch.zeros((c["e"], c["n"]), device="cuda"), x_scale=r.uniform(1e-3, 1e-2, c["rows"]),
                 w_scale=r.uniform(1e-3, 1e-2, c["e"], c["k"] // c["group"], c["n"]))
    elif c["kind"] == "moe_ffn":
        e, h, i, t = c["e"], c["hidden"], c["inter"], c["tokens"]
        s.update(e=e, x=r.normal(torch.bfloat16, t, h), experts=r.experts(t, c["top_k"], e, 0.0),
                 probs=torch.softmax(torch.randn((t, c["top_k"]), generator=r.g, device="cuda"), 1).to(torch.bfloat16),
                 up=r.int8(e, h, i), up_scale=r.uniform(1e-4, 1e-3, e, i), down=r.int8(e, i, h),
                 down_scale=r.uniform(1e-4, 1e-3, e, h).to(torch.bfloat16))
    else:
        e, k, n, rows = c["e"], c["k"], c["n"], c["tokens"] * c["top_k"]
        ends = r.group_list(c["tokens"], c["top_k"], e, c.get("zipf", 0.0))
        if c["kind"] == "grouped":
            s.update(x=r.int8(rows, k), w=_weight(r.int8(e, k, n), c["layout"], n), group_list=ends.to(torch.int32),
                     scale=r.uniform(1e-3, 1e-2, e, n), x_scale=r.uniform(1e-3, 1e-2, rows), transposed=c["layout"] == "nk",
                     bias=torch.randint(-1000, 1001, (e, n), generator=r.g, device="cuda", dtype=torch.int32) if c["bias"] else None)
        elif c["kind"] == "weight_only":
            dt = _HALF[c["x"]]
            w = ops.as_qint4x2(r.nibbles(e, k, n // 2)) if c["bits"] == 4 else _weight(r.int8(e, k, n), c["layout"], n)
            s.update(x=r.normal(dt, rows, k), w=w, group_list=ends, scale=r.uniform(1e-4, 1e-3, e, n).to(dt),
                     offset=torch.randint(-8, 9, (e, n), generator=r.g, device="cuda").to(dt) if c["offset"] else None,
                     format="FRACTAL_NZ" if c["layout"] == "packed" else "ND")
        else:
            scale = r.uniform(1e-3, 1e-2, e, 1, n).view(torch.int32).to(torch.int64).view(torch.uint64)   # float32 bits in 64-bit words
            s.update(x=r.int8(rows, k), w=ops.as_qint4x2(r.nibbles(e, k, n // 2)), group_list=ends, scale=scale,
                     x_scale=r.uniform(1e-3, 1e-2, rows, 1), out=_HALF[c["out"]])
    return s


def run(state):
    s = state
    if s["kind"] == "dense":
        return ops.quant_batch_matmul(s["x"], s["w"], s["scale"], bias=s["bias"], transpose_x2=s["transposed"], x2_format=s["format"],
                                      output_dtype=s["out"])
    if s["kind"] == "grouped":
        return ops.grouped_matmul(s["x"], s["w"], s["group_list"], bias=s["bias"], scale=s["scale"], per_token_scale=s["x_scale"],
                                  transpose_b=s["transposed"], output_dtype=torch.bfloat16)
    if s["kind"] == "weight_only":
        return ops.grouped_matmul_v4_cops([s["x"]], [s["w"]], antiquant_scale=[s["scale"]],
                                          antiquant_offset=[s["offset"]] if s["offset"] is not None else None,
                                          group_list=s["group_list"], split_item=3, group_type=0, weight_format=s["format"])[0]
    if s["kind"] == "a8w4":
        return ops.grouped_matmul_v4_cops([s["x"]], [s["w"]], scale=[s["scale"]], per_token_scale=[s["x_scale"]],
                                          group_list=s["group_list"], split_item=3, group_type=0, output_dtype=s["out"])[0]
    if s["kind"] == "w4":
        return ops.grouped_matmul_w4(s["x"], s["w"], s["group_list"], s["bias"], s["x_scale"], s["w_scale"])
    rows, row_scale, row_idx, ends = ops.moe_init_routing_quant(s["x"], s["experts"], s["e"], 1)
    ends = ends.to(torch.int64)
    h = ops.grouped_matmul_v4_cops([rows], [s["up"]], scale=[s["up_scale"]], per_token_scale=[row_scale], group_list=ends, split_item=3,
                                   group_type=0, act_type=5, output_dtype=torch.bfloat16)[0]
    y = ops.grouped_matmul_v4_cops([h], [s["down"]], antiquant_scale=[s["down_scale"]], group_list=ends, split_item=3, group_type=0)[0]
    return ops.moe_token_unpermute(y, row_idx, s["probs"])


def work(case):
    c = case
    rows, weights, ops_ = _size(c)
    if c["kind"] == "dense":
        return {"bytes": rows * c["k"] + weights + 2 * rows * c["n"] + 4 * c["n"] * (2 if c["bias"] else 1), "flops": ops_}
    if c["kind"] == "w4":
        hit = c["e"] * (1.0 - (1.0 - 1.0 / c["e"]) ** rows)
        return {"bytes": rows * (c["k"] + 4 + 2 * c["n"]) + hit * c["n"] * (c["k"] // 2 + 4 * c["k"] // c["group"]) + 4 * c["e"], "flops": ops_}
    hit = _experts_hit(c["tokens"], c["top_k"], c["e"], c.get("zipf", 0.0))
    if c["kind"] == "moe_ffn":
        # tokens in and out, the experts and probabilities, both weight matrices of the experts that are hit
        t, h, i = c["tokens"], c["hidden"], c["inter"]
        return {"bytes": 4 * t * h + 6 * rows + hit * (2 * h * i + 4 * i + 2 * h), "flops": ops_}
    k, n = c["k"], c["n"]
    if c["kind"] == "grouped":
        return {"bytes": rows * (k + 4 + 2 * n) + hit * n * (k + 4 + (4 if c["bias"] else 0)) + 4 * c["e"], "flops": ops_}
    if c["kind"] == "weight_only":
        return {"bytes": rows * (2 * k + 2 * n) + hit * n * (k * c["bits"] / 8 + (4 if c["offset"] else 2)) + 8 * c["e"], "flops": ops_}
    return {"bytes": rows * (k + 4 + 2 * n) + hit * n * (k / 2 + 8) + 8 * c["e"], "flops": ops_}


def tolerance(case):
    """Integer accumulation and a fixed order of roundings behind it: the same bits.  The others sum in float32 and round
    to 16 bits; against a float64 evaluation the 2-norm of the difference measures 1.66e-3 of the result for bfloat16 and
    2.1e-4 for float16 outputs (the output rounding, four times that is allowed), and 4.6e-3 for the whole layer, whose
    running sums are kept in bfloat16."""
    c = case
    if c["kind"] in ("dense", "grouped", "a8w4"):
        return "exact"
    if c["kind"] == "moe_ffn":
        return {"rel": 1e-2}
    return {"rel": 7e-3 if c.get("x") == "bf16" else 9e-4}
