"""What the witness generation of a DeepSeek-V3 forward pass asks of this library, as timed cases.

Every case goes through the operator API of `kernel.py`, chained as the layers chain it.  The kinds:

  linear    one projection: int64 activations against an int32 or int64 weight matrix, quotient and remainder
  mla       the attention block of one layer: residual and norm, LoRA projections, RoPE, absorbed attention over the
            cache, output projection.  One token is a decoding step, more are a prompt
  scores    the attention core alone on a whole prompt: scores, masked softmax, probabilities times values
  ffn       a gated feed-forward: gate and up projection, SiLU product, down projection; with `norm`, the residual and
            the norm in front of it as well
  moe       a mixture layer: gate, routing, routed experts, shared expert
  rowwise   one of the memory-bound operators on its own
  quantize  a checkpoint matrix in block-scaled fp8 turned into int32 weights

Sizes are those of the 671 B configuration (dim 7168, 128 heads, LoRA ranks 1536 and 512, head parts 128 / 64 / 128,
feed-forward 18432 and 2048, 256 experts of which 8 serve a token) and of the library's benchmark.  Fixed-point positions
follow the model's ladder: residual stream Q31, attention inputs Q19-Q21, cache and feed-forward Q23, RoPE table Q42,
int32 weights at per-tensor scales.  Everything is integer arithmetic, so results are compared bit for bit.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.abspath("zk-deepseek_amd"))
import kernel as K  # noqa: E402

DIM, HEADS, Q_LORA, KV_LORA, NOPE, ROPE, V_DIM = 7168, 128, 1536, 512, 128, 64, 128
DENSE, INTER, EXPERTS, TOPK, GROUPS, TOPK_GROUPS, VOCAB = 18432, 2048, 256, 8, 8, 4, 129280
MAX_TOKENS = 500            # rows of the RMS statistic's buffer: the most tokens a pass takes
MASK = -(64 << 36)

# the projections of the model as (in, out)
PROJECTIONS = ((DIM, Q_LORA), (Q_LORA, HEADS * NOPE), (Q_LORA, HEADS * ROPE), (DIM, KV_LORA + ROPE), (HEADS * V_DIM, DIM),
               (DIM, DENSE), (DENSE, DIM), (DIM, INTER), (INTER, DIM), (DIM, EXPERTS))


def listed():
    return [
        # the down-projection to the cache on a short prompt: the benchmark's first shape, a stream over a small matrix
        {"name": "linear_16x7168x576", "kind": "linear", "rows": 16, "k": DIM, "n": KV_LORA + ROPE, "w32": False,
         "a_bits": 20, "w_bits": 16, "shift": 29, "div": 1},
        # the benchmark's headline product: a long prompt against the widest projection
        {"name": "linear_512x7168x18432", "kind": "linear", "rows": 512, "k": DIM, "n": DENSE, "w32": False,
         "a_bits": 20, "w_bits": 16, "shift": 29, "div": 1},
        # the vocabulary head, once per generated token, weights divided by 256
        {"name": "head_1x7168x129280", "kind": "linear", "rows": 1, "k": DIM, "n": VOCAB, "w32": False,
         "a_bits": 26, "w_bits": 40, "shift": 43, "div": 256},
        # attention of one layer in a decoding step
        {"name": "mla_decode_1_of_779", "kind": "mla", "tokens": 1, "context": 779},
        # attention of one layer on a prompt of ordinary, odd length
        {"name": "mla_prompt_243", "kind": "mla", "tokens": 243, "context": 243},
        # the attention core on the longest prompt that the benchmark has
        {"name": "scores_1024", "kind": "scores", "tokens": 1024},
        # one expert's feed-forward on a batch of tokens, int64 weights (benchmark)
        {"name": "ffn_expert_128", "kind": "ffn", "tokens": 128, "inter": INTER, "w32": False, "norm": False},
        # the dense feed-forward of the first layers on a long, odd prompt
        {"name": "ffn_dense_411", "kind": "ffn", "tokens": 411, "inter": DENSE, "w32": True, "norm": True},
        # a mixture layer in a decoding step, and on a prompt that reaches every expert
        {"name": "moe_decode_1", "kind": "moe", "tokens": 1, "experts": EXPERTS},
        {"name": "moe_prompt_256", "kind": "moe", "tokens": 256, "experts": EXPERTS},
        # the activation of the dense layers (benchmark), bound by memory alone
        {"name": "silu_512x18432", "kind": "rowwise", "op": "silu_q23", "rows": 512, "width": DENSE},
        # loading an expert's weights from the checkpoint
        {"name": "quantize_2048x7168", "kind": "quantize", "rows": INTER, "cols": DIM},
    ]


def _log(rng, lo, hi):
    """a whole number from lo to hi, spread over the logarithm"""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("linear", "linear", "linear", "mla", "mla", "scores", "ffn", "ffn", "moe", "rowwise", "quantize"))
    if kind == "linear":
        rows = _log(rng, 1, 512)
        k, n = rng.choice(PROJECTIONS)
        if rng.random() < 0.4:          # not the model's: odd sizes, rows of weights off the 16-byte grid among them
            k, n = _log(rng, 200, 16384), _log(rng, 200, 20000)
        w32 = rng.random() < 0.6
        return {"kind": kind, "rows": rows, "k": k, "n": n, "w32": w32, "a_bits": rng.choice((20, 23, 27, 31)),
                "w_bits": rng.choice((24, 28, 30)) if w32 else rng.choice((16, 20, 24)), "shift": rng.choice((23, 29, 30, 33)), "div": 1}
    if kind == "mla":
        if rng.random() < 0.5:
            return {"kind": kind, "tokens": 1, "context": _log(rng, 16, 1024)}
        tokens = _log(rng, 2, MAX_TOKENS)
        return {"kind": kind, "tokens": tokens, "context": tokens}
    if kind == "scores":
        return {"kind": kind, "tokens": _log(rng, 32, 1024)}
    if kind == "ffn":
        tokens, w32 = _log(rng, 1, MAX_TOKENS), rng.random() < 0.7
        return {"kind": kind, "tokens": tokens, "inter": rng.choice((INTER, DENSE)) if w32 else INTER, "w32": w32, "norm": rng.random() < 0.5}
    if kind == "moe":
        return {"kind": kind, "tokens": _log(rng, 1, 300), "experts": rng.choice((64, 128))}
    if kind == "rowwise":
        op = rng.choice(("softmax_q19", "softmax_q21", "silu_q23", "sigmoid_q23", "silu_q25", "rms", "rope"))
        rows, width = _log(rng, 1, MAX_TOKENS), rng.choice((KV_LORA, Q_LORA, DIM, DENSE, _log(rng, 100, 20000)))
        if op.startswith("softmax"):
            rows, width = _log(rng, HEADS, 100000), _log(rng, 16, 1500)
        if op == "rope":
            width = ROPE * rng.choice((1, HEADS))
        return {"kind": kind, "op": op, "rows": rows, "width": width}
    return {"kind": kind, "rows": _log(rng, 100, 18432), "cols": rng.choice((Q_LORA, DIM, _log(rng, 100, 16384)))}


# ---- inputs ------------------------------------------------------------------------------------------------------------
class _Draw:
    """seeded tensors on the GPU"""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(int(seed))

    def uniform(self, bits, *shape, dtype=torch.int64):
        return torch.randint(-(1 << bits), 1 << bits, shape, generator=self.gen, dtype=dtype, device="cuda")

    def between(self, lo, hi, *shape, dtype=torch.int64):
        return torch.randint(lo, hi, shape, generator=self.gen, dtype=dtype, device="cuda")

    def normal(self, bits, *shape, dtype=torch.int64):
        """bell-shaped with a deviation of 2^bits; what would leave an int32 is cut to 31 bits"""
        t = torch.randn(shape, generator=self.gen, device="cuda", dtype=torch.float32).mul_(float(2 ** bits))
        return t.clamp_(-2.0e9, 2.0e9).to(dtype) if dtype == torch.int32 else t.to(dtype)

    def weights(self, n, k, w32=True):
        """int32 weights of the model (about 28.5 bits at a deviation of 2^26) or the benchmark's int64 ones (17 bits)"""
        return self.normal(26, n, k, dtype=torch.int32) if w32 else self.uniform(16, n, k)

    def rope_table(self, tokens):
        ang = torch.rand((1, tokens, 1, ROPE // 2), generator=self.gen, device="cuda", dtype=torch.float64) * (2 * math.pi)
        return torch.stack([torch.round(torch.cos(ang) * 2.0 ** 42), torch.round(torch.sin(ang) * 2.0 ** 42)], -1).to(torch.int64)


def _tables():
    """the exponential tables a program fills once"""
    if K.EXP2_FRAC_LUT_Q19 is None:
        K.softmax_init_q19()
        K.softmax_init_q21()
        K.silu_init_q23()
        K.silu_init_q25()


def _causal(tokens, context):
    """additive mask [tokens, context] of the last `tokens` positions"""
    return torch.full((tokens, context), MASK, dtype=torch.int64, device="cuda").triu_(1 + context - tokens)


def prepare(case, seed):
    _tables()
    d = _Draw(seed)
    s = {"case": case}
    kind = case["kind"]
    if kind == "linear":
        s["x"] = d.uniform(case["a_bits"], 1, case["rows"], case["k"])
        s["w"] = d.uniform(case["w_bits"], case["n"], case["k"], dtype=torch.int32 if case["w32"] else torch.int64)
    elif kind == "mla":
        t, ctx = case["tokens"], case["context"]
        s.update(x=d.normal(31, t, DIM), y=d.normal(22, t, DIM), attn_norm=d.between(1 << 18, 1 << 20, DIM, dtype=torch.int32),
                 q_norm=d.between(1 << 18, 1 << 20, Q_LORA, dtype=torch.int32), kv_norm=d.between(1 << 22, 1 << 24, KV_LORA, dtype=torch.int32),
                 wq_a=d.weights(Q_LORA, DIM), wq_b1=d.weights(HEADS * NOPE, Q_LORA), wq_b2=d.weights(HEADS * ROPE, Q_LORA),
                 wkv_a1=d.weights(KV_LORA, DIM), wkv_a2=d.weights(ROPE, DIM), wo=d.weights(DIM, HEADS * V_DIM),
                 wkv_b1=d.weights(HEADS * NOPE, KV_LORA).view(HEADS, NOPE, KV_LORA), wkv_b2=d.weights(HEADS * V_DIM, KV_LORA).view(HEADS, V_DIM, KV_LORA),
                 kv_cache=d.normal(23, 1, ctx, KV_LORA), pe_cache=d.normal(22, 1, ctx, ROPE), freqs=d.rope_table(t),
                 mask=_causal(t, ctx) if t > 1 else None)
    elif kind == "scores":
        t = case["tokens"]
        s.update(q_abs=d.normal(20, 1, t, HEADS, KV_LORA), q_pe=d.normal(20, 1, t, HEADS, ROPE), kv=d.normal(23, 1, t, KV_LORA),
                 pe=d.normal(22, 1, t, ROPE), mask=_causal(t, t))
    elif kind == "ffn":
        t, inter, w32 = case["tokens"], case["inter"], case["w32"]
        s.update(w1=d.weights(inter, DIM, w32), w3=d.weights(inter, DIM, w32), w2=d.weights(DIM, inter, w32))
        if case["norm"]:
            s.update(x=d.normal(31, t, DIM), y=d.normal(20, t, DIM), norm=d.between(1 << 21, 1 << 23, DIM, dtype=torch.int32))
        else:
            s["x"] = d.normal(22, 1, t, DIM) if w32 else d.uniform(20, 1, t, DIM)
    elif kind == "moe":
        t, e = case["tokens"], case["experts"]
        s.update(x=d.normal(22, t, DIM), gate=d.weights(e, DIM), bias=d.uniform(18, e, dtype=torch.int32),
                 w1=[d.weights(INTER, DIM) for _ in range(e)], w3=[d.weights(INTER, DIM) for _ in range(e)], w2=[d.weights(DIM, INTER) for _ in range(e)],
                 sw1=d.weights(INTER, DIM), sw3=d.weights(INTER, DIM), sw2=d.weights(DIM, INTER))
        s["tables"] = tuple(K.pointer_table(s[n]) for n in ("w1", "w3", "w2"))
    elif kind == "rowwise":
        op, rows, width = case["op"], case["rows"], case["width"]
        if op.startswith("softmax"):
            x = d.normal(int(op[-2:]) + 2, 1, (rows + HEADS - 1) // HEADS, HEADS, width)
            if width > 1:               # a prompt's scores: part of a row is masked
                x[:, ::2, :, width // 2:] += MASK
            s["x"] = x
        elif op == "rms":
            s.update(x=d.normal(31, rows, width), w=d.between(1 << 18, 1 << 20, width, dtype=torch.int32))
        elif op == "rope":
            s.update(x=d.normal(20, 1, rows, width // ROPE, ROPE // 2, 2), freqs=d.rope_table(rows))
        else:
            s["x"] = d.normal(int(op[-2:]) + 1, 1, rows, width).clamp_(-(20 << int(op[-2:])), 20 << int(op[-2:]))
    else:
        rows, cols = case["rows"], case["cols"]
        s["w"] = torch.randn((rows, cols), generator=d.gen, device="cuda").mul_(40.0).to(torch.float8_e4m3fn)
        s["scale"] = torch.rand(((rows + 127) // 128, (cols + 127) // 128), generator=d.gen, device="cuda").mul_(4e-4).add_(1e-5)
    return s


# ---- one pass ----------------------------------------------------------------------------------------------------------
def _project(x, w, shift):
    return K.int64_bmm_broadcast(x, w, 1, 1, shift, want_remainder=False)[0]


def _gated(x, w1, w3, w2, shift1, shift2):
    g, u = _project(x, w1, shift1), _project(x, w3, shift1)
    h = torch.empty_like(g)
    K.silu_mul_q23(g, u, h)
    return _project(h, w2, shift2)


def _attend(q_abs, q_pe, kv, pe, mask):
    s1 = K.einsum_bshc_btc_bsht(q_abs, kv, 23)
    s2 = K.einsum_bshc_btc_bsht(q_pe, pe, 21)
    scores, p = torch.empty_like(s1), torch.empty_like(s1)
    K.softmax_q19_scores(s1, s2, mask, p, scores)
    return scores, p, K.einsum_bsht_btc_bshc(p, kv, 23)


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "linear":
        return K.int64_bmm_broadcast(s["x"], s["w"], 1, case["div"], case["shift"])
    if kind == "mla":
        t, ctx = case["tokens"], case["context"]
        x, a, _ = K.RMS_Norm_residual_int64(s["x"], s["y"], 8, s["attn_norm"], 1, DIM, host_rms=False)
        a = a.unsqueeze(0)
        q_down, q_rem = K.int64_bmm_broadcast(a, s["wq_a"], 1, 1, 30)
        q, _ = K.RMS_Norm_int64(q_down[0], s["q_norm"], 1, Q_LORA, host_rms=False)
        q = q.unsqueeze(0)
        q_nope = _project(q, s["wq_b1"], 30).view(1, t, HEADS, NOPE)
        q_pe = K.complex_int64_mul_broadcast(_project(q, s["wq_b2"], 30).view(1, t, HEADS, ROPE // 2, 2), s["freqs"])
        kv, kv_rem = K.int64_bmm_broadcast(a, s["wkv_a1"], 1, 1, 29)
        k_pe = K.complex_int64_mul_broadcast(_project(a, s["wkv_a2"], 29).view(1, t, 1, ROPE // 2, 2), s["freqs"])
        kv, _ = K.RMS_Norm_int64(kv[0], s["kv_norm"], 1, KV_LORA, host_rms=False)
        s["kv_cache"][:, ctx - t:] = kv
        s["pe_cache"][:, ctx - t:] = k_pe.view(1, t, ROPE)
        q_abs = K.einsum_bshd_hdc_bshc(q_nope, s["wkv_b1"], 30)
        scores, p, o = _attend(q_abs, q_pe.view(1, t, HEADS, ROPE), s["kv_cache"], s["pe_cache"], s["mask"])
        o = K.einsum_bshc_hdc_bshd(o, s["wkv_b2"], 30)
        y = _project(o.view(1, t, HEADS * V_DIM), s["wo"], 32)
        return {"x": x, "y": y, "q_rem": q_rem, "kv_rem": kv_rem, "scores": scores, "p": p, "kv": s["kv_cache"], "pe": s["pe_cache"]}
    if kind == "scores":
        return _attend(s["q_abs"], s["q_pe"], s["kv"], s["pe"], s["mask"])
    if kind == "ffn":
        # shifts that bring every stage back to Q23 at these widths
        shift1, shift2 = (31, 33 if case["inter"] == DENSE else 32) if case["w32"] else (16, 16)
        if not case["norm"]:
            return _gated(s["x"], s["w1"], s["w3"], s["w2"], shift1, shift2)
        x, f, _ = K.RMS_Norm_residual_int64(s["x"], s["y"], 12, s["norm"], 1, DIM, host_rms=False)
        return x, _gated(f.unsqueeze(0), s["w1"], s["w3"], s["w2"], shift1, shift2)
    if kind == "moe":
        x = s["x"].unsqueeze(0)
        shared = _gated(x, s["sw1"], s["sw3"], s["sw2"], 31, 32)
        logits, rem = K.int64_bmm_broadcast(x, s["gate"], 1, 1, 31)
        scores, weights, indices = K.gate_sigmoid_route(logits[0], s["bias"], GROUPS, TOPK_GROUPS, TOPK)
        y = K.moe_experts(s["x"], weights, indices, *s["tables"], True, INTER, 31, 32)
        return {"y": y + shared[0], "rem": rem, "scores": scores, "weights": weights, "indices": indices}
    if kind == "rowwise":
        op = case["op"]
        if op == "rms":
            c, r = K.RMS_Norm_int64(s["x"], s["w"], 1, case["width"], host_rms=False)
            return c, r[:case["rows"]]
        if op == "rope":
            return K.complex_int64_mul_broadcast(s["x"], s["freqs"])
        out = torch.empty_like(s["x"])
        getattr(K, op)(s["x"], out)
        return out
    return K.quantize_fp8_weight(s["w"], s["scale"], 28)


# ---- what a pass cannot do without -------------------------------------------------------------------------------------
def _gemm(rows, k, n, wbytes, out=1):
    """bytes and flops of a product on its own: activations, weights, `out` int64 outputs per element"""
    return 8.0 * rows * k + wbytes * k * n + 8.0 * out * rows * n, 2.0 * rows * k * n


def work(case):
    kind = case["kind"]
    if kind == "linear":
        b, f = _gemm(case["rows"], case["k"], case["n"], 4.0 if case["w32"] else 8.0, 2)
    elif kind == "mla":
        t, ctx = case["tokens"], case["context"]
        weights = DIM * Q_LORA + Q_LORA * HEADS * (NOPE + ROPE) + DIM * (KV_LORA + ROPE) + HEADS * KV_LORA * (NOPE + V_DIM) + HEADS * V_DIM * DIM
        f = 2.0 * t * weights + 2.0 * t * HEADS * ctx * (2 * KV_LORA + ROPE)
        # weights, residual stream in and out, the output, remainders, cache, the two kept score tensors
        b = 4.0 * weights + 8.0 * t * (4 * DIM + Q_LORA + KV_LORA) + 8.0 * (ctx + t) * (KV_LORA + ROPE) + 16.0 * t * HEADS * ctx
    elif kind == "scores":
        t = case["tokens"]
        f = 2.0 * t * t * HEADS * (2 * KV_LORA + ROPE)
        b = 8.0 * t * HEADS * (2 * KV_LORA + ROPE) + 8.0 * t * (KV_LORA + ROPE + t) + 16.0 * t * t * HEADS
    elif kind == "ffn":
        t, inter = case["tokens"], case["inter"]
        f = 6.0 * t * DIM * inter
        b = 3.0 * (4.0 if case["w32"] else 8.0) * DIM * inter + 8.0 * t * DIM * (4 if case["norm"] else 2)
    elif kind == "moe":
        t, e = case["tokens"], case["experts"]
        hit = e * (1.0 - (1.0 - TOPK / e) ** t)         # experts that some token chooses, on average
        f = 2.0 * t * DIM * (3.0 * INTER * (TOPK + 1) + e)
        b = 4.0 * DIM * (3.0 * INTER * (hit + 1) + e) + 16.0 * t * DIM + 16.0 * t * (e + TOPK)
    elif kind == "rowwise":
        rows, width = case["rows"], case["width"]
        if case["op"].startswith("softmax"):
            rows = (rows + HEADS - 1) // HEADS * HEADS
        b, f = 16.0 * rows * width + 8.0 * width, 8.0 * rows * width
    else:
        b, f = 5.0 * case["rows"] * case["cols"], 2.0 * case["rows"] * case["cols"]
    return {"bytes": b, "flops": f}


def tolerance(case):
    """integers all through, the fp8 conversion included: every correct implementation gives the same bits"""
    return "exact"
