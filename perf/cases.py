"""The calls whose speed counts in use, one pass each through the framework's
public functions: the per-layer ops, the 4-bit projections, the routed experts
and the gated-delta recurrence, in prefill and in decode.

Shapes are those of the workloads in bench.py (Llama-3.2-1B, Qwen3-8B,
Gemma-2-9B and Qwen3-Next layers); drawn cases spread the batch, sequence and
width of the same calls over their whole range. Weights are 4-bit, group 64,
scaled so that a projection of unit-variance rows has about unit variance.
"""
from __future__ import annotations

import math

import torch

import higgs_amd as H
from higgs_amd import ops

BF16, F32, F64 = torch.bfloat16, torch.float32, torch.float64
GROUP = 64

# Qwen3-Next's token mixer and routed experts (bench.py's decode workloads)
NEXT_HIDDEN, NEXT_EXPERTS, NEXT_TOP_K, NEXT_EXPERT_DIM = 2048, 512, 10, 512
NEXT_HK, NEXT_DK, NEXT_HV, NEXT_DV = 16, 128, 32, 128

# The largest amount of arithmetic and of traffic that a case has.
MAX_FLOPS = 2 * 4096 * 12288 * 2048
MAX_BYTES = 2800 << 20


def listed():
    return [
        # the hidden-state norm of 512 tokens: the smallest call, all latency
        {"name": "norm_512", "kind": "norm", "rows": 512, "hidden": 2048, "add": False},
        # Gemma-2-9B's memory-bound prefill ops over 4 x 4096 tokens (bench.py's default)
        {"name": "gemma_ops_16384", "kind": "gemma_ops", "batch": 4, "seq": 4096,
         "hidden": 3584, "vocab": 256000, "inter": 14336, "heads": 16, "kv_heads": 8,
         "head_dim": 256},
        # Qwen3-8B attention prologue over 8 x 2048 tokens: q/k norm, RoPE, transpose
        {"name": "qk_rope_16384", "kind": "qk_rope", "batch": 8, "seq": 2048, "heads": 32,
         "kv_heads": 8, "head_dim": 128, "offset": 0},
        # the row-wise ops of a 48-layer decode step of 64 sequences, in one launch
        {"name": "decode_ops_64", "kind": "decode_ops", "tokens": 64, "layers": 48},
        # one user's next token through a Qwen3-8B MLP: three weight streams
        {"name": "mlp_decode_1", "kind": "mlp", "rows": 1, "hidden": 4096, "inter": 12288},
        # a continuous batch's next token through Qwen3-Next's in_proj_qkvz
        {"name": "linear_decode_64", "kind": "linear", "rows": 64, "n": 12288, "k": 2048},
        # an ordinary prompt of a ragged length through a Qwen3-8B MLP
        {"name": "mlp_prompt_301", "kind": "mlp", "rows": 301, "hidden": 4096, "inter": 12288},
        # a long prompt through in_proj_qkvz: matrix-core bound
        {"name": "linear_prefill_4096", "kind": "linear", "rows": 4096, "n": 12288, "k": 2048},
        # Qwen3-Next's routed experts (gate, up, SwiGLU, down) for one step of 64 sequences
        {"name": "experts_decode_64", "kind": "experts", "tokens": 64, "experts": NEXT_EXPERTS,
         "top_k": NEXT_TOP_K, "hidden": NEXT_HIDDEN, "expert_dim": NEXT_EXPERT_DIM},
        # ... and for a 4096-token prompt
        {"name": "experts_prefill_4096", "kind": "experts", "tokens": 4096,
         "experts": NEXT_EXPERTS, "top_k": NEXT_TOP_K, "hidden": NEXT_HIDDEN,
         "expert_dim": NEXT_EXPERT_DIM},
        # the linear-attention recurrence and its gated norm, one token of 64 sequences
        {"name": "delta_decode_64", "kind": "delta", "batch": 64, "seq": 1},
        # ... and the recurrence over 4 prompts of 512 tokens
        {"name": "delta_prefill_4x512", "kind": "delta", "batch": 4, "seq": 512},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["norm", "gemma_ops", "qk_rope", "decode_ops", "mlp", "linear", "linear",
                       "experts", "experts", "delta", "delta"])
    while True:
        c = _draw(rng, kind)
        w = work(c)
        if w["flops"] <= MAX_FLOPS and w["bytes"] <= MAX_BYTES:
            return c


def _draw(rng, kind):
    if kind == "norm":
        return {"kind": kind, "rows": _log_int(rng, 1, 16384),
                "hidden": rng.choice([2048, 3584, 4096]), "add": rng.random() < 0.5}
    if kind == "gemma_ops":
        return {"kind": kind, "batch": rng.randint(1, 4), "seq": _log_int(rng, 1, 4096),
                "hidden": 3584, "vocab": 256000, "inter": 14336, "heads": 16, "kv_heads": 8,
                "head_dim": 256}
    if kind == "qk_rope":
        return {"kind": kind, "batch": rng.randint(1, 8), "seq": _log_int(rng, 1, 2048),
                "heads": 32, "kv_heads": 8, "head_dim": 128, "offset": rng.choice([0, 1, 2047])}
    if kind == "decode_ops":
        return {"kind": kind, "tokens": _log_int(rng, 1, 64), "layers": 4 * rng.randint(1, 12)}
    if kind == "mlp":
        hidden, inter = rng.choice([(2048, 8192), (3584, 14336), (4096, 12288)])
        return {"kind": kind, "rows": _log_int(rng, 1, 640), "hidden": hidden, "inter": inter}
    if kind == "linear":
        return {"kind": kind, "rows": _log_int(rng, 1, 4096), "n": _log_int(rng, 64, 16384),
                "k": rng.choice([2048, 2048, 3584, 4096, 8192])}
    if kind == "experts":
        return {"kind": kind, "tokens": _log_int(rng, 1, 4096),
                "experts": rng.choice([64, 128, 256, 512]), "top_k": rng.randint(4, 10),
                "hidden": 2048, "expert_dim": rng.choice([512, 1024])}
    if rng.random() < 0.4:
        return {"kind": "delta", "batch": _log_int(rng, 1, 64), "seq": 1}
    return {"kind": "delta", "batch": rng.randint(1, 4), "seq": _log_int(rng, 2, 1024)}


# ------------------------------------------------------------------ inputs
class _Gen:
    def __init__(self, seed):
        self.dev = torch.device("cuda", torch.cuda.current_device())
        self.g = torch.Generator(device=self.dev)
        self.g.manual_seed(seed)

    def randn(self, *shape, mean=0.0, std=1.0, dtype=BF16):
        t = torch.empty(shape, dtype=F32, device=self.dev).normal_(mean, std, generator=self.g)
        return t.to(dtype)

    def uniform(self, lo, hi, *shape, dtype=BF16):
        t = torch.empty(shape, dtype=F32, device=self.dev).uniform_(lo, hi, generator=self.g)
        return t.to(dtype)

    def ints(self, lo, hi, *shape):
        return torch.randint(lo, hi, shape, dtype=torch.int32, device=self.dev, generator=self.g)

    def quantized(self, *shape, std=None):
        """Packed codes, scales and biases of a weight [..., N, K] whose values
        have standard deviation `std` (1 / sqrt(K) unless given): codes uniform
        in 0..15, the bias near the middle of each group's range."""
        *lead, k = shape
        std = 1.0 / math.sqrt(k) if std is None else std
        w = self.ints(-2 ** 31, 2 ** 31 - 1, *lead, k // 8)
        s = self.uniform(0.5, 1.5, *lead, k // GROUP, dtype=F32) * (std / 4.61)
        b = s * self.uniform(-9.0, -6.0, *lead, k // GROUP, dtype=F32)
        return w, s.to(BF16), b.to(BF16)

    def experts(self, tokens, top_k, experts):
        """Distinct experts per token, in router order."""
        r = torch.rand((tokens, experts), device=self.dev, generator=self.g)
        return r.topk(top_k, dim=1).indices.to(torch.int32).contiguous()


def _inputs(case, seed):
    """The tensors of a case, as a dict (the outputs' buffers not among them)."""
    g, kind = _Gen(seed), case["kind"]
    if kind == "norm":
        m, n = case["rows"], case["hidden"]
        return {"x": g.randn(m, n), "r": g.randn(m, n) if case["add"] else None,
                "w": g.randn(n, mean=1.0, std=0.02)}
    if kind == "gemma_ops":
        b, l, hd = case["batch"], case["seq"], case["hidden"]
        d = case["head_dim"]
        return {"table": g.quantized(case["vocab"], hd, std=0.02),
                "ids": g.ints(0, case["vocab"], b, l), "w": g.randn(hd, std=0.02),
                "q": g.randn(b, l, case["heads"], d), "k": g.randn(b, l, case["kv_heads"], d),
                "gate": g.randn(b * l, case["inter"]), "up": g.randn(b * l, case["inter"])}
    if kind == "qk_rope":
        b, l, d = case["batch"], case["seq"], case["head_dim"]
        return {"q": g.randn(b, l, case["heads"], d), "k": g.randn(b, l, case["kv_heads"], d),
                "wq": g.randn(d, mean=1.0, std=0.02), "wk": g.randn(d, mean=1.0, std=0.02)}
    if kind == "mlp":
        hd, it = case["hidden"], case["inter"]
        return {"x": g.randn(case["rows"], hd), "gate": g.quantized(it, hd),
                "up": g.quantized(it, hd), "down": g.quantized(hd, it)}
    if kind == "linear":
        return {"x": g.randn(case["rows"], case["k"]), "w": g.quantized(case["n"], case["k"])}
    if kind == "experts":
        e, hd, it = case["experts"], case["hidden"], case["expert_dim"]
        return {"x": g.randn(case["tokens"], hd), "ids": g.experts(case["tokens"], case["top_k"], e),
                "gate": g.quantized(e, it, hd), "up": g.quantized(e, it, hd),
                "down": g.quantized(e, hd, it)}
    if kind == "delta":
        b, t = case["batch"], case["seq"]
        z = g.randn(b, t, NEXT_HK, 768)[..., 512:].unflatten(-1, (2, NEXT_DV))
        return {"q": g.randn(b, t, NEXT_HK, NEXT_DK), "k": g.randn(b, t, NEXT_HK, NEXT_DK),
                "v": g.randn(b, t, NEXT_HV, NEXT_DV), "a": g.uniform(-1, 1, b, t, NEXT_HV),
                "b": g.uniform(-1, 1, b, t, NEXT_HV),
                "a_log": g.uniform(-1, 0, NEXT_HV, dtype=F32),
                "dt_bias": g.uniform(-0.5, 0.5, NEXT_HV, dtype=F32),
                "state": g.uniform(-0.1, 0.1, b, NEXT_HV, NEXT_DV, NEXT_DK), "z": z,
                "w": g.randn(NEXT_DV, mean=1.0, std=0.02)}
    if kind == "decode_ops":
        t, hd = case["tokens"], NEXT_HIDDEN
        layers = []
        for i in range(case["layers"]):
            d = {"r_prev": g.randn(t, hd), "r_attn": g.randn(t, hd),
                 "gate": g.randn(t, NEXT_TOP_K, NEXT_EXPERT_DIM),
                 "up": g.randn(t, NEXT_TOP_K, NEXT_EXPERT_DIM)}
            if i % 4 == 3:  # full attention: q is the first half of each head's block
                d["q"] = g.randn(t, 16, 512)[:, :, :256]
                d["k"] = g.randn(t, 2, 256)
            else:           # linear attention: z in place in in_proj_qkvz's output
                d["y"] = g.randn(t, NEXT_HV, NEXT_DV)
                d["z"] = g.randn(t, NEXT_HK, 768)[:, :, 512:].unflatten(-1, (2, NEXT_DV))
            layers.append(d)
        return {"h": g.randn(t, hd), "layers": layers, "offsets": g.ints(1, 32769, t),
                "w_in": g.randn(hd, mean=1.0, std=0.02), "w_post": g.randn(hd, mean=1.0, std=0.02),
                "wg": g.randn(NEXT_DV, mean=1.0, std=0.02), "wq": g.randn(256, mean=1.0, std=0.02),
                "wk": g.randn(256, mean=1.0, std=0.02)}
    raise ValueError(kind)


def prepare(case, seed):
    d = _inputs(case, seed)
    d["case"] = case
    kind = case["kind"]
    if kind == "gemma_ops":
        d["embed"] = H.QuantizedEmbedding(*d["table"])
    elif kind == "delta":
        d["wq"], d["wk"] = ops.gdn_qk_norm_weights(NEXT_DK, BF16, d["q"].device)
    elif kind == "decode_ops":
        d["seq"], d["out"] = _decode_plan(case, d)
    return d


def _decode_plan(case, d):
    """The op list a serving loop records once, and its outputs: one tensor per
    kind of output, its first axis the layer."""
    n, full, h = case["layers"], case["layers"] // 4, d["h"]
    new = lambda *shape: torch.empty(shape, dtype=BF16, device=h.device)
    hidden, act = new(n, 4, *h.shape), new(n, *d["layers"][0]["gate"].shape)
    gated = new(n - full, *d["layers"][0]["y"].shape)
    q_out, k_out = new(full, h.shape[0], 16, 256), new(full, h.shape[0], 2, 256)
    seq = H.OpSequence(BF16, h.device)
    for i, l in enumerate(d["layers"]):
        h_a, y_a, h_b, y_b = hidden[i]
        seq.add_rms_norm(h, l["r_prev"], d["w_in"], 1e-6, y_a, h_a)
        if "q" in l:
            seq.qk_norm_rope(l["q"], l["k"], d["wq"], d["wk"], 1e-6, 64, 1e7, q_out[i // 4],
                             k_out[i // 4], offsets=d["offsets"])
        else:
            seq.gated_rms_norm(l["y"], l["z"], d["wg"], 1e-6, gated[i - i // 4])
        seq.add_rms_norm(h_a, l["r_attn"], d["w_post"], 1e-6, y_b, h_b)
        seq.glu(0, l["gate"], l["up"], act[i])
        h = h_b
    seq.upload()
    return seq, (hidden, gated, q_out, k_out, act)


# -------------------------------------------------------------------- calls
def run(state):
    case = state["case"]
    kind, s = case["kind"], state
    if kind == "norm":
        if case["add"]:
            return H.add_rms_norm(s["x"], s["r"], s["w"], 1e-6)
        return H.rms_norm(s["x"], s["w"], 1e-6)
    if kind == "gemma_ops":
        h = s["embed"].forward(s["ids"], out_scale=ops.gemma_embed_scale(case["hidden"]))
        y = H.rms_norm(h, s["w"], 1e-6, plus_one=True)
        q, k = H.qk_norm_rope(s["q"], s["k"], None, None, 1e-6, case["head_dim"], 10000.0)
        act = H.gelu_approximate_mul(s["gate"], s["up"], out_dtype=F32)
        return h, y, q, k, act
    if kind == "qk_rope":
        return H.qk_norm_rope(s["q"], s["k"], s["wq"], s["wk"], 1e-6, case["head_dim"], 1e6,
                              offset=case["offset"])
    if kind == "mlp":
        gate = H.quantized_matmul(s["x"], *s["gate"])
        up = H.quantized_matmul(s["x"], *s["up"])
        return H.quantized_matmul(H.silu_mul(gate, up), *s["down"])
    if kind == "linear":
        return H.quantized_matmul(s["x"], *s["w"])
    if kind == "experts":
        act = H.gather_qmm_swiglu(s["x"], *s["gate"], *s["up"], s["ids"], x_row_div=case["top_k"])
        return H.gather_qmm(act, *s["down"], s["ids"])
    if kind == "delta":
        args = (s["q"], s["k"], s["v"], s["a_log"], s["a"], s["dt_bias"], s["b"], s["state"])
        if case["seq"] == 1:
            return H.gated_delta_gated_norm(*args, s["z"], s["w"], 1e-6, q_norm_w=s["wq"],
                                            k_norm_w=s["wk"])
        return H.gated_delta(*args, q_norm_w=s["wq"], k_norm_w=s["wk"])
    s["seq"].run(case["tokens"])
    return s["out"]


# --------------------------------------------------------------------- work
def _weight_bytes(*shape):
    n = math.prod(shape)
    return n // 2 + 4 * (n // GROUP)


def work(case):
    kind = case["kind"]
    if kind == "norm":
        m, n = case["rows"], case["hidden"]
        return {"bytes": (8 if case["add"] else 4) * m * n + 2 * n, "flops": 4 * m * n}
    if kind == "gemma_ops":
        t, hd, it = case["batch"] * case["seq"], case["hidden"], case["inter"]
        qk = t * (case["heads"] + case["kv_heads"]) * case["head_dim"]
        gather = t * (4 + _weight_bytes(1, hd) + 2 * hd)
        return {"bytes": gather + t * hd * 6 + 2 * hd + 4 * qk + 8 * t * it,
                "flops": t * (6 * hd + 12 * it) + 6 * qk}
    if kind == "qk_rope":
        d = case["head_dim"]
        n = case["batch"] * case["seq"] * (case["heads"] + case["kv_heads"]) * d
        return {"bytes": 4 * n + 4 * d, "flops": 10 * n}
    if kind == "mlp":
        m, hd, it = case["rows"], case["hidden"], case["inter"]
        return {"bytes": 3 * _weight_bytes(hd, it) + 4 * m * hd, "flops": 6 * m * hd * it}
    if kind == "linear":
        m, n, k = case["rows"], case["n"], case["k"]
        return {"bytes": _weight_bytes(n, k) + 2 * m * (n + k), "flops": 2 * m * n * k}
    if kind == "experts":
        t, e, kk = case["tokens"], case["experts"], case["top_k"]
        hd, it = case["hidden"], case["expert_dim"]
        hit = e * (1.0 - (1.0 - kk / e) ** t)  # distinct experts, on average
        return {"bytes": int(3 * hit * _weight_bytes(it, hd)) + 2 * t * hd + 2 * t * kk * hd + 4 * t * kk,
                "flops": 6 * t * kk * hd * it}
    if kind == "delta":
        b, t = case["batch"], case["seq"]
        st = b * NEXT_HV * NEXT_DV * NEXT_DK
        tok = 2 * NEXT_HK * NEXT_DK + 2 * NEXT_HV * NEXT_DV + 2 * NEXT_HV
        z = b * NEXT_HV * NEXT_DV if t == 1 else 0
        return {"bytes": 4 * st + 2 * b * t * tok + 2 * z, "flops": 7 * st * t}
    t, layers = case["tokens"], case["layers"]
    full, lin = layers // 4, layers - layers // 4
    per = (layers * (2 * 4 * NEXT_HIDDEN + 3 * NEXT_TOP_K * NEXT_EXPERT_DIM)
           + full * 2 * 18 * 256 + lin * 3 * NEXT_HV * NEXT_DV)
    return {"bytes": 2 * t * per, "flops": 5 * t * per}


# ---------------------------------------------------------------- tolerance
def tolerance(case):
    """bf16 outputs round at 2^-9; a chain of bf16 steps, or a value that an
    intermediate rounding tips the other way, shows a little more."""
    return {"rel": {"norm": 6e-3, "gemma_ops": 1e-2, "qk_rope": 1e-2, "decode_ops": 1e-2,
                    "mlp": 1e-2, "linear": 6e-3, "experts": 1e-2, "delta": 1.2e-2}[case["kind"]]}


# -------------------------------------------------------------------- exact
def _rms(x, w, eps, add_one=False):
    n = x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)
    return n if w is None else n * (w.to(F64) + (1.0 if add_one else 0.0))


def _held(x):
    """A value as the bf16 tensor between two ops holds it."""
    return x.to(BF16).to(F64)


def _rope(x, dims, base, pos):
    """x [..., D] with positions `pos` broadcast over all but the last axis."""
    half = dims // 2
    inv = base ** (-torch.arange(half, dtype=F64, device=x.device) * 2 / dims)
    ang = pos.to(F64).unsqueeze(-1) * inv
    c, s = ang.cos(), ang.sin()
    a, b = x[..., :half], x[..., half:dims]
    return torch.cat([a * c - b * s, a * s + b * c, x[..., dims:]], -1)


def _dequant(q):
    w, s, b = q
    sh = torch.arange(0, 32, 4, device=w.device, dtype=torch.int32)
    codes = ((w.unsqueeze(-1) >> sh) & 15).flatten(-2).to(F64)
    return codes * s.to(F64).repeat_interleave(GROUP, -1) + b.to(F64).repeat_interleave(GROUP, -1)


def _qmm(x, q):
    w, s, b = q
    out = []
    for i in range(0, w.shape[0], 16384):  # bounds the 64-bit copy of the weight
        out.append(x.to(F64) @ _dequant((w[i:i + 16384], s[i:i + 16384], b[i:i + 16384])).t())
    return torch.cat(out, -1)


def _silu(x):
    return x * torch.sigmoid(x)


def exact(case, seed):
    d, kind = _inputs(case, seed), case["kind"]
    if kind == "norm":
        if case["add"]:
            h = d["x"].to(F64) + d["r"].to(F64)
            return h, _rms(_held(h), d["w"], 1e-6)
        return _rms(d["x"].to(F64), d["w"], 1e-6)
    if kind == "gemma_ops":
        ids, hd = d["ids"].long(), case["hidden"]
        rows = _dequant(tuple(t[ids.reshape(-1)] for t in d["table"]))
        h = _held(rows) * float(torch.tensor(math.sqrt(hd)).to(BF16))
        y = _rms(_held(h), d["w"], 1e-6, add_one=True)
        pos = torch.arange(case["seq"], device=ids.device)
        q, k = (_rope(d[n].to(F64).transpose(1, 2), case["head_dim"], 10000.0, pos) for n in "qk")
        out = [h.view(*ids.shape, hd), y.view(*ids.shape, hd), q, k]
        act = torch.empty(d["gate"].shape, dtype=F64, device=ids.device)
        for i in range(0, act.shape[0], 4096):
            x = d["gate"][i:i + 4096].to(F64)
            t = torch.tanh(math.sqrt(2.0 / math.pi) * (x + 0.044715 * x ** 3))
            act[i:i + 4096] = 0.5 * x * (1.0 + t) * d["up"][i:i + 4096].to(F64)
        return (*out, act)
    if kind == "qk_rope":
        pos = torch.arange(case["seq"], device=d["q"].device) + case["offset"]
        return tuple(_rope(_held(_rms(d[n].to(F64), d["w" + n], 1e-6)).transpose(1, 2),
                           case["head_dim"], 1e6, pos) for n in "qk")
    if kind == "mlp":
        gate, up = (_held(_qmm(d["x"], d[n])) for n in ("gate", "up"))
        return _qmm(_held(_held(_silu(gate)) * up), d["down"])
    if kind == "linear":
        return _qmm(d["x"], d["w"])
    if kind == "experts":
        return _exact_experts(case, d)
    if kind == "delta":
        return _exact_delta(case, d)
    return _exact_decode_ops(d)


def _exact_experts(case, d):
    ids, kk = d["ids"].reshape(-1), case["top_k"]
    out = torch.empty((ids.numel(), case["hidden"]), dtype=F64, device=ids.device)
    order = torch.argsort(ids, stable=True)
    count = torch.bincount(ids.long(), minlength=case["experts"]).tolist()
    for e, pairs in enumerate(order.split(count)):
        if pairs.numel():
            x = d["x"][pairs // kk]
            gate, up = (_held(_qmm(x, tuple(t[e] for t in d[n]))) for n in ("gate", "up"))
            act = _held(_held(_silu(gate)) * up)
            out[pairs] = _qmm(act, tuple(t[e] for t in d["down"]))
    return out


def _exact_delta(case, d):
    rep = NEXT_HV // NEXT_HK
    s = float(NEXT_DK) ** -0.5
    q = _held(_rms(d["q"].to(F64), None, 1e-6) * s * s).repeat_interleave(rep, 2)
    k = _held(_rms(d["k"].to(F64), None, 1e-6) * s).repeat_interleave(rep, 2)
    v, st = d["v"].to(F64), d["state"].to(F64)
    step = torch.nn.functional.softplus(d["a"].to(F64) + d["dt_bias"].to(F64))
    g = torch.exp(-torch.exp(d["a_log"].to(F64)) * step)
    beta = torch.sigmoid(d["b"].to(F64))
    ys = []
    for t in range(case["seq"]):
        kt, qt = k[:, t].unsqueeze(-2), q[:, t].unsqueeze(-2)
        st = st * g[:, t, :, None, None]
        delta = (v[:, t] - (st * kt).sum(-1)) * beta[:, t, :, None]
        st = st + kt * delta.unsqueeze(-1)
        ys.append((st * qt).sum(-1))
    y = torch.stack(ys, 1)
    if case["seq"] == 1:
        z = d["z"].to(F64).reshape(y.shape)
        y = _held(_silu(z)) * _held(_rms(_held(y), d["w"], 1e-6))
    return y, st


def _exact_decode_ops(d):
    h, pos = d["h"].to(F64), d["offsets"].unsqueeze(-1)
    hidden, gated, q_out, k_out, acts = [], [], [], [], []
    for l in d["layers"]:
        h_a = h + l["r_prev"].to(F64)
        y_a = _rms(_held(h_a), d["w_in"], 1e-6)
        if "q" in l:
            for n, out in (("q", q_out), ("k", k_out)):
                out.append(_rope(_held(_rms(l[n].to(F64), d["w" + n], 1e-6)), 64, 1e7, pos))
        else:
            z = l["z"].to(F64).reshape(l["y"].shape)
            gated.append(_held(_silu(z)) * _held(_rms(l["y"].to(F64), d["wg"], 1e-6)))
        h_b = _held(h_a) + l["r_attn"].to(F64)
        hidden.append(torch.stack([h_a, y_a, h_b, _rms(_held(h_b), d["w_post"], 1e-6)]))
        acts.append(_held(_silu(l["gate"].to(F64))) * l["up"].to(F64))
        h = _held(h_b)
    return tuple(torch.stack(x) for x in (hidden, gated, q_out, k_out, acts))
