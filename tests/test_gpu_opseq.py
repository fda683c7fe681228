"""The decode op sequence in one launch (hgk_op_list_upload / hgk_op_list_run,
Python OpSequence) against the separate calls it replaces, bit for bit, and
the residual chain against the oracle.

The sequence is the Qwen3-Next decode layer's per-layer ops in the order of
the reference loop (qwen3_next.rs:1508-1547): input_layernorm as residual add
+ RMSNorm, the gated RMSNorm (linear-attention layers, z read in place from
in_proj_qkvz) or q/k RMSNorm + partial RoPE (every fourth layer, q the first
256 of each 512-wide block, per-sequence offsets), post_attention_layernorm
(add + RMSNorm), the routed experts' and the shared expert's SwiGLU. The
projections' outputs are random stand-ins."""
from __future__ import annotations

import time

import numpy as np
import pytest
import torch

import higgs_amd as H
import oracle as O
from higgs_amd._lib import ACT_SILU
from bits import exact_frac, ulp_dist
from gpu_util import to_host

pytestmark = pytest.mark.gpu


def _layers(dev, dt, T, n_layers, seed):
    """Buffers of an n-layer decode step: the residual chain and every op's
    inputs and outputs (Qwen3-Next-80B-A3B shapes)."""
    g = torch.Generator(device=dev)
    g.manual_seed(seed)

    def rnd(*shape, mean=0.0, std=1.0):
        t = torch.empty(shape, dtype=torch.float32, device=dev)
        t.normal_(mean, std, generator=g)
        return t.to(dt)

    Hd, Hv, Dv, Hq, Hk, D, E, I = 2048, 32, 128, 16, 2, 256, 10, 512
    L = dict(h0=rnd(T, Hd), w_in=rnd(Hd, mean=1.0, std=0.02), w_post=rnd(Hd, mean=1.0, std=0.02),
             w_g=rnd(Dv, mean=1.0, std=0.02), wq=rnd(D, mean=1.0, std=0.02),
             wk=rnd(D, mean=1.0, std=0.02),
             offsets=torch.randint(1, 32769, (T,), dtype=torch.int32, device=dev, generator=g),
             layers=[])
    for layer in range(n_layers):
        d = dict(r_prev=rnd(T, Hd), r_attn=rnd(T, Hd), gate=rnd(T, E, I), up=rnd(T, E, I),
                 sgate=rnd(T, I), sup=rnd(T, I))
        if layer % 4 == 3:
            d["q"] = rnd(T, Hq, 2 * D)[:, :, :D]
            d["k"] = rnd(T, Hk, D)
        else:
            d["y"] = rnd(T, Hv, Dv)
            d["z"] = rnd(T, Hv // 2, 768)[:, :, 512:].unflatten(-1, (2, Dv))
        L["layers"].append(d)
    return L


def _outputs(L, dev, dt, T):
    Hd, Hv, Dv, Hq, Hk, D, E, I = 2048, 32, 128, 16, 2, 256, 10, 512
    e = lambda *s: torch.full(s, float("nan"), dtype=dt, device=dev)
    outs = []
    for d in L["layers"]:
        o = dict(h_a=e(T, Hd), y_a=e(T, Hd), h_b=e(T, Hd), y_b=e(T, Hd), act=e(T, E, I),
                 sact=e(T, I))
        if "q" in d:
            o["qo"], o["ko"] = e(T, Hq, D), e(T, Hk, D)
        else:
            o["go"] = e(T, Hv, Dv)
        outs.append(o)
    return outs


def _record(L, outs, dt):
    seq = H.OpSequence(dt, L["h0"].device)
    h = L["h0"]
    for d, o in zip(L["layers"], outs):
        seq.add_rms_norm(h, d["r_prev"], L["w_in"], 1e-6, o["y_a"], o["h_a"])
        if "q" in d:
            seq.qk_norm_rope(d["q"], d["k"], L["wq"], L["wk"], 1e-6, 64, 1e7, o["qo"], o["ko"],
                             offsets=L["offsets"])
        else:
            seq.gated_rms_norm(d["y"], d["z"], L["w_g"], 1e-6, o["go"])
        seq.add_rms_norm(o["h_a"], d["r_attn"], L["w_post"], 1e-6, o["y_b"], o["h_b"])
        seq.glu(ACT_SILU, d["gate"], d["up"], o["act"])
        seq.glu(ACT_SILU, d["sgate"], d["sup"], o["sact"])
        h = o["h_b"]
    return seq


def _separate(L, outs, T):
    """The same ops as the separate calls, into `outs`."""
    h = L["h0"]
    for d, o in zip(L["layers"], outs):
        H.add_rms_norm(h[:T], d["r_prev"][:T], L["w_in"], 1e-6, h_out=o["h_a"][:T], out=o["y_a"][:T])
        if "q" in d:
            qo, ko = H.qk_norm_rope(d["q"][:T].unsqueeze(1), d["k"][:T].unsqueeze(1), L["wq"],
                                    L["wk"], 1e-6, 64, 1e7, 1.0, 0, offsets=L["offsets"][:T])
            o["qo"][:T] = qo[:, :, 0, :]
            o["ko"][:T] = ko[:, :, 0, :]
        else:
            H.gated_rms_norm(d["y"][:T], d["z"][:T], L["w_g"], 1e-6, out=o["go"][:T])
        H.add_rms_norm(o["h_a"][:T], d["r_attn"][:T], L["w_post"], 1e-6, h_out=o["h_b"][:T],
                       out=o["y_b"][:T])
        H.swiglu(d["gate"][:T], d["up"][:T], out=o["act"][:T])
        H.swiglu(d["sgate"][:T], d["sup"][:T], out=o["sact"][:T])
        h = o["h_b"]


def _same_bits(a, b, what):
    a16, b16 = a.view(torch.int16), b.view(torch.int16)
    bad = (a16 != b16)
    assert not bool(bad.any()), f"{what}: {int(bad.sum())} elements differ, first at {bad.nonzero()[0].tolist()}"


@pytest.mark.parametrize("dt,T,n_layers", [(torch.bfloat16, 64, 8), (torch.float16, 9, 4)])
def test_op_sequence_matches_the_separate_calls_bitwise(dev, dt, T, n_layers):
    """Every output of an n-layer op sequence (the full 64-sequence batch in
    bf16; 9 sequences in f16) equals the separate calls' bit for bit."""
    L = _layers(dev, dt, T, n_layers, 71)
    got, ref = _outputs(L, dev, dt, T), _outputs(L, dev, dt, T)
    seq = _record(L, got, dt)
    print(f"[opseq] {len(seq)} ops, {T} tokens, {dt}", flush=True)
    seq.run(T)
    _separate(L, ref, T)
    torch.cuda.synchronize()
    for layer, (g, r) in enumerate(zip(got, ref)):
        for k in g:
            _same_bits(g[k], r[k], f"layer {layer} {k}")


@pytest.mark.parametrize("T,n_layers", [(96, 4), (97, 4), (129, 1), (223, 4), (224, 4), (600, 2)])
def test_op_sequence_of_more_tokens(dev, T, n_layers):
    """Every number of workgroups per token (8, 4, 3 and 1) gives the separate
    calls' bits, also for the first ops of a list alone."""
    dt = torch.bfloat16
    L = _layers(dev, dt, T, n_layers, 74)
    got, ref = _outputs(L, dev, dt, T), _outputs(L, dev, dt, T)
    seq = _record(L, got, dt)
    seq.run(T)
    _separate(L, ref, T)
    for layer, (g, r) in enumerate(zip(got, ref)):
        for k in g:
            _same_bits(g[k], r[k], f"layer {layer} {k}")
    from higgs_amd import _lib
    again = _outputs(L, dev, dt, T)
    seq = _record(L, again, dt).upload()
    _lib.check(_lib.lib().hgk_op_list_run(_lib.BF16, H.ops._ptr(seq._list), 3, T,
                                          H.ops._stream(torch.device(dev))))
    written = ("h_a", "y_a", "h_b", "y_b", "go")
    for k, v in again[0].items():
        if k in written:
            _same_bits(v, ref[0][k], f"first ops {k}")
        else:
            assert bool(torch.isnan(v.float()).all()), f"{k}: written by an op past the first 3"


def test_many_tokens_cost_one_workgroup_each(dev):
    """A one-op list over more tokens than the chip holds workgroups: the least
    of ten runs takes at most 7 times the separate call's (measured: 4.4 with a
    workgroup per token, 11 with one per token and chain)."""
    T, n, dt = 8192, 2048, torch.bfloat16
    x, r, y = (torch.zeros(T, n, dtype=dt, device=dev) for _ in range(3))
    seq = H.OpSequence(dt, torch.device(dev))
    seq.glu(ACT_SILU, x, r, y)
    seq.upload()

    def least(f):
        times = []
        for _ in range(12):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(10):
                f()
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b) * 100)
        return min(times[2:])

    one, call = least(lambda: seq.run(T)), least(lambda: H.swiglu(x, r, out=y))
    print(f"[opseq] {T} tokens: list {one:.1f} us, call {call:.1f} us", flush=True)
    assert one <= 7 * call


def test_op_sequence_residual_chain_against_the_oracle(dev):
    """Two layers' residual chain (h = x + r, y = rms_norm(h)) of the op
    sequence against the oracle's add and RMSNorm, composed on the CPU."""
    T, dt = 64, torch.bfloat16
    L = _layers(dev, dt, T, 2, 72)
    got = _outputs(L, dev, dt, T)
    _record(L, got, dt).run(T)
    torch.cuda.synchronize()
    h = to_host(L["h0"])
    for layer, (d, o) in enumerate(zip(L["layers"], got)):
        for r, w, hk, yk in ((d["r_prev"], L["w_in"], "h_a", "y_a"),
                             (d["r_attn"], L["w_post"], "h_b", "y_b")):
            h = O.add(h, to_host(r), O.BF16)
            y = O.rms_norm(h, O.BF16, to_host(w), O.BF16, 1e-6)
            assert np.array_equal(to_host(o[hk]), h), f"layer {layer} {hk}"
            gy = to_host(o[yk])
            assert ulp_dist(gy, y, O.BF16).max() <= 1 and exact_frac(gy, y, O.BF16) >= 0.9999


def test_op_sequence_fewer_tokens_and_a_foreign_list(dev):
    """A run over the first 5 tokens writes only their rows; a list the upload
    did not write (zeros) launches and touches nothing."""
    T, dt = 16, torch.bfloat16
    L = _layers(dev, dt, T, 4, 73)
    got, ref = _outputs(L, dev, dt, T), _outputs(L, dev, dt, T)
    seq = _record(L, got, dt)
    seq.run(5)
    _separate(L, ref, 5)
    torch.cuda.synchronize()
    for layer, (g, r) in enumerate(zip(got, ref)):
        for k in g:
            _same_bits(g[k][:5], r[k][:5], f"layer {layer} {k}")
            assert bool(torch.isnan(g[k][5:].float()).all()), f"layer {layer} {k}: rows past 5 written"
    from higgs_amd import _lib
    blank = torch.zeros(int(_lib.lib().hgk_op_list_bytes(len(seq))) + 16, dtype=torch.uint8,
                        device=dev)
    before = {k: v.clone() for k, v in got[0].items()}
    _lib.check(_lib.lib().hgk_op_list_run(_lib.BF16, H.ops._ptr(blank), len(seq), T,
                                          H.ops._stream(blank.device)))
    # the f16 kernel given the bf16 list is also refused by the list's header
    _lib.check(_lib.lib().hgk_op_list_run(_lib.F16, H.ops._ptr(seq._list), len(seq), T,
                                          H.ops._stream(blank.device)))
    torch.cuda.synchronize()
    for k, v in got[0].items():
        _same_bits(v, before[k], f"foreign list {k}")


@pytest.mark.parametrize("seed", range(10))
def test_dependent_ops_over_shared_buffers(dev, seed):
    """Random lists of all five kinds of op over a small pool of buffers, so that
    ops read, overwrite and re-read each other's results (in place, through
    column slices and, in every other list, with views of two token strides),
    against the separate calls bit for bit. Chains of dependent ops run in order
    whatever else runs beside."""
    T, n, dt = 5, 256, torch.bfloat16
    r = np.random.default_rng(100 + seed)
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    w = torch.randn(n, generator=g, device=dev).to(dt)
    wh = torch.randn(64, generator=g, device=dev).to(dt)
    offsets = torch.randint(0, 99, (T,), dtype=torch.int32, device=dev, generator=g)
    base = [torch.randn(3 * T, 2 * n, generator=g, device=dev).to(dt) for _ in range(5)]
    start = [b.clone() for b in base]

    def view(pool, i, half, rows):  # [T, n]: one half of buffer i's rows 0, 1, .. or T, T + 2, ..
        return (pool[i][T::2] if rows else pool[i])[:T, half * n:(half + 1) * n]

    def heads(v):  # [T, 4, 64]
        return v.unflatten(-1, (4, 64))

    # (the views of one buffer have one stride: where two meet, it is for different tokens, whose
    # order no list defines)
    two = seed % 2 == 1
    at = lambda i: int(two and i >= 3)
    pick = lambda: (lambda i: (i, int(r.integers(2)), at(i)))(int(r.integers(5)))
    ops, carry = [], None
    for _ in range(40):
        kind = r.choice(["add", "add", "add", "rms", "glu", "gated", "rope"])
        a, b, c, d = pick(), pick(), pick(), pick()
        if kind == "add" and carry is not None and r.random() < 0.7:
            a = carry  # the residual stream, sometimes updated in place
            d = a if r.random() < 0.3 else d
        if kind == "rope":
            if len({a, b, c, d}) < 4:
                continue
        elif c == d or (kind in ("add", "gated") and c in (a, b)):
            continue
        if kind == "add" and d == b:
            continue
        ops.append((kind, a, b, c, d))
        carry = d if kind == "add" else carry
    seq = H.OpSequence(dt, torch.device(dev))
    for kind, a, b, c, d in ops:
        x, y, out, h = (view(base, *p) for p in (a, b, c, d))
        if kind == "add":
            seq.add_rms_norm(x, y, w, 1e-6, out, h)
        elif kind == "rms":
            seq.rms_norm(x, w, 1e-6, out)
        elif kind == "gated":
            seq.gated_rms_norm(heads(x), heads(y), wh, 1e-6, heads(out))
        elif kind == "rope":
            # (two tables in turn: a chain's ops reuse one only where it is theirs)
            seq.qk_norm_rope(heads(x), heads(y), wh, wh, 1e-6, 32, 1e4 if a[1] else 1e6, heads(out),
                             heads(h), offsets=offsets)
        else:
            seq.glu(ACT_SILU, x, y, out)
    ref = [b.clone() for b in start]
    for kind, a, b, c, d in ops:
        x, y, out, h = (view(ref, *p) for p in (a, b, c, d))
        x, y = x.contiguous(), y.contiguous()
        if kind == "add":
            hh, yy = H.add_rms_norm(x, y, w, 1e-6)
            h.copy_(hh)
            out.copy_(yy)
        elif kind == "rms":
            out.copy_(H.rms_norm(x, w, 1e-6))
        elif kind == "gated":
            out.copy_(H.gated_rms_norm(heads(x), heads(y), wh, 1e-6).flatten(1))
        elif kind == "rope":
            q, k = H.qk_norm_rope(heads(x).unsqueeze(1), heads(y).unsqueeze(1), wh, wh, 1e-6, 32,
                                  1e4 if a[1] else 1e6, 1.0, 0, offsets=offsets)
            out.copy_(q[:, :, 0].flatten(1))
            h.copy_(k[:, :, 0].flatten(1))
        else:
            out.copy_(H.swiglu(x, y))
    for _ in range(2):  # the same list again, from the same start
        for b, s in zip(base, start):
            b.copy_(s)
        seq.run(T)
        for i, (got, want) in enumerate(zip(base, ref)):
            assert np.array_equal(to_host(got), to_host(want)), f"buffer {i}"


def test_a_long_list_uploads_in_proportion(dev):
    """Sorting a list into chains takes time in proportion to its length: 4096
    ops (the most a list holds) upload in at most 24 times the time of 512, the
    least of three times each (8 times the ops; pairs of ops: 64)."""
    T, n, dt = 2, 64, torch.bfloat16
    x = torch.zeros(T, n, dtype=dt, device=dev)
    pool = torch.zeros(3 * 4096, T, n, dtype=dt, device=dev)
    w = torch.ones(n, dtype=dt, device=dev)
    least = {}
    for n_ops in (512, 4096):
        seq, h = H.OpSequence(dt, torch.device(dev)), x
        for i in range(n_ops):
            seq.add_rms_norm(h, pool[3 * i], w, 1e-6, pool[3 * i + 1], pool[3 * i + 2])
            h = pool[3 * i + 2]
        times = []
        for _ in range(3):
            t0 = time.perf_counter()
            seq.upload()
            times.append(time.perf_counter() - t0)
        least[n_ops] = min(times)
    print(f"[opseq] upload: 512 ops {least[512] * 1e3:.2f} ms, 4096 {least[4096] * 1e3:.2f} ms", flush=True)
    assert least[4096] <= 24 * least[512]


@pytest.mark.parametrize("n", [64, 2048])
def test_a_norm_written_over_its_residual(dev, n):
    """y on the address of h: y is stored last, so the next op reads y, whether
    or not it could have taken h from registers."""
    T, dt = 5, torch.bfloat16
    g = torch.Generator(device=dev)
    g.manual_seed(n)
    x, r1, r2, r3 = (torch.randn(T, n, generator=g, device=dev).to(dt) for _ in range(4))
    w = torch.randn(n, generator=g, device=dev).to(dt)
    a, h2, y2, h3, y3 = (torch.zeros(T, n, dtype=dt, device=dev) for _ in range(5))
    seq = H.OpSequence(dt, torch.device(dev))
    seq.add_rms_norm(x, r1, w, 1e-6, a, a)
    seq.add_rms_norm(a, r2, w, 1e-6, y2, h2)
    seq.add_rms_norm(h2, r3, w, 1e-6, y3, h3)
    seq.run(T)
    _, y1 = H.add_rms_norm(x, r1, w, 1e-6)
    want2 = H.add_rms_norm(y1, r2, w, 1e-6)
    want3 = H.add_rms_norm(want2[0], r3, w, 1e-6)
    for what, got, want in (("y1", a, y1), ("h2", h2, want2[0]), ("y2", y2, want2[1]),
                            ("h3", h3, want3[0]), ("y3", y3, want3[1])):
        _same_bits(got, want, what)


def test_buffers_that_meet_at_a_later_token(dev):
    """Two ops whose outputs share bytes only from some token on (views with
    different token strides): up to there they run side by side, over more
    tokens the list runs in order. Token t of the first op is rows[2 t], of the
    second rows[8 + t], so token 8's first output is token 8's second."""
    n, dt = 64, torch.bfloat16
    g = torch.Generator(device=dev)
    g.manual_seed(7)
    x, z = (torch.randn(16, n, generator=g, device=dev).to(dt) for _ in range(2))
    for T in (8, 12):
        rows = torch.zeros(40, n, dtype=dt, device=dev)
        seq = H.OpSequence(dt, torch.device(dev))
        seq.glu(ACT_SILU, x, z, rows[0:32:2])
        seq.glu(ACT_SILU, z, x, rows[8:24])
        seq.run(T)
        got, a, b = to_host(rows), to_host(H.swiglu(x, z)), to_host(H.swiglu(z, x))
        # rows one op writes alone, and the row both write for the same token
        for t in range(T):
            if not (2 * t - 8 in range(T)):
                assert np.array_equal(got[2 * t], a[t])
            if (8 + t) % 2 or (8 + t) // 2 >= T or (8 + t) // 2 == t:
                assert np.array_equal(got[8 + t], b[t])
