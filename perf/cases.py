"""The calls this framework's speed is judged by: what a user has it do, through its public entry points.

Each case is a dict of sizes and options, its "kind" the entry point:

  layer      race_causal_attention, bf16 [B,H,T,D], forward and backward (training a RACE layer)
  attend     nanochat.race_attend on [B,T,H,D] activations, forward and backward, as the attention
             layers of nanochat.py and hybrid.py call it: precision "bf16" (the fused kernels, grouped
             query heads) or "fp32" (the default of GPTConfig)
  module     RaceCausalCuda on fp32 inputs, forward and backward: the reference's fp32 layer
  noncausal  noncausal.BatchedACE with its learnable temperature, fp32, forward and backward
  linear     causal_linear_attention, fp32, forward and backward
  prefill    RaceDecodeState.prefill: a prompt's outputs and the bucket state that decoding goes on from
  decode     RaceDecodeState.step: one token of every sequence on the carried state
"""
import math

import torch

from race_attention_amd import RaceDecodeState, build_planes_protos, race_causal_attention
from race_attention_amd.linear_attention import causal_linear_attention
from race_attention_amd.nanochat import race_attend
from race_attention_amd.noncausal import BatchedACE
from race_attention_amd.race_causal_cuda import RaceCausalCuda

DEV = "cuda"
EPS = 1e-6
F64 = torch.float64


def listed():
    return [
        # The benchmark's headline: one long-context training step of a bf16 layer (a million tokens).
        dict(name="layer_1m", kind="layer", B=1, H=4, T=1 << 20, D=64, L=8, K=4, std=0.125),
        # The same layer over a batch of ordinary sequences with 256 buckets (two bucket tiles).
        dict(name="layer_256_buckets", kind="layer", B=4, H=16, T=65536, D=64, L=16, K=4, std=1.0),
        # Training attention of the 1B-shaped hybrid model: grouped query heads, [B,T,H,D] activations.
        dict(name="attend_gqa", kind="attend", precision="bf16", B=8, Hq=32, Hkv=8, T=8192, D=64, L=8, K=4),
        # The nanochat default layer (6 heads of 128, 3 tables of 3 bits), 2047 tokens of a 2048-token
        # window, with the fused bf16 kernels and with its default fp32 computation.
        dict(name="attend_nanochat_bf16", kind="attend", precision="bf16", B=16, Hq=6, Hkv=6, T=2047, D=128,
             L=3, K=3),
        dict(name="attend_nanochat_fp32", kind="attend", precision="fp32", B=16, Hq=6, Hkv=6, T=2047, D=128,
             L=3, K=3),
        # The reference's fp32 layer at its own benchmark sizes, and on one long sequence of odd length.
        dict(name="module_fp32", kind="module", B=2, H=8, T=2048, D=64, L=8, K=4),
        dict(name="module_fp32_long", kind="module", B=1, H=4, T=200003, D=64, L=8, K=4),
        # Non-causal attention at the reference benchmark's defaults, a million tokens.
        dict(name="noncausal_1m", kind="noncausal", B=1, H=4, T=1 << 20, D=128, L=3, K=3),
        # The comparison kernel of the reference's benchmarks on a million tokens.
        dict(name="linear_1m", kind="linear", B=1, H=4, T=1 << 20, D=64),
        # Serving: prompts of 512 tokens for 256 sequences, then a token for each of them, and a token
        # for the 8 sequences of a small server (the smallest call: launch and host time count).
        dict(name="prefill_256", kind="prefill", B=256, Hq=32, Hkv=8, T=512, D=64, L=8, K=4),
        dict(name="decode_256", kind="decode", B=256, Hq=32, Hkv=8, D=64, L=8, K=4, dtype="bf16"),
        dict(name="decode_8", kind="decode", B=8, Hq=32, Hkv=8, D=64, L=8, K=4, dtype="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _batch(rng, rows, most=8):
    """Sequences that fit `rows` rows of activations, at most `most`."""
    return max(1, min(_log(rng, 1, most), rows))


def draw(rng):
    """Another call of the same ranges: sizes spread over their logarithm, mostly not round. Rows
    (tokens x heads) are bounded so that a drawn case costs no more than the largest listed ones."""
    kind = rng.choice(["layer", "attend", "attend", "module", "noncausal", "linear", "prefill", "decode"])
    D = rng.choice([64, 64, 128])
    L, K = rng.choice([(8, 4), (8, 4), (3, 3), (4, 4), (4, 3), (2, 2)])
    if kind == "layer":
        H, T = rng.choice([4, 6, 8, 16]), _log(rng, 1000, 1 << 18)
        return dict(kind=kind, B=_batch(rng, (1 << 20) // (H * T)), H=H, T=T, D=D, L=L, K=K, std=rng.choice([0.125, 1.0]))
    if kind == "attend":
        Hq, Hkv = rng.choice([(32, 8), (16, 4), (8, 8), (6, 6), (6, 2), (8, 1)])
        T = _log(rng, 500, 16384)
        return dict(kind=kind, precision=rng.choice(["bf16", "bf16", "fp32"]),
                    B=_batch(rng, (1 << 20) // (Hq * T), 16), Hq=Hq, Hkv=Hkv, T=T, D=D, L=L, K=K)
    if kind == "module":
        H, T = rng.choice([4, 8, 12]), _log(rng, 500, 65536)
        return dict(kind=kind, B=_batch(rng, (1 << 19) // (H * T), 4), H=H, T=T, D=D, L=L, K=K)
    if kind == "noncausal":
        H, T = rng.choice([4, 8]), _log(rng, 1000, 1 << 18)
        L, K = rng.choice([(3, 3), (2, 2), (4, 3), (4, 4)])
        return dict(kind=kind, B=_batch(rng, (1 << 21) // (H * T), 4), H=H, T=T, D=D, L=L, K=K)
    if kind == "linear":
        H, T, D = rng.choice([4, 8]), _log(rng, 500, 1 << 18), rng.choice([32, 64, 64])
        return dict(kind=kind, B=_batch(rng, (1 << 21) // (H * T), 4), H=H, T=T, D=D)
    Hq, Hkv = rng.choice([(32, 8), (32, 8), (16, 4), (8, 8)])
    if kind == "prefill":
        T = _log(rng, 60, 8192)
        return dict(kind=kind, B=_batch(rng, (1 << 21) // (Hq * T), 256), Hq=Hq, Hkv=Hkv, T=T, D=D, L=L, K=K)
    return dict(kind="decode", B=_log(rng, 1, 600), Hq=Hq, Hkv=Hkv, D=D, L=L, K=K, dtype=rng.choice(["bf16", "bf16", "fp32"]))


# ---------------------------------------------------------------- the calls

def _heads(c):
    return (c["H"], c["H"]) if "H" in c else (c["Hq"], c["Hkv"])


def prepare(case, seed):
    c = dict(case)
    g = torch.Generator(device=DEV).manual_seed(seed)

    def normal(*shape, std=1.0, dtype=torch.float32):
        return (torch.randn(*shape, generator=g, device=DEV) * std).to(dtype)

    kind, B, D = c["kind"], c["B"], c["D"]
    Hq, Hkv = _heads(c)
    T = c.get("T")
    if kind == "linear":  # positive features, as the reference's comparison draws them
        q, k = (torch.rand(B, Hq, T, D, generator=g, device=DEV).requires_grad_() for _ in range(2))
        return dict(c, q=q, k=k, v=normal(B, Hq, T, D).requires_grad_(), go=normal(B, Hq, T, D))
    if kind == "noncausal":
        state = torch.random.get_rng_state()
        torch.manual_seed(seed)  # the module draws its planes from the global generator
        ace = BatchedACE(D, c["K"], c["L"], 1, device="cpu", share_planes=True).to(DEV)
        torch.random.set_rng_state(state)
        k, v, q = (normal(1, B, T, Hq, D).requires_grad_() for _ in range(3))
        return dict(c, ace=ace, k=k, v=v, q=q, go=normal(1, B, T, Hq, D))
    planes, protos = build_planes_protos(D, c["K"], c["L"], 1, device=DEV, seed=seed)
    if kind == "layer":
        q, k, v = (normal(B, Hq, T, D, std=c["std"], dtype=torch.bfloat16).requires_grad_() for _ in range(3))
        return dict(c, planes=planes, q=q, k=k, v=v, go=normal(B, Hq, T, D, dtype=torch.bfloat16))
    if kind == "attend":  # bf16 activations of a model; q, k normalised to 1.2 rms as nanochat's are
        q, k, v = (normal(B, T, h, D, std=s, dtype=torch.bfloat16).requires_grad_()
                   for h, s in ((Hq, 1.2), (Hkv, 1.2), (Hkv, 1.0)))
        return dict(c, planes=planes, protos=protos, q=q, k=k, v=v, go=normal(B, T, Hq * D, dtype=torch.bfloat16))
    if kind == "module":
        mod = RaceCausalCuda(D, c["K"], c["L"], 1, device=DEV, eps=EPS, seed=seed)
        q, k, v = (normal(B, Hq, T, D).requires_grad_() for _ in range(3))
        return dict(c, mod=mod, q=q, k=k, v=v, go=normal(B, Hq, T, D))
    st = RaceDecodeState(B, Hq, Hkv, D, c["L"], c["K"], planes, eps=EPS, device=DEV)
    if kind == "prefill":
        q, k, v = (normal(B, h, T, D, dtype=torch.bfloat16) for h in (Hq, Hkv, Hkv))
        return dict(c, st=st, planes=planes, q=q, k=k, v=v)
    # the state of 512 tokens: bucket masses around 512 / 2^K, value sums of random sign
    dt = torch.bfloat16 if c["dtype"] == "bf16" else torch.float32
    mass = 512.0 / (1 << c["K"])
    st.A.copy_(mass * torch.exp(normal(*st.A.shape, std=0.3)))
    st.Bs.copy_(normal(*st.Bs.shape, std=math.sqrt(mass / 8)))
    st.tokens = 512
    return dict(c, st=st, planes=planes, q=normal(B, Hq, D, dtype=dt), k=normal(B, Hkv, D, dtype=dt), v=normal(B, Hkv, D, dtype=dt))


def run(s):
    kind = s["kind"]
    if kind == "decode":
        return s["st"].step(s["q"], s["k"], s["v"]), s["st"].A, s["st"].Bs
    if kind == "prefill":
        s["st"].reset()
        out = s["st"].prefill(s["q"], s["k"], s["v"])
        return out, s["st"].A, s["st"].Bs
    q, k, v = s["q"], s["k"], s["v"]
    q.grad = k.grad = v.grad = None
    if kind == "layer":
        out = race_causal_attention(q, k, v, s["planes"], s["L"], s["K"], eps=EPS)
    elif kind == "attend":
        y = race_attend(q, k, v, s["planes"], s["L"], s["K"], EPS, precision=s["precision"], protos_T=s["protos"])
        out = y.reshape(s["B"], s["T"], -1)
    elif kind == "module":
        out = s["mod"](q, k, v)
    elif kind == "linear":
        out = causal_linear_attention(q, k, v)
    else:
        s["ace"].logit_temp.grad = None
        out = s["ace"](k, v, q, EPS)
    out.backward(s["go"])
    if kind == "noncausal":
        return out.detach(), q.grad, k.grad, v.grad, s["ace"].logit_temp.grad
    return out.detach(), q.grad, k.grad, v.grad


# ---------------------------------------------------------------- what a pass cannot do without

def work(case):
    c = case
    Hq, Hkv = _heads(c)
    D, S, LK = c["D"], 0, 0
    if c["kind"] != "linear":
        S, LK = c["L"] << c["K"], c["L"] * c["K"]
    R = 1 << c.get("K", 0)
    elt = 4 if c["kind"] in ("module", "noncausal", "linear") or c.get("dtype") == "fp32" else 2
    if c["kind"] == "decode":  # the state read and written, one row of each tensor
        n = c["B"] * Hkv
        return {"bytes": 2 * 4 * n * S * (D + 1) + elt * c["B"] * (2 * Hq + 2 * Hkv) * D,
                "flops": n * 4 * S * D + c["B"] * Hq * 2 * S * D + c["B"] * (Hq + Hkv) * 2 * D * LK}
    q_rows, kv_rows = c["B"] * c["T"] * Hq, c["B"] * c["T"] * Hkv
    hash_f = 2 * D * LK + 2 * LK * R + 4 * S
    if c["kind"] == "prefill":
        return {"bytes": elt * D * (2 * q_rows + 2 * kv_rows) + 4 * c["B"] * Hkv * S * (D + 1),
                "flops": q_rows * (2 * S * D + hash_f) + kv_rows * (2 * S * D + hash_f)}
    # q, go, out, dq and k, v, dk, dv once each
    nbytes = elt * D * 4 * (q_rows + kv_rows)
    if c["kind"] == "linear":
        return {"bytes": nbytes, "flops": 12 * D * D * q_rows}
    # forward: two contractions with the state; backward: five (per query head, the value side per kv head)
    return {"bytes": nbytes, "flops": q_rows * (8 * S * D + 3 * hash_f) + kv_rows * (6 * S * D + 3 * hash_f)}


def tolerance(case):
    """About four times the error against 64 bits that the path shows at these sizes."""
    if case["kind"] == "decode":  # bf16: the output's own rounding
        return {"rel": 1e-5} if case["dtype"] == "fp32" else {"rel": 6e-3, "max": 0.03}
    if case["kind"] in ("module", "noncausal", "linear"):
        return {"rel": 1e-5}
    if case["kind"] == "attend" and case["precision"] == "fp32":  # bf16 inputs and outputs around fp32 sums
        return {"rel": 4e-3, "max": 0.03}
    if case["kind"] == "prefill":
        return {"rel": 8e-3, "max": 0.2}
    # bf16 operands in every contraction: gradients 5e-3 to 1.1e-2 off, most at a sequence's first tokens,
    # where the two terms of dk cancel
    return {"rel": 2.5e-2, "max": 0.8}


# ---------------------------------------------------------------- the same results in 64 bits

def _hash64(x, planes, L, K, scale):
    """Bucket probabilities [N,T,L*2^K] of rows x [N,T,D]: the softmax over the corners of each table."""
    bits = torch.arange(1 << K, device=x.device)[:, None] >> torch.arange(K - 1, -1, -1, device=x.device)
    corners = ((bits & 1) * 2 - 1).to(F64)
    u = torch.tanh(x @ planes) / scale
    logits = u.view(*x.shape[:2], L, K) @ corners.T
    return torch.softmax(logits, -1).flatten(2)


def _scan64(pK, pQ, V, go, eps, normalise=True, c=64):
    """Causal readout sum_s W_t[s] sum_{tau<=t} pK_tau[s] v_tau, W = pQ / (sum pK + eps) (or pQ alone), of
    [N,T,S] and [N,T,D], in chunks of c tokens; with go its gradients too. Returns (out, gpK, gpQ, gV, A, B)."""
    N, T, S = pK.shape
    pad = -T % c
    if pad:
        pK, pQ, V = (torch.nn.functional.pad(x, (0, 0, 0, pad)) for x in (pK, pQ, V))
        go = None if go is None else torch.nn.functional.pad(go, (0, 0, 0, pad))
    nc = (T + pad) // c

    def cut(x):
        return x.reshape(N, nc, c, -1)

    def flat(x):
        return x.reshape(N, T + pad, -1)[:, :T]

    tri = torch.ones(c, c, dtype=F64, device=pK.device).tril()
    A = pK.cumsum(1)
    inv = cut(1.0 / (A + eps)) if normalise else 1.0
    A_end = A[:, -1]
    k, q, v = cut(pK), cut(pQ), cut(V)
    tot = k.transpose(-1, -2) @ v
    B_end = tot.sum(1)
    B0 = tot.cumsum(1) - tot
    del tot, A
    W = q * inv
    P = (W @ k.transpose(-1, -2)) * tri
    out = W @ B0 + P @ v
    if go is None:
        return flat(out), None, None, None, A_end, B_end
    g = cut(go)
    M = (g @ v.transpose(-1, -2)) * tri
    gpQ = (g @ B0.transpose(-1, -2) + M @ k) * inv
    del B0
    tot = W.transpose(-1, -2) @ g
    dS = tot.flip(1).cumsum(1).flip(1) - tot
    del tot
    gpK = v @ dS.transpose(-1, -2) + M.transpose(-1, -2) @ W
    if normalise:
        gA = -gpQ * W
        gpK = gpK + cut(gA.reshape(N, nc * c, S).flip(1).cumsum(1).flip(1))
    gV = k @ dS + P.transpose(-1, -2) @ g
    return flat(out), flat(gpK), flat(gpQ), flat(gV), A_end, B_end


def _layer64(q, k, v, go, planes, L, K, eps):
    """(out, dq, dk, dv, A, B) of the causal layer, q and go [B,Hq,T,D], k and v [B,Hkv,T,D], a few streams at a time."""
    B, Hq, T, D = q.shape
    Hkv, G, scale = k.shape[1], Hq // k.shape[1], math.sqrt(D)
    planes = planes.to(F64)
    qs, gos = (None if x is None else x.reshape(B * Hkv, G, T, D) for x in (q, go))
    ks, vs = k.reshape(B * Hkv, T, D), v.reshape(B * Hkv, T, D)
    step = max(1, (1 << 20) // (G * T))
    parts = []
    for z in range(0, B * Hkv, step):
        x, y = qs[z:z + step].to(F64).requires_grad_(go is not None), ks[z:z + step].to(F64).requires_grad_(go is not None)
        n = x.shape[0]
        w = vs[z:z + step].to(F64)
        with torch.enable_grad():
            pQ, pK = _hash64(x.reshape(n * G, T, D), planes, L, K, scale), _hash64(y, planes, L, K, scale)
        rep = lambda t: t.detach().repeat_interleave(G, 0)  # noqa: E731
        g = None if go is None else gos[z:z + step].to(F64).reshape(n * G, T, D)
        o, gk, gq, gv, A, Bs = _scan64(rep(pK), pQ.detach(), rep(w), g, eps)
        if go is None:
            parts.append((o.view(n, G, T, D), A[::G], Bs[::G]))
            continue
        dq, = torch.autograd.grad(pQ, x, gq)
        dk, = torch.autograd.grad(pK, y, gk.view(n, G, T, -1).sum(1))
        parts.append((o.view(n, G, T, D), dq, dk, gv.view(n, G, T, D).sum(1)))
        del x, y, w, pQ, pK, g, o, gk, gq, gv
    got = [torch.cat(p) for p in zip(*parts)]
    if go is None:
        return got[0].view(B, Hq, T, D), got[1], got[2]
    return got[0].view(B, Hq, T, D), got[1].view(B, Hq, T, D), got[2].view(B, Hkv, T, D), got[3].view(B, Hkv, T, D)


def _noncausal64(s):
    _, B, T, H, D = s["q"].shape
    lt = s["ace"].logit_temp.detach().to(F64).requires_grad_()
    planes = s["ace"].planes_T.to(F64)
    out, dq, dk, dv = (torch.empty(1, B, T, H, D, dtype=F64, device=DEV) for _ in range(4))
    dlt = torch.zeros((), dtype=F64, device=DEV)
    for b in range(B):
        for h in range(H):
            q, k, v = (s[n][0, b, :, h].detach().to(F64)[None].requires_grad_() for n in "qkv")
            scale = lt.exp().clamp(1e-2, 10.0)
            pK, pQ = (_hash64(x, planes, s["L"], s["K"], scale) for x in (k, q))
            o = pQ @ ((pK.transpose(1, 2) @ v) / (pK.sum(1).unsqueeze(-1) + EPS))
            gq, gk, gv, gt = torch.autograd.grad(o, (q, k, v, lt), s["go"][0, b, :, h].to(F64)[None])
            for dst, x in ((out, o), (dq, gq), (dk, gk), (dv, gv)):
                dst[0, b, :, h] = x[0].detach()
            dlt += gt
    return out, dq, dk, dv, dlt


def exact(case, seed):
    s = prepare(case, seed)
    kind = s["kind"]
    if kind == "noncausal":
        return _noncausal64(s)
    with torch.no_grad():
        if kind == "linear":
            B, H, T, D = s["q"].shape
            parts = []
            for z in range(B * H):
                q, k, v, go = (s[n].detach().view(B * H, T, D)[z:z + 1].to(F64) for n in ("q", "k", "v", "go"))
                o, gk, gq, gv, _, _ = _scan64(k, q, v, go, 0.0, normalise=False)
                parts.append((o, gq, gk, gv))
            return tuple(torch.cat(p).view(B, H, T, D) for p in zip(*parts))
        if kind == "decode":
            # bf16 inputs hash with planes rounded to bf16, as the reference does
            st, D = s["st"], s["D"]
            planes = (s["planes"].bfloat16() if s["dtype"] == "bf16" else s["planes"]).to(F64)
            n, G = s["B"] * s["Hkv"], s["Hq"] // s["Hkv"]
            hash_ = lambda x: _hash64(x.to(F64)[:, None], planes, s["L"], s["K"], math.sqrt(D))[:, 0]  # noqa: E731
            pK, pQ = hash_(s["k"].reshape(n, D)), hash_(s["q"].reshape(n * G, D)).view(n, G, -1)
            A = st.A.to(F64) + pK
            Bs = st.Bs.to(F64) + pK[:, :, None] * s["v"].reshape(n, 1, D).to(F64)
            out = (pQ / (A + EPS)[:, None]) @ Bs
            return out.view(s["B"], s["Hq"], D), A, Bs
        if kind == "module":
            return _layer64(s["q"].detach(), s["k"].detach(), s["v"].detach(), s["go"], s["mod"].planes_T, s["L"], s["K"], EPS)
        rounded = s["planes"] if s.get("precision") == "fp32" else s["planes"].bfloat16()
        if kind == "prefill":
            return _layer64(s["q"], s["k"], s["v"], None, rounded, s["L"], s["K"], EPS)
        if kind == "layer":
            return _layer64(s["q"].detach(), s["k"].detach(), s["v"].detach(), s["go"], rounded, s["L"], s["K"], EPS)
        B, T, Hq, D = s["q"].shape
        bhtd = lambda x: x.detach().transpose(1, 2)  # noqa: E731
        out, dq, dk, dv = _layer64(bhtd(s["q"]), bhtd(s["k"]), bhtd(s["v"]), bhtd(s["go"].view(B, T, Hq, D)), rounded,
                                   s["L"], s["K"], EPS)
        return tuple(x.transpose(1, 2).contiguous() for x in (out.contiguous(), dq, dk, dv))
