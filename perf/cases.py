"""Performance cases: the layer calls a decode engine makes through ``qengine_amd``.

Each case is one part of a model pass over several layers, every layer with its own cache, weights
or state (so that a pass streams them from HBM as a whole model does). Decode, verify, projection
and Gated DeltaNet passes are captured once in a hipGraph and replayed, as the engine runs them;
prompt chunks, whose sizes change from call to call, are called eagerly.

Shapes are those of the repository's benchmark and tests: 24 query heads over 4 KV heads of 256
dims (also 16 / 2 and 32 / 8), hidden size 5120, 16 key / 48 value heads of 128 in the Gated
DeltaNet layers, a vocabulary of 248,320.
"""
from __future__ import annotations

import math

import torch
import torch.nn.functional as F

import qengine_amd as qa
from qengine_amd import _C
from qengine_amd.layer import rope_inv_freq

BF, F32, F64 = torch.bfloat16, torch.float32, torch.float64
DEV = "cuda"
D = 256            # head dim of the attention layers
DK = 128           # head dim of the Gated DeltaNet layers
EPS = 1e-6
THETA, ROTARY = 1e7, 64
HIDDEN, VOCAB = 5120, 248320
KV_SCALE = 1.0 / 16  # fp8 cache: one scale for unit-scale K and V
FP8 = torch.float8_e4m3fn


def listed():
    return [
        # one token of a short conversation: latency and launches count, hardly any bytes
        dict(name="decode_1k", kind="decode", hq=24, hkv=4, rows=1, pos=1000, max_len=2048,
             layers=16, kv="bf16"),
        # one token at an ordinary context length (odd, in a cache with room left)
        dict(name="decode_16k", kind="decode", hq=24, hkv=4, rows=1, pos=16201, max_len=16384,
             layers=8, kv="bf16"),
        # one token at a long context on the half-size cache
        dict(name="decode_fp8_64k", kind="decode", hq=24, hkv=4, rows=1, pos=65500,
             max_len=65536, layers=4, kv="fp8"),
        # speculative verify of four drafts
        dict(name="verify_5_4k", kind="decode", hq=24, hkv=4, rows=5, pos=4096, max_len=4104,
             layers=16, kv="bf16"),
        # the widest verify pass, on the other head grouping (8 query heads per KV head)
        dict(name="verify_8_gqa8_6k", kind="decode", hq=16, hkv=2, rows=8, pos=6001, max_len=8192,
             layers=16, kv="bf16"),
        # a long prompt's later chunk: the large, compute-bound call
        dict(name="prefill_2048_on_2048", kind="prefill", hq=24, hkv=4, rows=2048, pos=2048,
             max_len=4096, layers=4, kv="bf16"),
        # a user's next turn in a conversation of 12k positions
        dict(name="prefill_301_on_12k", kind="prefill", hq=24, hkv=4, rows=301, pos=12007,
             max_len=16384, layers=4, kv="bf16"),
        # a whole short prompt from an empty fp8 cache
        dict(name="prefill_777_fp8", kind="prefill", hq=24, hkv=4, rows=777, pos=0, max_len=2048,
             layers=4, kv="fp8"),
        # the projections around attention, one token: weight streaming
        dict(name="proj_1", kind="proj", rows=1, layers=4),
        # the recurrent layers of one token (the last one kept): 48 layers, one state each
        dict(name="gdn_1", kind="gdn", rows=1, pending=1, layers=48),
        # the recurrent layers of a verify pass after three kept rows
        dict(name="gdn_6_pending_3", kind="gdn", rows=6, pending=3, layers=48),
        # the head of a verify pass: final norm with residual, vocabulary logits, argmax
        dict(name="head_5", kind="head", rows=5),
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "verify", "verify", "prefill", "prefill", "prefill",
                       "proj", "gdn", "head"])
    hq, hkv = rng.choice([(24, 4), (24, 4), (24, 4), (16, 2), (32, 8)])
    kv = rng.choice(["bf16", "bf16", "fp8"])
    if kind in ("decode", "verify"):
        rows = 1 if kind == "decode" else rng.randint(2, 8)
        pos = _log(rng, 200, 131000)
        max_len = pos + rows + rng.choice([0, rng.randint(1, 4000)])
        layer_bytes = 4 * D * hkv * pos  # rough: bf16 K and V
        return dict(kind="decode", hq=hq, hkv=hkv, rows=rows, pos=pos, max_len=max_len,
                    layers=max(1, min(16, int(6e8 / layer_bytes))), kv=kv)
    if kind == "prefill":
        rows = _log(rng, 9, 2048)
        most = 1.5e11 / (4 * D * hq * rows) - rows / 2  # no more than the largest listed call
        pos = rng.choice([0, _log(rng, 16, max(17, min(48000, int(most))))])
        max_len = pos + rows + rng.choice([0, rng.randint(1, 4000)])
        return dict(kind="prefill", hq=hq, hkv=hkv, rows=rows, pos=pos, max_len=max_len, layers=4,
                    kv=kv)
    if kind == "gdn":
        rows = rng.randint(1, 8)
        return dict(kind="gdn", rows=rows, pending=rng.randint(0, 8), layers=rng.randint(24, 48))
    if kind == "proj":
        return dict(kind="proj", rows=rng.randint(1, 8), layers=rng.randint(2, 5))
    return dict(kind="head", rows=rng.randint(1, 8))


# ---------------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape, scale=1.0, dtype=BF):
    x = torch.empty(shape, dtype=dtype, device=DEV).normal_(generator=g)
    return x if scale == 1.0 else x.mul_(scale)


def _capture(call):
    """The pass as a hipGraph, after one eager call."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    return graph


def _attn_inputs(case, seed):
    """Projection rows, norm weights and filled caches of every layer. One key row in a hundred
    is four times the others' length, so that some of the softmax is peaked."""
    g = _gen(seed)
    hq, hkv, n, nl = case["hq"], case["hkv"], case["rows"], case["layers"]
    s = dict(case=case)
    s["proj"] = _randn(g, nl, n, hq * 2 * D + 2 * hkv * D)
    s["qnw"] = _randn(g, nl, D, scale=0.3)
    s["knw"] = _randn(g, nl, D, scale=0.3)
    s["inv_freq"] = rope_inv_freq(THETA, ROTARY, DEV)
    s["pos"] = torch.tensor([case["pos"]], dtype=torch.int32, device=DEV)
    kc, vc = (torch.zeros(nl, hkv, case["max_len"], D, dtype=BF, device=DEV) for _ in range(2))
    kc[:, :, : case["pos"]].normal_(generator=g)
    vc[:, :, : case["pos"]].normal_(generator=g)
    if case["pos"]:
        peak = torch.rand(nl, hkv, case["pos"], 1, device=DEV, generator=g) < 0.01
        kc[:, :, : case["pos"]] *= 1 + 3 * peak.to(BF)
    if case["kv"] == "fp8":
        kc, vc = (t.div_(KV_SCALE).to(FP8) for t in (kc, vc))
    s["kc"], s["vc"] = kc, vc
    return s


def _split_proj(case, proj):
    q0 = case["hq"] * 2 * D
    k1 = q0 + case["hkv"] * D
    return proj[:, :q0], proj[:, q0:k1], proj[:, k1:]


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        s = _attn_inputs(case, seed)
        n, hq, nl = case["rows"], case["hq"], case["layers"]
        s["q"] = torch.zeros(nl, n, hq * D, dtype=BF, device=DEV)
        s["out"] = torch.zeros(nl, n, hq * D, dtype=BF, device=DEV)
        if kind == "decode":
            ns = qa.default_splits(case["max_len"], case["hkv"], kv8=case["kv"] == "fp8")
            s["part_o"], s["part_ml"] = qa.alloc_partials(n, hq, ns, DEV)
            s["graph"] = _capture(lambda: _decode_layers(s))
        return s
    g = _gen(seed)
    if kind == "proj":
        n, nl = case["rows"], case["layers"]
        s = dict(case=case, x=_randn(g, nl, n, HIDDEN), a=_randn(g, nl, n, 24 * D),
                 w_in=_randn(g, nl, 14336, HIDDEN, scale=HIDDEN ** -0.5),
                 w_o=_randn(g, nl, HIDDEN, 24 * D, scale=(24 * D) ** -0.5))
        s["y_in"] = torch.zeros(nl, n, 14336, dtype=BF, device=DEV)
        s["y_o"] = torch.zeros(nl, n, HIDDEN, dtype=BF, device=DEV)
        s["graph"] = _capture(lambda: _proj_layers(s))
        return s
    if kind == "gdn":
        return _prepare_gdn(case, g)
    n = case["rows"]  # head
    s = dict(case=case, x0=_randn(g, n, HIDDEN), delta=_randn(g, n, HIDDEN, scale=0.3),
             w=_randn(g, HIDDEN, scale=0.1), head=_randn(g, VOCAB, HIDDEN, scale=HIDDEN ** -0.5))
    h = (s["x0"] + s["delta"]).float()
    h = h * torch.rsqrt(h.square().mean(-1, keepdim=True) + EPS) * (1 + s["w"].float())
    ids = torch.arange(n, device=DEV) * 30011 + 17  # one token of every row stands out
    s["head"][ids] += (h * (8.0 / HIDDEN)).to(BF)
    s["x"] = s["x0"].clone()
    s["hid"] = torch.zeros(n, HIDDEN, dtype=BF, device=DEV)
    s["logits"] = torch.zeros(n, VOCAB, dtype=BF, device=DEV)
    s["ws_v"] = torch.zeros(n * 256, dtype=F32, device=DEV)
    s["ws_i"] = torch.zeros(n * 256, dtype=torch.int32, device=DEV)
    s["ids"] = torch.zeros(n, dtype=torch.int32, device=DEV)
    s["graph"] = _capture(lambda: _head(s))
    return s


def _prepare_gdn(case, g):
    nl, n, hk, hv = case["layers"], case["rows"], 16, 48
    C = 2 * hk * DK + hv * DK
    width = (C + hv * DK + 2 * hv + 7) // 8 * 8
    s = dict(case=case, proj=_randn(g, nl, n, width),
             conv_w=_randn(g, nl, C, 4, scale=0.5),
             A_log=torch.empty(nl, hv, device=DEV).uniform_(-3.0, 1.0, generator=g).to(BF),
             dt=_randn(g, nl, hv), norm_w=(1 + _randn(g, nl, DK, scale=0.1)))
    first = dict(
        S=_randn(g, nl, hv, DK, DK, scale=0.1, dtype=F32), ring=_randn(g, nl, 16, C),
        st_k=F.normalize(_randn(g, nl, 8, hv, DK, dtype=F32), dim=-1),
        st_v=_randn(g, nl, 8, hv, DK, scale=0.3, dtype=F32),
        st_g=torch.rand(nl, 8, hv, 2, device=DEV, generator=g))
    s["ctl"] = torch.tensor([1000, case["pending"]], dtype=torch.int32, device=DEV)
    s["out"] = torch.zeros(nl, n, hv * DK, dtype=BF, device=DEV)
    s.update({k: v.clone() for k, v in first.items()})
    s["graph"] = _capture(lambda: _gdn_layers(s))
    for k, v in first.items():  # as before the eager call of the capture
        s[k].copy_(v)
    return s


# ---------------------------------------------------------------------------------- passes
def _prep(s, l):
    case = s["case"]
    qg, k, v = _split_proj(case, s["proj"][l])
    args = (qg, k, v, s["qnw"][l], s["knw"][l], s["inv_freq"], s["pos"], s["q"][l], s["kc"][l],
            s["vc"][l], EPS)
    if case["kv"] == "fp8":
        _C.attn_prep_fp8(*args, KV_SCALE, KV_SCALE)
    elif case["kind"] == "prefill":
        _C.attn_prep_chunk(*args)
    else:
        _C.attn_prep(*args)
    return qg


def _decode_layers(s):
    fp8 = s["case"]["kv"] == "fp8"
    for l in range(s["case"]["layers"]):
        qg = _prep(s, l)
        args = (s["q"][l], s["kc"][l], s["vc"][l], s["pos"], qg, s["part_o"], s["part_ml"],
                s["out"][l])
        if fp8:
            _C.attn_decode_fp8(*args, KV_SCALE, KV_SCALE)
        else:
            _C.attn_decode(*args)


def _prefill_layers(s):
    fp8 = s["case"]["kv"] == "fp8"
    for l in range(s["case"]["layers"]):
        qg = _prep(s, l)
        args = (s["q"][l], s["kc"][l], s["vc"][l], s["pos"], qg, s["out"][l])
        if fp8:
            _C.attn_prefill_fp8(*args, KV_SCALE, KV_SCALE)
        else:
            _C.attn_prefill(*args)


def _proj_layers(s):
    for l in range(s["case"]["layers"]):
        _C.gemv_bf16(s["w_in"][l], s["x"][l], s["y_in"][l])
        _C.gemv_bf16(s["w_o"][l], s["a"][l], s["y_o"][l])


def _gdn_layers(s):
    hk, hv = 16, 48
    c0 = 2 * hk * DK + hv * DK
    c1 = c0 + hv * DK
    for l in range(s["case"]["layers"]):
        pr = s["proj"][l]
        _C.gdn_step_n(pr[:, :c0], pr[:, c0:c1], pr[:, c1:c1 + hv], pr[:, c1 + hv:c1 + 2 * hv],
                      s["ring"][l], s["conv_w"][l], s["A_log"][l], s["dt"][l], s["norm_w"][l],
                      s["S"][l], s["st_k"][l], s["st_v"][l], s["st_g"][l], s["ctl"], s["out"][l],
                      hk, EPS)


def _head(s):
    s["x"].copy_(s["x0"])  # the residual stream that the layers before would have written
    _C.rmsnorm1p(s["x"], s["delta"], s["w"], s["hid"], EPS)
    _C.gemv_bf16(s["head"], s["hid"], s["logits"])
    _C.argmax(s["logits"], s["ws_v"], s["ws_i"], s["ids"])


_OUT = {"decode": ("out", "q", "kc", "vc"), "prefill": ("out", "q", "kc", "vc"),
        "proj": ("y_in", "y_o"), "gdn": ("out", "S", "ring", "st_k", "st_v", "st_g"),
        "head": ("ids", "logits", "x", "hid")}


def run(s):
    kind = s["case"]["kind"]
    if kind == "prefill":
        _prefill_layers(s)
    else:
        s["graph"].replay()
    return {k: s[k] for k in _OUT[kind]}


# ------------------------------------------------------------------------ work and precision
def work(case):
    kind, n = case["kind"], case["rows"]
    if kind in ("decode", "prefill"):
        hq, hkv = case["hq"], case["hkv"]
        e = 1 if case["kv"] == "fp8" else 2
        attended = [min(case["pos"] + t + 1, case["max_len"]) for t in range(n)]
        kv = 2 * hkv * D * e * (attended[-1] + n)     # K and V read once, the new rows written
        rows = n * 2 * (hq * 2 * D + 2 * hkv * D + 2 * hq * D)  # projection in, q and out
        return {"bytes": case["layers"] * (kv + rows),
                "flops": case["layers"] * 4 * D * hq * sum(attended)}
    if kind == "proj":
        w = 14336 * HIDDEN + HIDDEN * 24 * D
        io = n * (HIDDEN + 14336 + 24 * D + HIDDEN)
        return {"bytes": case["layers"] * 2 * (w + io), "flops": case["layers"] * 2 * n * w}
    if kind == "gdn":
        hk, hv, pend = 16, 48, case["pending"]
        C = 2 * hk * DK + hv * DK
        state = 4 * hv * DK * DK * (2 if pend else 1)
        staged = (pend + n) * 4 * hv * (2 * DK + 2)
        rows = n * 2 * (C + 2 * hv * DK + 2 * hv)
        return {"bytes": case["layers"] * (state + staged + rows + 2 * C * (4 + 3 + n)),
                "flops": case["layers"] * hv * DK * DK * (4 * pend + 6 * n)}
    return {"bytes": 2 * (VOCAB * HIDDEN + n * (4 * HIDDEN + VOCAB)),
            "flops": 2 * n * VOCAB * HIDDEN}


def tolerance(case):
    # bf16 results: another summation order moves some values by one rounding (2^-8 of the value)
    return {"rel": 1e-2, "max": 0.25, "differ": 0.005}


def _norm_rope(x, w, pos0, inv_freq):
    """RMSNorm with weight 1 + w and rotate-half RoPE of x [n, heads, D], in 64 bits."""
    x = x.to(F64)
    x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * (1 + w.to(F64))
    p = torch.arange(x.shape[0], device=DEV, dtype=F32) + pos0
    ang = (p[:, None] * inv_freq[None]).to(F64)[:, None]  # the angle is an fp32 product
    c, s, h = ang.cos(), ang.sin(), inv_freq.numel()
    a, b = x[..., :h], x[..., h:2 * h]
    return torch.cat([a * c - b * s, b * c + a * s, x[..., 2 * h:]], -1)


def _exact_attn(case, seed):
    s = _attn_inputs(case, seed)
    n, hq, hkv, pos, ml = (case[k] for k in ("rows", "hq", "hkv", "pos", "max_len"))
    fp8, grp = case["kv"] == "fp8", hq // hkv
    L = min(pos + n, ml)
    qs, outs = [], []
    kcs, vcs = (s[t].to(F64) if not fp8 else s[t].to(F32) for t in ("kc", "vc"))
    for l in range(case["layers"]):
        qg, k, v = _split_proj(case, s["proj"][l])
        qg = qg.reshape(n, hq, 2, D)
        q = _norm_rope(qg[:, :, 0], s["qnw"][l], pos, s["inv_freq"])
        k = _norm_rope(k.reshape(n, hkv, D), s["knw"][l], pos, s["inv_freq"])
        v = v.reshape(n, hkv, D).to(F64)
        if fp8:
            k, v = ((t.to(BF).to(F32) / KV_SCALE).to(FP8).to(F64) for t in (k, v))
        m = max(0, L - pos)
        kcs[l, :, pos:L] = k[:m].transpose(0, 1)
        vcs[l, :, pos:L] = v[:m].transpose(0, 1)
        scale = KV_SCALE if fp8 else 1.0
        end = (torch.arange(n, device=DEV) + pos + 1).clamp(max=ml)
        seen = torch.arange(L, device=DEV)[None] < end[:, None]
        o = torch.empty(n, hq, D, dtype=F64, device=DEV)
        for g in range(hkv):
            K, V = kcs[l, g, :L].to(F64) * scale, vcs[l, g, :L].to(F64) * scale
            for h in range(g * grp, (g + 1) * grp):
                sc = (q[:, h] @ K.t().contiguous()) / 16
                o[:, h] = torch.softmax(sc.masked_fill(~seen, -math.inf), -1) @ V
        outs.append((o * torch.sigmoid(qg[:, :, 1].to(F64))).reshape(n, hq * D))
        qs.append(q.reshape(n, hq * D))
    return {"out": torch.stack(outs), "q": torch.stack(qs), "kc": kcs, "vc": vcs}


def _delta(S, k, v, g):
    """One delta-rule update of S [layers, heads, 128, 128]."""
    S.mul_(g[..., 0, None, None])
    kv = (S.transpose(-1, -2) @ k[..., None])[..., 0]
    S.add_(k[..., None] * ((v - kv) * g[..., 1, None])[..., None, :])


def _exact_gdn(case, seed):
    s = _prepare_gdn(case, _gen(seed))
    nl, n, hk, hv = case["layers"], case["rows"], 16, 48
    C, pos = 2 * hk * DK + hv * DK, 1000
    S, st_k, st_v, st_g = (s[k].to(F64) for k in ("S", "st_k", "st_v", "st_g"))
    ring, x = s["ring"].to(F64), s["proj"].to(F64)
    for t in range(case["pending"]):
        _delta(S, st_k[:, t], st_v[:, t], st_g[:, t])
    committed, outs = S.clone(), []
    c1 = C + hv * DK
    for t in range(n):
        taps = [x[:, i, :C] if (i := t - back) >= 0 else ring[:, (pos + i) % 16]
                for back in (3, 2, 1, 0)]
        y = F.silu((torch.stack(taps, -1) * s["conv_w"].to(F64)).sum(-1))
        unit = [y[:, i * hk * DK:(i + 1) * hk * DK].view(nl, hk, DK) for i in (0, 1)]
        q, k = (u * torch.rsqrt(u.square().sum(-1, keepdim=True) + 1e-6) for u in unit)
        q, k = (u.repeat_interleave(hv // hk, 1) for u in (q / math.sqrt(DK), k))
        v = y[:, 2 * hk * DK:].view(nl, hv, DK)
        b, a = x[:, t, c1:c1 + hv], x[:, t, c1 + hv:c1 + 2 * hv]
        g = torch.stack([torch.exp(-s["A_log"].to(F64).exp() * F.softplus(a + s["dt"].to(F64))),
                         torch.sigmoid(b)], -1)
        st_k[:, t], st_v[:, t], st_g[:, t] = k, v, g
        _delta(S, k, v, g)
        o = (S.transpose(-1, -2) @ q[..., None])[..., 0]
        o = o * torch.rsqrt(o.square().mean(-1, keepdim=True) + EPS) * s["norm_w"].to(F64)[:, None]
        outs.append((o * F.silu(x[:, t, C:c1].view(nl, hv, DK))).reshape(nl, -1))
    for t in range(n):
        ring[:, (pos + t) % 16] = x[:, t, :C]
    return {"out": torch.stack(outs, 1), "S": committed, "ring": ring, "st_k": st_k, "st_v": st_v,
            "st_g": st_g}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        return _exact_attn(case, seed)
    if kind == "gdn":
        return _exact_gdn(case, seed)
    s = prepare(case, seed)
    if kind == "proj":
        return {"y_in": torch.stack([x @ w.t() for x, w in zip(s["x"].to(F64), s["w_in"].to(F64))]),
                "y_o": torch.stack([x @ w.t() for x, w in zip(s["a"].to(F64), s["w_o"].to(F64))])}
    x = s["x0"].to(F64) + s["delta"].to(F64)
    h = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * (1 + s["w"].to(F64))
    logits = torch.cat([h @ w.to(F64).t() for w in s["head"].split(VOCAB // 16)], -1)
    return {"ids": logits.argmax(-1).to(torch.int32), "logits": logits, "x": x, "hid": h}
