"""The work that users of this decoder have it do, as measurable cases.

Sizes are those of the Qwen3-4B layer (hidden 2560, intermediate 9728, 32 query and 8 KV heads of
128, vocabulary 151936).  Kinds:

  norm         residual add + RMSNorm over `rows` token rows (the smallest call of a step)
  proj         one layer's four projections over `rows` rows: norm + qkv, o + residual, norm +
               gate/up + SwiGLU, down + residual -- batched decode, tree verification and prefill
               differ here only by the row count
  head         final norm + LM head with its fp32 logits, for samplers that need them
  attn_decode  one new token for each of B sequences against their caches
  attn_causal  a prompt chunk's attention: q/k norm + RoPE + cache write, then causal attention
  attn_tree    the same for a draft tree under its ancestor masks (speculative verification)
  decode       a whole decode step of a model of `layers` layers, with the next token's logits
  prefill      a whole prompt forward, with the last token's logits
"""

import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "htn-2026_amd")
if _PKG not in sys.path:
    sys.path.insert(1, _PKG)

from qdecode import _lib, model as _model, ops  # noqa: E402

H, I, V, HQ, HKV, D = 2560, 9728, 151936, 32, 8, 128
QD, NQKV = HQ * D, (HQ + 2 * HKV) * D
EPS, THETA = 1e-6, 5000000.0
LAYER_W = NQKV * H + H * QD + 3 * I * H          # weights of one layer's projections
BF16, F64 = torch.bfloat16, torch.float64


def listed():
    return [
        # one token's residual add + norm: launch latency
        {"name": "norm_1", "kind": "norm", "rows": 1, "add": True},
        # a layer's projections for a mid-sized serving batch, not a power of two
        {"name": "proj_48", "kind": "proj", "rows": 48},
        # ... for a short prompt of odd length
        {"name": "proj_601", "kind": "proj", "rows": 601},
        # ... for a few prompts of some hundred tokens
        {"name": "proj_3000", "kind": "proj", "rows": 3000},
        # ... for a large prompt chunk (8 x 2048 tokens)
        {"name": "proj_16384", "kind": "proj", "rows": 16384},
        # logits for a serving batch's sampler
        {"name": "head_40", "kind": "head", "rows": 40},
        # 20 conversations of 3000 tokens, one new token each
        {"name": "attn_decode_20x3000", "kind": "attn_decode", "B": 20, "ctx": 3000},
        # two long prompts
        {"name": "attn_causal_2x4096", "kind": "attn_causal", "B": 2, "T": 4096, "base": 0},
        # 64-node draft trees over long contexts
        {"name": "attn_tree_4x64", "kind": "attn_tree", "B": 4, "T": 64, "base": 8192},
        # the full model generating one conversation's next token
        {"name": "decode_1", "kind": "decode", "layers": 36, "B": 1, "ctx": 700},
        # a batch of 32 conversations, one new token each; four of the 36 equal layers
        {"name": "decode_32", "kind": "decode", "layers": 4, "B": 32, "ctx": 2100},
        # the full model reading a 512-token prompt: the wait for the first token
        {"name": "prefill_512", "kind": "prefill", "layers": 36, "B": 1, "T": 512},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    kind = rng.choice(["norm", "proj", "proj", "head", "attn_decode", "attn_causal", "attn_tree",
                       "decode", "prefill"])
    if kind == "norm":
        return {"kind": kind, "rows": _log_int(rng, 1, 32768), "add": rng.random() < 0.7}
    if kind == "proj":
        return {"kind": kind, "rows": _log_int(rng, 1, 16384)}
    if kind == "head":
        return {"kind": kind, "rows": _log_int(rng, 1, 256)}
    if kind == "attn_decode":
        B = _log_int(rng, 1, 96)
        return {"kind": kind, "B": B, "ctx": _log_int(rng, 64, max(128, 131072 // B))}
    if kind == "attn_causal":
        B = _log_int(rng, 1, 8)
        return {"kind": kind, "B": B, "T": _log_int(rng, 17, 8192 // B),
                "base": rng.choice([0, 0, _log_int(rng, 64, 8192)])}
    if kind == "attn_tree":
        return {"kind": kind, "B": _log_int(rng, 1, 8), "T": rng.randint(8, 64),
                "base": _log_int(rng, 100, 16384)}
    if kind == "decode":
        B = _log_int(rng, 1, 128)
        return {"kind": kind, "layers": 4, "B": B, "ctx": _log_int(rng, 64, max(128, 131072 // B))}
    B = _log_int(rng, 1, 4)
    return {"kind": kind, "layers": 4, "B": B, "T": _log_int(rng, 16, 4096 // B)}


# ------------------------------------------------------------------ preparation
class _Rand:
    """bf16 (or int64) tensors on the GPU from one seed."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape, std=1.0, mean=0.0):
        return torch.empty(shape, dtype=BF16, device="cuda").normal_(mean, std, generator=self.g)

    def fill(self, t, std=1.0, mean=0.0):
        t.normal_(mean, std, generator=self.g)

    def ids(self, *shape):
        return torch.randint(0, V, shape, generator=self.g, device="cuda", dtype=torch.int64)


def _empty(*shape, dtype=BF16):
    return torch.empty(shape, dtype=dtype, device="cuda")


def _tree(B, T, seed):
    """Random draft trees: node 0 is the root, each later node hangs under an earlier one at most
    six levels deep.  depth [B, T], ancestor-or-self masks [B, T] (bit j: node j)."""
    g = torch.Generator()
    g.manual_seed(seed)
    depth, anc = [], []
    for _ in range(B):
        d, a = [0], [1]
        for j in range(1, T):
            par = int(torch.randint(0, j, (1,), generator=g))
            while d[par] >= 6:
                par = int(torch.randint(0, j, (1,), generator=g))
            d.append(d[par] + 1)
            a.append(a[par] | (1 << j))
        depth.append(d)
        anc.append([x - (1 << 64) if x >= 1 << 63 else x for x in a])
    return (torch.tensor(depth, dtype=torch.int64, device="cuda"),
            torch.tensor(anc, dtype=torch.int64, device="cuda"))


def _attn_cap(c):
    """Cache slots of the attention kinds: what is used, and some room to go on."""
    used = c["ctx"] + 1 if c["kind"] in ("attn_decode", "decode") else c["base"] + c["T"]
    return used + 32


def _fill_model(m, r):
    """Random weights of the benchmark's scale; norm weights around one."""
    for t in (m.embed, m.w_qkv, m.w_o, m.w_gu, m.w_down):
        r.fill(t, 0.02)
    for t in (m.final_norm, m.ln1, m.ln2, m.q_norm, m.k_norm):
        r.fill(t, 0.1, 1.0)


def prepare(case, seed):
    c, k, r = case, case["kind"], _Rand(seed)
    s = {"case": dict(c)}
    if k == "norm":
        rows = c["rows"]
        s["res"], s["w"] = r.normal(rows, H), r.normal(H, std=0.1, mean=1.0)
        s["x"] = r.normal(rows, H, std=0.5) if c["add"] else None
        s["res_out"] = _empty(rows, H) if c["add"] else None
        s["y"] = _empty(rows, H)
        return s
    if k == "proj":
        rows = c["rows"]
        s["x"], s["attn"] = r.normal(rows, H), r.normal(rows, QD, std=0.5)
        s["ln1"], s["ln2"] = r.normal(H, std=0.1, mean=1.0), r.normal(H, std=0.1, mean=1.0)
        s["w_qkv"], s["w_o"] = r.normal(NQKV, H, std=0.02), r.normal(H, QD, std=0.02)
        s["w_gu"], s["w_down"] = r.normal(2 * I, H, std=0.02), r.normal(H, I, std=0.02)
        s["qkv"], s["x1"] = _empty(rows, NQKV), _empty(rows, H)
        s["act"], s["x2"] = _empty(rows, I), _empty(rows, H)
        need = max(_lib.LIB.qd_linear_workspace_bytes(rows, n, kk, norm)
                   for n, kk, norm in ((NQKV, H, 1), (H, QD, 0), (I, H, 1), (H, I, 0)))
        s["ws"] = ops.workspace(need, "cuda")
        return s
    if k == "head":
        rows = c["rows"]
        s["x"], s["norm"] = r.normal(rows, H), r.normal(H, std=0.1, mean=1.0)
        s["w"] = r.normal(V, H, std=0.02)
        s["tok"] = _empty(rows, dtype=torch.int64)
        s["logits"] = _empty(rows, V, dtype=torch.float32)
        s["ws"] = ops.workspace(_lib.LIB.qd_lm_head_workspace_bytes(rows, V, H), "cuda")
        return s
    if k.startswith("attn"):
        B, cap = c["B"], _attn_cap(c)
        s["qn"], s["kn"] = r.normal(D, std=0.1, mean=1.0), r.normal(D, std=0.1, mean=1.0)
        s["k"], s["v"] = r.normal(B, HKV, cap, D), r.normal(B, HKV, cap, D, std=0.5)
        cos, sin = _model.rope_tables(cap, THETA, D)
        s["cos"], s["sin"] = cos.cuda(), sin.cuda()
        if k == "attn_decode":
            s["qkv"], s["out"] = r.normal(B, NQKV), _empty(B, HQ, D)
            s["pos"] = torch.full((1,), c["ctx"], dtype=torch.int64, device="cuda")
            s["ws"] = ops.workspace(_lib.LIB.qd_decode_attn_workspace_bytes(B, HQ, HKV, cap), "cuda")
            return s
        T = c["T"]
        s["qkv"], s["q"], s["out"] = r.normal(B * T, NQKV), _empty(B, T, HQ, D), _empty(B, T, HQ, D)
        s["base"] = torch.full((B,), c["base"], dtype=torch.int64, device="cuda")
        s["depth"], s["anc"] = _tree(B, T, seed) if k == "attn_tree" else (None, None)
        s["ws"] = ops.workspace(_lib.LIB.qd_block_attn_workspace_bytes(B, T, HQ, cap), "cuda")
        return s
    # whole calls: a model, its cache and a runner on a stream of its own, as the engine keeps them
    B = c["B"]
    cfg = dict(_model.QWEN3_4B, num_hidden_layers=c["layers"])
    m = s["model"] = _model.Qwen3Model(cfg, "cuda")
    _fill_model(m, r)
    s["stream"] = torch.cuda.Stream()
    s["logits"] = _empty(B, V, dtype=torch.float32)
    s["tok"] = _empty(B, dtype=torch.int64)
    s["ws"] = ops.workspace(_lib.LIB.qd_lm_head_workspace_bytes(B, V, H), "cuda")
    if k == "decode":
        kv = s["kv"] = _model.KVState(m, B, _attn_cap(c))
        r.fill(kv.k)
        r.fill(kv.v, 0.5)
        s["ids"] = r.ids(B)
        s["runner"] = _model.DecodeRunner(kv, s["stream"])
        torch.cuda.synchronize()
        s["runner"].capture()
        return s
    T = c["T"]
    kv = s["kv"] = _model.KVState(m, B, T + 32)
    s["ids"] = r.ids(B, T)
    s["runner"] = _model.BlockRunner(kv, s["stream"], T, causal=True, lm_mode=_lib.LM_LAST)
    torch.cuda.synchronize()
    _prompt(s)                                   # records the forward's graph, as a first prompt does
    torch.cuda.synchronize()
    return s


# ------------------------------------------------------------------ one pass
def _prompt(s):
    run = s["runner"]
    with torch.cuda.stream(s["stream"]):
        run.tokens.copy_(s["ids"])
        run.base.zero_()
        run.launch(s["case"]["T"])


def run(s):
    c = s["case"]
    k = c["kind"]
    if k == "norm":
        ro, y = ops.add_rmsnorm(s["res"], s["w"], EPS, x=s["x"], res_out=s["res_out"], y=s["y"])
        return {"y": y} if ro is None else {"res": ro, "y": y}
    if k == "proj":
        ops.linear(s["x"], s["w_qkv"], norm_w=s["ln1"], eps=EPS, out=s["qkv"], ws=s["ws"])
        ops.linear(s["attn"], s["w_o"], ops.EPI_RES, res=s["x"], out=s["x1"], ws=s["ws"])
        ops.linear(s["x1"], s["w_gu"], ops.EPI_SWIGLU, norm_w=s["ln2"], eps=EPS, out=s["act"],
                   ws=s["ws"])
        ops.linear(s["act"], s["w_down"], ops.EPI_RES, res=s["x1"], out=s["x2"], ws=s["ws"])
        return {"qkv": s["qkv"], "x1": s["x1"], "act": s["act"], "x2": s["x2"]}
    if k == "head":
        ops.lm_head_argmax(s["x"], s["w"], s["norm"], EPS, tok=s["tok"], logits=s["logits"],
                           ws=s["ws"])
        return {"logits": s["logits"], "tok": s["tok"]}
    if k == "attn_decode":
        ops.decode_attention(s["qkv"], s["qn"], s["kn"], s["cos"], s["sin"], s["pos"], s["k"],
                             s["v"], HQ, HKV, EPS, out=s["out"], ws=s["ws"])
        p = c["ctx"]
        return {"out": s["out"], "k": s["k"][:, :, p], "v": s["v"][:, :, p]}
    if k.startswith("attn"):
        B, T, b = c["B"], c["T"], c["base"]
        ops.qk_norm_rope(s["qkv"], s["qn"], s["kn"], s["cos"], s["sin"], s["base"],
                         ops.POS_ROW if s["depth"] is None else ops.POS_TREE, s["q"], s["k"],
                         s["v"], B, T, HQ, HKV, EPS, depth=s["depth"])
        ops.block_attention(s["q"], s["k"], s["v"], s["base"], anc=s["anc"], out=s["out"],
                            ws=s["ws"])
        return {"out": s["out"], "k": s["k"][:, :, b:b + T], "v": s["v"][:, :, b:b + T]}
    m, kv, st, cur = s["model"], s["kv"], s["stream"], torch.cuda.current_stream()
    st.wait_stream(cur)
    if k == "decode":
        p, x = c["ctx"], s["runner"].x
        with torch.cuda.stream(st):
            kv.tok.copy_(s["ids"])
            kv.pos.fill_(p)
            s["runner"].replay()
        new = slice(p, p + 1)
    else:
        T = c["T"]
        x = s["runner"].x.view(-1, T, H)[:, T - 1]        # the last token's rows
        _prompt(s)
        new = slice(0, T)
    with torch.cuda.stream(st):
        ops.lm_head_argmax(x, m.lm_head, m.final_norm, EPS, tok=s["tok"], logits=s["logits"],
                           ws=s["ws"])
    cur.wait_stream(st)
    return {"logits": s["logits"], "k": kv.k[:, :, :, new], "v": kv.v[:, :, :, new]}


# ------------------------------------------------------------------ what a pass cannot do without
def _kv_bytes(tokens):
    return tokens * 2 * HKV * D * 2


def work(case):
    c, k = case, case["kind"]
    if k == "norm":
        n = c["rows"] * H
        return {"bytes": 2 * n * (4 if c["add"] else 2) + 2 * H, "flops": n * (6 if c["add"] else 5)}
    if k == "proj":
        # x and attn in; qkv, x1, act and x2 out
        return {"bytes": 2 * LAYER_W + 2 * c["rows"] * (H + QD + NQKV + 2 * H + I),
                "flops": 2 * c["rows"] * LAYER_W}
    if k == "head":
        return {"bytes": 2 * V * H + c["rows"] * (2 * H + 4 * V), "flops": 2 * c["rows"] * V * H}
    if k == "attn_decode":
        B, n = c["B"], c["ctx"]
        return {"bytes": B * (_kv_bytes(n + 1) + 2 * (NQKV + QD)), "flops": 4 * B * HQ * D * (n + 1)}
    if k.startswith("attn"):
        B, T, b = c["B"], c["T"], c["base"]
        keys = T * b + (T * (T + 1) // 2 if k == "attn_causal" else 4 * T)    # visible (query, key) pairs
        return {"bytes": B * (_kv_bytes(b + T) + 2 * T * (NQKV + QD)), "flops": 4 * B * HQ * D * keys}
    L, B = c["layers"], c["B"]
    if k == "decode":
        n = c["ctx"]
        return {"bytes": 2 * L * LAYER_W + 2 * V * H + L * B * _kv_bytes(n + 1) + 4 * B * V,
                "flops": 2 * B * (L * LAYER_W + V * H) + 4 * L * B * HQ * D * (n + 1)}
    T = c["T"]
    return {"bytes": 2 * L * LAYER_W + 2 * V * H + L * B * _kv_bytes(T) + 4 * B * V,
            "flops": 2 * B * (T * L * LAYER_W + V * H) + 4 * L * B * HQ * D * (T * (T + 1) // 2)}


# Relative errors: about four times what the path shows against `exact` on MI355X (norm 2.8e-3,
# proj 5.7e-3, head 2.3e-3, attention 4.2e-3).  A whole model's bf16 roundings travel through its
# layers: 1.9e-2 at 4 of them, 5.0e-2 at 36, about as their square root.
_REL = {"norm": 1.1e-2, "proj": 2.3e-2, "head": 9e-3, "attn_decode": 1.7e-2, "attn_causal": 1.7e-2,
        "attn_tree": 1.7e-2}


def tolerance(case):
    if case["kind"] in ("decode", "prefill"):
        return {"rel": 3.4e-2 * math.sqrt(case["layers"])}
    t = {"rel": _REL[case["kind"]]}
    if case["kind"] == "head":
        # a row whose two best logits share a bf16 value may go either way
        t["differ"] = max(0.1, 1.0 / case["rows"])
    return t


# ------------------------------------------------------------------ 64-bit references
def _norm64(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.to(F64)


def _rope64(x, pos):
    """Rotate [..., D] heads at positions pos (broadcast over the head dimension) with the bf16
    cos / sin values that the decoder's tables hold."""
    inv = 1.0 / (THETA ** (torch.arange(0, D, 2, dtype=torch.int64).float() / D))
    ang = pos.cpu().float()[..., None] * inv
    ang = torch.cat((ang, ang), -1)
    cos, sin = (t.to(BF16).to(F64).cuda() for t in (ang.cos(), ang.sin()))
    half = torch.cat((-x[..., D // 2:], x[..., :D // 2]), -1)
    return x * cos + half * sin


def _mlp64(x, s, l=None):
    w = (lambda n: s[n]) if l is None else (lambda n: getattr(s, n)[l])
    gu = _norm64(x, w("ln2")) @ w("w_gu").to(F64).t()
    act = torch.nn.functional.silu(gu[:, :I]) * gu[:, I:]
    return act, x + act @ w("w_down").to(F64).t()


def _qkv_heads64(qkv, qn, kn, pos):
    """q [B, T, HQ, D], k and v [B, T, HKV, D] from packed rows [B, T, NQKV]; pos [B, T]."""
    B, T, _ = qkv.shape
    x = qkv.reshape(B, T, HQ + 2 * HKV, D)
    p = pos[:, :, None].expand(B, T, 1)
    return (_rope64(_norm64(x[:, :, :HQ], qn), p), _rope64(_norm64(x[:, :, HQ:HQ + HKV], kn), p),
            x[:, :, HQ + HKV:])


def _attend64(q, k, v, mask):
    """q [T, HQ, D] against k, v [n, HKV, D]; mask [T, n] of visible keys."""
    T, out, g = q.shape[0], torch.empty_like(q), HQ // HKV
    step = max(1, (1 << 26) // k.shape[0])
    for h in range(HQ):
        for t in range(0, T, step):
            sc = q[t:t + step, h] @ k[:, h // g].t() / math.sqrt(D)
            sc.masked_fill_(~mask[t:t + step], -math.inf)
            out[t:t + step, h] = torch.softmax(sc, -1) @ v[:, h // g]
    return out


def _decode_attn64(q, k, v, k_cache, v_cache, n):
    """One new token per sequence: q [B, HQ, D], k and v [B, HKV, D], caches [B, HKV, cap, D]
    holding n earlier tokens."""
    outs = []
    for b in range(q.shape[0]):
        kk = torch.cat((k_cache[b, :, :n].to(F64), k[b][:, None]), 1)
        vv = torch.cat((v_cache[b, :, :n].to(F64), v[b][:, None]), 1)
        p = torch.softmax(q[b].reshape(HKV, HQ // HKV, D) @ kk.transpose(1, 2) / math.sqrt(D), -1)
        outs.append((p @ vv).reshape(HQ, D))
    return torch.stack(outs)


def _visible(c, anc, b):
    """[T, base + T] keys that each token of sequence b sees."""
    T, base = c["T"], c.get("base", 0)
    if anc is None:
        blk = torch.ones((T, T), dtype=torch.bool, device="cuda").tril()
    else:
        blk = (anc[b][:, None] >> torch.arange(T, device="cuda")[None]) & 1 == 1
    return torch.cat((torch.ones((T, base), dtype=torch.bool, device="cuda"), blk), 1)


def exact(case, seed):
    c, k, s = case, case["kind"], prepare(case, seed)
    if k == "norm":
        r = s["res"].to(F64)
        if not c["add"]:
            return {"y": _norm64(r, s["w"])}
        r = r + s["x"].to(F64)
        return {"res": r, "y": _norm64(r, s["w"])}
    if k == "proj":
        x = s["x"].to(F64)
        qkv = _norm64(x, s["ln1"]) @ s["w_qkv"].to(F64).t()
        x1 = x + s["attn"].to(F64) @ s["w_o"].to(F64).t()
        act, x2 = _mlp64(x1, s)
        return {"qkv": qkv, "x1": x1, "act": act, "x2": x2}
    if k == "head":
        return {"logits": _norm64(s["x"].to(F64), s["norm"]) @ s["w"].to(F64).t(), "tok": None}
    if k == "attn_decode":
        B, n = c["B"], c["ctx"]
        pos = torch.full((B, 1), n, dtype=torch.int64)
        q, kk, vv = _qkv_heads64(s["qkv"].to(F64).view(B, 1, NQKV), s["qn"], s["kn"], pos)
        return {"out": _decode_attn64(q[:, 0], kk[:, 0], vv[:, 0], s["k"], s["v"], n),
                "k": kk[:, 0], "v": vv[:, 0]}
    if k.startswith("attn"):
        B, T, base = c["B"], c["T"], c["base"]
        off = torch.arange(T, device="cuda").expand(B, T) if s["depth"] is None else s["depth"]
        q, kk, vv = _qkv_heads64(s["qkv"].to(F64).view(B, T, NQKV), s["qn"], s["kn"], base + off)
        out = torch.empty((B, T, HQ, D), dtype=F64, device="cuda")
        for b in range(B):
            kf = torch.cat((s["k"][b, :, :base].to(F64).transpose(0, 1), kk[b]), 0)
            vf = torch.cat((s["v"][b, :, :base].to(F64).transpose(0, 1), vv[b]), 0)
            out[b] = _attend64(q[b], kf, vf, _visible(c, s["anc"], b))
        return {"out": out, "k": kk.transpose(1, 2), "v": vv.transpose(1, 2)}
    m, B = s["model"], c["B"]
    T = 1 if k == "decode" else c["T"]
    x = m.embed[s["ids"].reshape(-1)].to(F64)
    pos = (torch.full((B, 1), c["ctx"], dtype=torch.int64) if k == "decode"
           else torch.arange(T).expand(B, T))
    ks, vs = [], []
    for l in range(c["layers"]):
        qkv = _norm64(x, m.ln1[l]) @ m.w_qkv[l].to(F64).t()
        q, kk, vv = _qkv_heads64(qkv.view(B, T, NQKV), m.q_norm[l], m.k_norm[l], pos)
        if k == "decode":
            a = _decode_attn64(q[:, 0], kk[:, 0], vv[:, 0], s["kv"].k[l], s["kv"].v[l], c["ctx"])
        else:
            a = torch.stack([_attend64(q[b], kk[b], vv[b], _visible(c, None, b)) for b in range(B)])
        x = x + a.reshape(B * T, QD) @ m.w_o[l].to(F64).t()
        x = _mlp64(x, m, l)[1]
        ks.append(kk.transpose(1, 2))
        vs.append(vv.transpose(1, 2))
    logits = _norm64(x.view(B, T, H)[:, T - 1], m.final_norm) @ m.lm_head.to(F64).t()
    return {"logits": logits, "k": torch.stack(ks), "v": torch.stack(vs)}
