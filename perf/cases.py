"""The work this package does for its users, as cases that can be timed and checked.

Every case is one of five kinds, each through public entry points:

- ``attention``: one ``DecodeAttention`` call (the op alone, as a serving loop with
  its own projections calls it);
- ``layers``: a decode step through consecutive decoder layers (``build_decode_gemvs``
  and ``decode_layer``), captured in a graph by the caller and replayed per token;
- ``prefill``: the prompt forward (``prefill.prefill``) into a fresh KV cache;
- ``generate``: whole ``Engine.generate`` calls on a shape the engine has served
  before, prompt and new tokens;
- ``verify``: one ``Engine.verify_step`` of speculative decoding.

The model is the Qwen3-4B architecture at fewer layers (every layer has its own
weights, more than the last-level cache holds). A trained model is confident in most of
its tokens; random weights are not, and a rounding would then change the text. So
``generate`` and ``verify`` run with an LM head that favours one successor for each
token, over layers with random weights.
"""

import math
import time

import torch

from kernel_optim_amd.engine import Engine, attn_units_per_seq, build_decode_gemvs, decode_layer
from kernel_optim_amd.kernels.fused import DecodeAttention, rope_rows
from kernel_optim_amd.model import Qwen3Config, random_weights
from kernel_optim_amd.prefill import prefill

DEV = "cuda:0"
BF16 = torch.bfloat16
F64 = torch.float64
NQ, NKV, D = 32, 8, 128
TUNE_S = 30.0  # a program's budget for tuning the projections at setup


def listed():
    return [
        # One sequence and a short context: the smallest attention call, made eagerly, where
        # the launches and the call itself are what a caller waits for.
        dict(name="attn_b1_512", kind="attention", B=1, T=1, ctx=512, ragged=False, fused=False),
        # A full batch with long contexts: one split-K attention call at memory speed.
        dict(name="attn_b16_8192", kind="attention", B=16, T=1, ctx=8192, ragged=False,
             fused=False),
        # A serving batch in which every sequence has its own length, in a cache padded to the
        # longest one.
        dict(name="attn_ragged_b64", kind="attention", B=64, T=1, ctx=16384, ragged=True,
             fused=False),
        # One user's decode step: four launches per layer, all weights read for one row.
        dict(name="layers_b1_1024", kind="layers", B=1, ctx=1024, layers=4, ragged=False),
        # A few users with medium prompts (batch 4, 2048 tokens).
        dict(name="layers_b4_2048", kind="layers", B=4, ctx=2048, layers=4, ragged=False),
        # The batch that the decode benchmark runs beside batch 1.
        dict(name="layers_b16_1024", kind="layers", B=16, ctx=1024, layers=4, ragged=False),
        # The largest batch whose decode graph is made of the fused projections by default.
        dict(name="layers_b32_1024", kind="layers", B=32, ctx=1024, layers=4, ragged=False),
        # A short prompt of one user: the time to the first token, bound by launches.
        dict(name="prefill_b1_512", kind="prefill", B=1, S=512, layers=4),
        # Four prompts of 2048 tokens in one forward: the largest prompt work.
        dict(name="prefill_b4_2048", kind="prefill", B=4, S=2048, layers=4),
        # A whole answer for one user, prompt and 32 tokens.
        dict(name="generate_b1_512", kind="generate", B=1, S=512, N=32, layers=8),
        # Short answers for a large batch (the decode step for more than 32 sequences).
        dict(name="generate_b64_128", kind="generate", B=64, S=128, N=16, layers=4),
        # Speculative decoding's check of six drafted tokens (seven rows of one sequence).
        dict(name="verify_b1_1024", kind="verify", B=1, S=1024, layers=4),
    ]


def _log_int(rng, lo, hi):
    """A whole number from lo to hi, even over its logarithm."""
    return max(lo, min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    kind = rng.choice(["attention", "attention", "layers", "layers", "layers", "prefill",
                       "generate", "generate", "verify"])
    if kind == "attention":
        T = rng.choice([1, 1, 1, 2, 4, 5, 8])
        B = _log_int(rng, 1, 128 if T == 1 else 16)
        # at most the keys of the ragged batch
        ctx = _log_int(rng, 16, min(32768, 64 * 8192 // B))
        return dict(kind=kind, B=B, T=T, ctx=ctx, ragged=rng.random() < 0.4,
                    fused=rng.random() < 0.4)
    if kind == "layers":
        B = _log_int(rng, 1, 64)
        ctx = _log_int(rng, 33, min(8192, 32 * 1024 // B))
        return dict(kind=kind, B=B, ctx=ctx, layers=rng.choice([2, 3, 4]),
                    ragged=rng.random() < 0.3)
    if kind == "prefill":
        B = _log_int(rng, 1, 16)
        return dict(kind=kind, B=B, S=_log_int(rng, 7, min(4096, 8192 // B)),
                    layers=rng.choice([2, 3, 4]))
    if kind == "generate":
        B = _log_int(rng, 1, 96)
        return dict(kind=kind, B=B, S=_log_int(rng, 5, 8192 // B if B > 8 else 1024),
                    N=rng.randint(4, 16), layers=rng.choice([2, 3, 4]))
    B = rng.choice([1, 1, 2, 3, 4])
    return dict(kind=kind, B=B, S=_log_int(rng, 9, 2048 // B), layers=rng.choice([2, 3, 4]))


# ---------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=BF16)


def _tables(n, theta=1.0e6):
    """RoPE cos/sin rows [n, D] in bf16."""
    inv = 1.0 / (theta ** (torch.arange(0, D, 2, dtype=torch.float) / D))
    f = torch.outer(torch.arange(n, dtype=torch.float), inv).to(DEV)
    e = torch.cat((f, f), -1)
    return e.cos().to(BF16), e.sin().to(BF16)


def _spread(g, B, lo, hi):
    """B whole numbers from lo to hi, the first one hi."""
    v = torch.randint(lo, hi + 1, (B,), generator=g, device=DEV, dtype=torch.int32)
    v[0] = hi
    return v


def _attention_inputs(c, seed):
    g = _gen(seed)
    B, T, ctx = c["B"], c["T"], c["ctx"]
    cap = -(-max(ctx, T) // 16) * 16
    ctx = max(ctx, T)
    lens = (_spread(g, B, max(T, min(128, ctx)), ctx) if c["ragged"]
            else torch.full((B,), ctx, dtype=torch.int32, device=DEV))
    return dict(q=_randn(g, B * T, NQ * D), k=_randn(g, B, NKV, cap, D),
                v=_randn(g, B, NKV, cap, D), lens=lens, cap=cap)


def _gains(w, g):
    """Norm gains near one, as a trained model has them."""
    for lw in w["layers"]:
        for name in ("w_in", "w_post", "q_norm", "k_norm"):
            lw[name] = (1.0 + 0.1 * _randn(g, lw[name].shape[0]).float()).to(BF16)
    w["final_norm"] = (1.0 + 0.1 * _randn(g, w["final_norm"].shape[0]).float()).to(BF16)
    return w


def _layers_inputs(c, seed):
    """Hidden rows, weights and a filled KV cache; sequence b's new token is at pos[b]."""
    g = _gen(seed)
    B, ctx, L = c["B"], c["ctx"], c["layers"]
    cfg = Qwen3Config(layers=L, vocab=1024)
    w = _gains(random_weights(cfg, seed=seed, device=DEV), g)
    cap = -(-(ctx + 1) // 16) * 16
    pos = (_spread(g, B, ctx // 2, ctx) if c["ragged"]
           else torch.full((B,), ctx, dtype=torch.int32, device=DEV))
    return dict(cfg=cfg, w=w, cap=cap, pos=pos, x=_randn(g, B, cfg.hidden),
                k=_randn(g, L, B, NKV, cap, D), v=_randn(g, L, B, NKV, cap, D))


def _prefill_inputs(c, seed):
    g = _gen(seed)
    cfg = Qwen3Config(layers=c["layers"])
    w = _gains(random_weights(cfg, seed=seed, device=DEV), g)
    prompt = torch.randint(0, cfg.vocab, (c["B"], c["S"]), generator=g, device=DEV)
    return dict(cfg=cfg, w=w, prompt=prompt)


def _chat_inputs(c, seed):
    """A model whose LM head favours one successor of every token, prompts for it, and the
    rows a verify step checks."""
    g = _gen(seed)
    cfg = Qwen3Config(layers=c["layers"], tied=False)
    w = random_weights(Qwen3Config(layers=c["layers"]), seed=seed, device=DEV)
    w = _gains(w, g)
    w["embed"] = w["embed"] * 50                   # rows of unit scale
    order = torch.randperm(cfg.vocab, generator=g, device=DEV)
    w["lm_head"] = torch.empty_like(w["embed"])
    w["lm_head"][order] = (w["embed"].float() * 0.02).to(BF16)   # token t is followed by order[t]
    prompt = torch.randint(0, cfg.vocab, (c["B"], c["S"]), generator=g, device=DEV)
    rows = torch.randint(0, cfg.vocab, (c["B"], 7), generator=g, device=DEV)
    return dict(cfg=cfg, w=w, prompt=prompt, rows=rows)


# ------------------------------------------------------------------- what a program keeps
def prepare(case, seed):
    c = case
    if c["kind"] == "attention":
        s = _attention_inputs(c, seed)
        s["op"] = DecodeAttention(c["B"], c["T"], s["cap"], NQ, NKV, D, DEV,
                                  fused_combine=c["fused"])
        s["out"] = torch.zeros_like(s["q"])
    elif c["kind"] == "layers":
        s = _prepare_layers(c, seed)
    elif c["kind"] == "prefill":
        s = _prefill_inputs(c, seed)
        cfg = s["cfg"]
        cap = -(-(c["S"] + 32) // 16) * 16
        s["k"] = torch.zeros(cfg.layers, c["B"], NKV, cap, D, dtype=BF16, device=DEV)
        s["v"] = torch.zeros_like(s["k"])
        s["cos"], s["sin"] = _tables(cap)
    else:
        s = _chat_inputs(c, seed)
        s["eng"] = Engine.from_weights(s["cfg"], s["w"], keep_logits=True,
                                       spec=c["kind"] == "verify")
        prompt = s["prompt"].tolist()
        if c["kind"] == "generate":
            # the program has served this shape before (buffers, tuning, graphs)
            list(s["eng"].generate(s["prompt"].flip(1).tolist(), c["N"]))
            s["ids"] = prompt
        else:
            list(s["eng"].generate(prompt, 4))     # the cache holds the prompt
            T = s["eng"].T
            s["rows"] = s["rows"][:, :T].cpu()
            s["at"] = torch.full((c["B"],), c["S"], dtype=torch.int32)
    s["case"] = dict(c)
    return s


def _prepare_layers(c, seed):
    s = _layers_inputs(c, seed)
    cfg, B, L = s["cfg"], c["B"], c["layers"]
    lws = s["w"]["layers"]
    raw = {n: [lw[n] for lw in lws] for n in ("qkv", "o", "gu", "down")}
    gv, W = build_decode_gemvs(cfg, B, raw, time.monotonic() + TUNE_S)
    attn = DecodeAttention(B, 1, s["cap"], NQ, NKV, D, DEV, fused_combine=True,
                           units_per_seq=attn_units_per_seq(B, NKV))
    s["cos"], s["sin"] = _tables(s["cap"], cfg.theta)
    s["h"] = torch.zeros(B, cfg.hidden, dtype=BF16, device=DEV)
    buf = dict(qkv=torch.zeros(B, cfg.nqkv, dtype=BF16, device=DEV),
               att=torch.zeros(B, NQ * D, dtype=BF16, device=DEV),
               act=torch.zeros(B, cfg.inter, dtype=BF16, device=DEV),
               rope=torch.zeros(B, 2, D, dtype=BF16, device=DEV))
    fuse_o = attn.oproj_fusable()

    def step():
        s["h"].copy_(s["x"])
        rope_rows(s["pos"], s["cos"], s["sin"], buf["rope"])
        for i in range(L):
            decode_layer(gv, W, i, lws[i], attn, s["h"], buf["qkv"], buf["att"], buf["act"],
                         s["k"][i], s["v"][i], s["cos"], s["sin"], s["pos"], buf["rope"],
                         cfg.eps, fuse_o)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    s["graph"] = torch.cuda.CUDAGraph()
    with torch.cuda.graph(s["graph"]):
        step()
    s["keep"] = (gv, W, attn, buf)
    return s


# ------------------------------------------------------------------------------ one pass
def run(state):
    s, c = state, state["case"]
    if c["kind"] == "attention":
        s["op"].with_lengths(s["q"], s["k"], s["v"], s["lens"], s["out"])
        return s["out"]
    if c["kind"] == "layers":
        s["graph"].replay()
        return dict(h=s["h"], k=s["k"], v=s["v"])
    if c["kind"] == "prefill":
        ids, logits = prefill(s["cfg"], s["w"], s["prompt"], s["k"], s["v"], s["cos"], s["sin"])
        return dict(ids=ids, logits=logits, k=s["k"], v=s["v"])
    if c["kind"] == "generate":
        toks = list(s["eng"].generate(s["ids"], c["N"]))
        return dict(tokens=torch.tensor(toks), logits=s["eng"].logits)
    ids, logits = s["eng"].verify_step(s["rows"], s["at"])
    return dict(ids=ids, logits=logits)


# --------------------------------------------------------------- what a pass cannot do without
def work(case):
    c = case
    if c["kind"] == "attention":
        B, T, ctx = c["B"], c["T"], max(c["ctx"], c["T"])
        keys = B * ctx if not c["ragged"] else int(
            (B - 1) * (max(T, min(128, ctx)) + ctx) / 2 + ctx)   # expected
        return dict(bytes=keys * NKV * D * 4 + 4 * B * T * NQ * D, flops=4.0 * keys * T * NQ * D)
    cfg = Qwen3Config(layers=c["layers"])
    B, L = c["B"], c["layers"]
    params = cfg.layer_bytes() / 2
    kv = NKV * D * 4                  # K and V bytes of one key of one layer
    head = cfg.vocab * cfg.hidden

    def decode(rows, keys, lm):       # one step of `rows` rows over `keys` cached keys in all
        return (L * (2 * params + keys * kv + rows * kv) + (2 * head + 2 * rows * cfg.vocab) * lm
                + 4 * rows * cfg.hidden,
                2.0 * rows * (L * params + head * lm) + 4.0 * L * keys * NQ * D)

    def prompt(S):
        return (L * (2 * params + B * S * kv) + 2 * head + 2 * B * S * cfg.hidden,
                2.0 * B * S * L * params + 2.0 * L * B * S * S * NQ * D + 2.0 * B * head)

    if c["kind"] == "layers":
        keys = B * c["ctx"] if not c["ragged"] else int((B - 1) * 0.75 * c["ctx"] + c["ctx"])
        b, f = decode(B, keys, 0)
    elif c["kind"] == "prefill":
        b, f = prompt(c["S"])
    elif c["kind"] == "generate":
        b, f = prompt(c["S"])
        for j in range(1, c["N"]):
            db, df = decode(B, B * (c["S"] + j - 1), 1)
            b, f = b + db, f + df
    else:
        b, f = decode(7 * B, B * c["S"], 1)
        f += 6 * 4.0 * L * B * c["S"] * NQ * D
    return dict(bytes=b, flops=f)


def tolerance(case):
    """About twice what two correct bf16 implementations can differ by, each being off the
    64-bit result by (2-norm, measured) 0.0023 for one attention call, 0.011 for the hidden
    rows after four layers, 0.011-0.020 for the logits after a prompt or a whole answer."""
    k = case["kind"]
    if k == "attention":
        return {"rel": 1e-2}
    if k == "layers":
        return {"rel": 2e-2}
    return {"rel": 2.5e-2, "max": 0.5, "differ": 0.002}


# ----------------------------------------------------------------- the same in 64-bit torch
def _norm64(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.to(F64)


def _rope64(x, cos, sin):
    """x [..., D], cos/sin broadcast against it."""
    h = D // 2
    rot = torch.cat((-x[..., h:], x[..., :h]), -1)
    return x * cos.to(F64) + rot * sin.to(F64)


def _attend64(q, k, v, last):
    """q [T, NQ, D], k/v [NKV, n, D] of one sequence; query t sees keys 0..last[t]."""
    T = q.shape[0]
    q = q.view(T, NKV, NQ // NKV, D).permute(1, 2, 0, 3).reshape(NKV, -1, D)
    s = torch.bmm(q, k.to(F64).transpose(1, 2).contiguous()) * D ** -0.5
    hide = torch.arange(k.shape[1], device=DEV)[None, :] > last[:, None]
    s = s.view(NKV, NQ // NKV, T, -1).masked_fill_(hide[None, None], float("-inf"))
    p = torch.softmax(s, -1).view(NKV, -1, k.shape[1])
    o = torch.bmm(p, v.to(F64).contiguous())
    return o.view(NKV, NQ // NKV, T, D).permute(2, 0, 1, 3).reshape(T, NQ * D)


def _layer64(lw, eps, x, cos, sin, k, v, at):
    """One layer over x [B, T, H]; sequence b's rows go to slots at[b] .. at[b] + T - 1 of
    k/v [B, NKV, cap, D] (64-bit)."""
    B, T, H = x.shape
    h = _norm64(x, lw["w_in"], eps) @ lw["qkv"].to(F64).t()
    q, kn, vn = h.split((NQ * D, NKV * D, NKV * D), -1)
    q = _norm64(q.view(B, T, NQ, D), lw["q_norm"], eps)
    kn = _norm64(kn.view(B, T, NKV, D), lw["k_norm"], eps)
    o = torch.empty(B, T, NQ * D, dtype=F64, device=DEV)
    for b in range(B):
        p0 = at[b]
        cs, sn = cos[p0:p0 + T, None], sin[p0:p0 + T, None]
        k[b, :, p0:p0 + T] = _rope64(kn[b], cs, sn).transpose(0, 1)
        v[b, :, p0:p0 + T] = vn[b].view(T, NKV, D).transpose(0, 1)
        last = torch.arange(p0, p0 + T, device=DEV)
        o[b] = _attend64(_rope64(q[b], cs, sn), k[b, :, :p0 + T], v[b, :, :p0 + T], last)
    x = x + o @ lw["o"].to(F64).t()
    gu = _norm64(x, lw["w_post"], eps) @ lw["gu"].to(F64).t()
    g, u = gu.chunk(2, -1)
    return x + (torch.nn.functional.silu(g) * u) @ lw["down"].to(F64).t()


def _rows64(s, tokens, k, v, cos, sin, at, last_only):
    """Logits [B, V] of the last row, or [B, T, V] of every row."""
    w, eps = s["w"], s["cfg"].eps
    x = w["embed"][tokens].to(F64)
    for i, lw in enumerate(w["layers"]):
        x = _layer64(lw, eps, x, cos, sin, k[i], v[i], at)
    x = _norm64(x[:, -1:] if last_only else x, w["final_norm"], eps)
    y = torch.cat([x @ part.to(F64).t() for part in w["lm_head"].split(32768)], -1)
    return y[:, 0] if last_only else y


def exact(case, seed):
    c = case
    with torch.no_grad():
        if c["kind"] == "attention":
            s = _attention_inputs(c, seed)
            T, out = c["T"], []
            for b in range(c["B"]):
                n = int(s["lens"][b])
                q = s["q"][b * T:(b + 1) * T].to(F64).view(T, NQ, D)
                out.append(_attend64(q, s["k"][b, :, :n], s["v"][b, :, :n],
                                     torch.arange(n - T, n, device=DEV)))
            return torch.cat(out)
        if c["kind"] == "layers":
            s = _layers_inputs(c, seed)
            cos, sin = _tables(s["cap"], s["cfg"].theta)
            x, at, ks, vs = s["x"].to(F64)[:, None], s["pos"].tolist(), [], []
            for i, lw in enumerate(s["w"]["layers"]):
                ks.append(s["k"][i].to(F64))
                vs.append(s["v"][i].to(F64))
                x = _layer64(lw, s["cfg"].eps, x, cos, sin, ks[i], vs[i], at)
            return dict(h=x[:, 0], k=torch.stack(ks), v=torch.stack(vs))
        s = _prefill_inputs(c, seed) if c["kind"] == "prefill" else _chat_inputs(c, seed)
        B, S, L = c["B"], c["S"], c["layers"]
        cap = -(-(S + 32) // 16) * 16
        k = torch.zeros(L, B, NKV, cap, D, dtype=F64, device=DEV)
        v = torch.zeros_like(k)
        cos, sin = _tables(cap)
        y = _rows64(s, s["prompt"], k, v, cos, sin, [0] * B, True)
        if c["kind"] == "prefill":
            return dict(ids=None, logits=y, k=k, v=v)
        if c["kind"] == "generate":
            for j in range(1, c["N"]):
                y = _rows64(s, y.argmax(-1)[:, None], k, v, cos, sin, [S + j - 1] * B, True)
            return dict(tokens=None, logits=y)
        y = _rows64(s, s["rows"], k, v, cos, sin, [S] * B, False)
        return dict(ids=None, logits=y.view(B * s["rows"].shape[1], -1))
