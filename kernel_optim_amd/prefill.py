"""Prompt forward (prefill) on PyTorch-ROCm GEMMs and SDPA, writing the static KV cache.

The reference's prefill (engine/engine.py:343-386) exists to produce exactly
the K/V and last-position logits of Transformers' own Qwen3 forward: a prefill
that drifts a little per layer can flip which key a sharp attention row picks
and cost whole logits downstream (engine.py:344-351). So this one has
the bits of the same torch operations, in the same order and with the same shapes, as
Transformers' modules (modeling_qwen3.py Qwen3RMSNorm, Qwen3Attention,
Qwen3MLP, Qwen3DecoderLayer):
- separate q / k / v and gate / up GEMMs (row slices of the engine's
  concatenated weights are the same matrices, so the same GEMM shapes);
- RMSNorm, per-head q/k RMSNorm, RoPE, SiLU-multiply and the residual adds with the
  modules' bits (fp32 statistics, bf16 rounding before the gain): one HIP row kernel
  each (csrc/prefill_ops.hip) where those add in torch's order, else the modules'
  torch operations;
- attention = torch's scaled_dot_product_attention, causal, on the modules'
  [B, heads, S, d] layouts, with ``enable_gqa`` only where a probe shows it
  bit-equal to repeated KV heads on this torch (engine.py:96-116), else on
  repeated KV heads; restricted to the fused SDPA kernels (a flash or
  memory-efficient backend), never the bf16 batched-matmul math path;
- the final RMSNorm and the LM head on the last position only (engine.py:383-385).
The prompt's K (normed + roped) and V go to cache slots 0..S-1.
"""

import torch
import torch.autograd.forward_ad as forward_ad
import torch.nn.functional as F
from torch.utils._device import DeviceContext

from .kernels.fused import prefill_norm, prefill_qkv, silu_mul2

BF16 = torch.bfloat16
F32 = torch.float32

_GQA_EXACT = {}


def _sdpa_kernels():
    """Context restricting SDPA to its fused GPU kernels."""
    from torch.nn.attention import SDPBackend, sdpa_kernel
    return sdpa_kernel([SDPBackend.FLASH_ATTENTION, SDPBackend.EFFICIENT_ATTENTION])


def gqa_exact(device):
    """Whether SDPA with enable_gqa (the KV heads read in place) returns the same
    bits as SDPA on KV heads repeated 4x on causal prefill-shaped inputs, on this
    device and torch (the reference's probe, engine.py:96-116). Cached per device."""
    key = str(device)
    if key not in _GQA_EXACT:
        ok = True
        try:
            g = torch.Generator(device=device).manual_seed(0)
            with _sdpa_kernels():
                for B, S in ((1, 300), (4, 1024)):
                    q = torch.randn(B, 32, S, 128, device=device, dtype=BF16, generator=g)
                    k = torch.randn(B, 8, S, 128, device=device, dtype=BF16, generator=g) * 4
                    v = torch.randn(B, 8, S, 128, device=device, dtype=BF16, generator=g)
                    ref = F.scaled_dot_product_attention(q, k.repeat_interleave(4, 1),
                                                         v.repeat_interleave(4, 1), is_causal=True,
                                                         scale=128 ** -0.5)
                    got = F.scaled_dot_product_attention(q, k, v, is_causal=True, scale=128 ** -0.5,
                                                         enable_gqa=True)
                    ok = ok and torch.equal(ref, got)
        except RuntimeError:
            ok = False
        _GQA_EXACT[key] = ok
    return _GQA_EXACT[key]


def rmsnorm(x, w, eps):
    """Qwen3RMSNorm.forward."""
    xf = x.to(F32)
    variance = xf.pow(2).mean(-1, keepdim=True)
    xf = xf * torch.rsqrt(variance + eps)
    return w * xf.to(x.dtype)


def rotate_half(x):
    h = x.shape[-1] // 2
    return torch.cat((-x[..., h:], x[..., :h]), dim=-1)


def causal_attention(q, k, v, scale, exact_gqa):
    """q [B, nq, S, d], k/v [B, nkv, S, d] bf16 -> [B, nq, S, d] bf16, causal, by
    torch SDPA on its fused kernels."""
    rep = q.shape[1] // k.shape[1]
    with _sdpa_kernels():
        if exact_gqa:
            return F.scaled_dot_product_attention(q, k, v, attn_mask=None, dropout_p=0.0,
                                                  scale=scale, is_causal=True, enable_gqa=True)
        kr = k[:, :, None].expand(-1, -1, rep, -1, -1).reshape(k.shape[0], -1, *k.shape[2:])
        vr = v[:, :, None].expand(-1, -1, rep, -1, -1).reshape(v.shape[0], -1, *v.shape[2:])
        return F.scaled_dot_product_attention(q, kr, vr, attn_mask=None, dropout_p=0.0,
                                              scale=scale, is_causal=True)


_ROW_SUMS = {}


def _row_sums_exact(device, n):
    """Whether the row kernels add the squares of a row of n values, and of a head, in
    the order of torch's mean on this device and torch: both are compared with the torch
    operations bit for bit on one sample. Cached per device and row width; a stream
    that is being captured is not the place for the comparison (not cached then)."""
    key = (str(device), n)
    if key not in _ROW_SUMS:
        if torch.cuda.is_current_stream_capturing():
            return False
        g = torch.Generator(device=device).manual_seed(0)
        x = torch.randn(64, n, device=device, generator=g).to(BF16)
        w = torch.randn(n, device=device, generator=g).to(BF16)
        got = torch.empty_like(x)
        prefill_norm(x, None, w, got, 1e-6)
        q, k, v = (torch.randn(16, 4 * 128, device=device, generator=g).to(BF16)
                   for _ in range(3))
        cos, sin = (torch.randn(16, 128, device=device, generator=g).to(BF16) for _ in range(2))
        hw = w[:128].contiguous()
        kc, vc = (torch.zeros(1, 4, 16, 128, dtype=BF16, device=device) for _ in range(2))
        want = rmsnorm(k.view(1, 16, 4, 128), hw, 1e-6).transpose(1, 2)
        want = want * cos + rotate_half(want) * sin
        prefill_qkv(q, k, v, hw, hw, cos, sin, kc, vc, 1e-6)
        _ROW_SUMS[key] = torch.equal(got, rmsnorm(x, w, 1e-6)) and torch.equal(kc, want)
    return _ROW_SUMS[key]


def _observed():
    """Whether something records, rewrites or differentiates the torch operations of this
    call: a trace (jit, dynamo, make_fx), a dispatch or function mode, a functorch transform
    (vmap, functionalize, jvp) or a forward-mode level. The row kernels work by address and
    would be missing from what it sees. A default device (DeviceContext) rewrites nothing here."""
    return (torch.compiler.is_compiling() or torch.jit.is_tracing()
            or torch._C._len_torch_dispatch_stack() > 0
            or torch._ops._len_torch_dispatch_stack_pre_dispatch() > 0
            or any(not isinstance(m, DeviceContext)
                   for m in torch.overrides._get_current_function_mode_stack())
            or torch._C._functorch.peek_interpreter_stack() is not None
            or forward_ad._current_level >= 0)


def _on_gpu(dev):
    return dev.type == "cuda" and dev.index in (None, torch.cuda.current_device())


def _is_plain(t):
    """No subclass, whose operations may be its own: a layer with one, and the layers that
    read what it returns, keep the torch operations."""
    return type(t) in (torch.Tensor, torch.nn.Parameter)


def _plain(t, dev, *shape):
    return (_is_plain(t) and t.dtype == BF16 and t.device == dev
            and tuple(t.shape) == shape and t.is_contiguous() and t.data_ptr() % 16 == 0)


def _rows_served(cfg, embed, B, S, k_cache, v_cache, cos, sin):
    """Whether the row kernels serve this call: made eagerly (_observed), with bf16 tensors
    on the current GPU in the engine's layouts, heads of 128, and rows whose mean of squares
    they add in torch's order (which changes below 8 rows, below 256 values and past 8064)."""
    if _observed():
        return False
    H, d, dev = cfg.hidden, cfg.head_dim, k_cache.device

    def cache(t):
        return (_is_plain(t) and t.dtype == BF16 and t.device == dev and t.dim() == 5
                and t.shape[1] == B
                and t.shape[2] == cfg.nkv and t.shape[3] >= S and t.shape[4] == d
                and t.stride(4) == 1 and t.stride(3) == d and t.data_ptr() % 16 == 0
                and all(t.stride(i) % 8 == 0 for i in range(3)))

    return (_on_gpu(dev) and B * S >= 8 and 256 <= H <= 8064 and H % 8 == 0 and d == 128
            and cfg.inter % 8 == 0
            and cache(k_cache) and cache(v_cache) and k_cache.stride() == v_cache.stride()
            and _plain(cos, dev, cos.shape[0], d) and _plain(sin, dev, sin.shape[0], d)
            and min(cos.shape[0], sin.shape[0]) >= S and _is_plain(embed) and embed.dtype == BF16
            and not torch.is_autocast_enabled() and _row_sums_exact(dev, H))


def _layer_served(cfg, lw, x):
    H, d, dev = cfg.hidden, cfg.head_dim, x.device
    return (_plain(x, dev, *x.shape) and _plain(lw["w_in"], dev, H) and _plain(lw["w_post"], dev, H)
            and _plain(lw["q_norm"], dev, d) and _plain(lw["k_norm"], dev, d)
            and all(_is_plain(lw[n]) and lw[n].dtype == BF16 for n in ("qkv", "o", "gu", "down")))


def _layer_rows(cfg, lw, x, delta, h, kc, vc, cos, sin, exact_gqa):
    """One layer with the row kernels between its GEMMs: the GEMMs and the SDPA call of
    _layer_torch, and its bits. x is the residual stream without the last layer's
    output ``delta``, updated in place; returns this layer's output, to be added to
    it; h is a buffer like x. SDPA reads the prompt's K/V from the cache."""
    B, S = x.shape[:2]
    nq, nkv, d, I, eps = cfg.nq, cfg.nkv, cfg.head_dim, cfg.inter, cfg.eps
    qkv, gu = lw["qkv"], lw["gu"]
    prefill_norm(x, delta, lw["w_in"], h, eps)
    q = F.linear(h, qkv[:nq * d])
    prefill_qkv(q, F.linear(h, qkv[nq * d:(nq + nkv) * d]), F.linear(h, qkv[(nq + nkv) * d:]),
                lw["q_norm"], lw["k_norm"], cos, sin, kc, vc, eps)
    o = causal_attention(q.view(B, S, nq, d).transpose(1, 2), kc[:, :, :S], vc[:, :, :S],
                         d ** -0.5, exact_gqa)
    delta = F.linear(o.transpose(1, 2).reshape(B, S, -1).contiguous(), lw["o"])
    prefill_norm(x, delta, lw["w_post"], h, eps)
    gate = F.linear(h, gu[:I])
    silu_mul2(gate, F.linear(h, gu[I:]), gate)
    return F.linear(gate, lw["down"])


def _layer_torch(cfg, lw, x, kc, vc, cos, sin, exact_gqa):
    """One layer as Transformers' modules write it."""
    B, S = x.shape[:2]
    nq, nkv, d, I, eps = cfg.nq, cfg.nkv, cfg.head_dim, cfg.inter, cfg.eps
    c = cos[:S][None, None]          # apply_rotary_pos_emb's unsqueeze(1)
    s_ = sin[:S][None, None]
    shape = (B, S, -1, d)
    residual = x
    h = rmsnorm(x, lw["w_in"], eps)
    qkv = lw["qkv"]
    q = rmsnorm(F.linear(h, qkv[:nq * d]).view(shape), lw["q_norm"], eps).transpose(1, 2)
    k = rmsnorm(F.linear(h, qkv[nq * d:(nq + nkv) * d]).view(shape), lw["k_norm"],
                eps).transpose(1, 2)
    v = F.linear(h, qkv[(nq + nkv) * d:]).view(shape).transpose(1, 2)
    q = (q * c) + (rotate_half(q) * s_)
    k = (k * c) + (rotate_half(k) * s_)
    kc[:, :, :S] = k
    vc[:, :, :S] = v
    o = causal_attention(q, k, v, d ** -0.5, exact_gqa)
    o = o.transpose(1, 2).reshape(B, S, -1).contiguous()
    x = residual + F.linear(o, lw["o"])
    residual = x
    h = rmsnorm(x, lw["w_post"], eps)
    gu = lw["gu"]
    return residual + F.linear(F.silu(F.linear(h, gu[:I])) * F.linear(h, gu[I:]), lw["down"])


@torch.no_grad()
def prefill(cfg, w, prompt, k_cache, v_cache, cos, sin):
    """prompt [B, S] int64 on the device; caches [L, B, nkv, cap, d]; cos/sin
    [>= S, d] bf16 (Qwen3RotaryEmbedding's rows for positions 0..S-1). Returns
    the greedy next ids [B] (int64) and the last-position logits [B, V] (bf16)."""
    B, S = prompt.shape
    exact_gqa = gqa_exact(prompt.device)
    x = F.embedding(prompt, w["embed"])
    rows = (_is_plain(prompt)
            and _rows_served(cfg, w["embed"], B, S, k_cache, v_cache, cos, sin))
    h = torch.empty_like(x) if rows else None
    delta = None   # the last layer's output where it is not yet in x
    for i, lw in enumerate(w["layers"]):
        if rows and _layer_served(cfg, lw, x):
            delta = _layer_rows(cfg, lw, x, delta, h, k_cache[i], v_cache[i], cos, sin, exact_gqa)
            continue
        if delta is not None:
            x, delta = x + delta, None
        x = _layer_torch(cfg, lw, x, k_cache[i], v_cache[i], cos, sin, exact_gqa)
    if delta is not None:
        x = x + delta
    xl = rmsnorm(x[:, -1:], w["final_norm"], cfg.eps)
    logits = F.linear(xl, w["lm_head"])[:, -1]
    return torch.argmax(logits, dim=-1), logits
