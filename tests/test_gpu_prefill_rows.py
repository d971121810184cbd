"""The prompt forward's row kernels against the torch operations they replace, bit for
bit (the bar is equality: prefill has to leave Transformers' bits)."""

import pytest
import torch
import torch.nn.functional as F

import kernel_optim_amd.prefill as P
from kernel_optim_amd.kernels.fused import prefill_norm, prefill_qkv, silu_mul2
from kernel_optim_amd.model import Qwen3Config, random_weights

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _randn(g, *shape):
    return torch.randn(*shape, device="cuda", generator=g).to(BF)


def _same(a, b):
    """Equal bits, or NaN in the same places."""
    return torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(), b.nan_to_num())


# one wavefront per workgroup up to 2048 rows, 4 above (with a part-filled last one);
# 10 quads per lane up to 2560 values, 32 above; the smallest and largest row
@pytest.mark.parametrize("rows,n", [(8, 2560), (77, 256), (2048, 2560), (2051, 2560), (30, 2564),
                                    (16, 8064), (300, 1000), (16384, 512)])
def test_prefill_norm(dev, rows, n):
    g = torch.Generator(device=dev).manual_seed(rows + n)
    x, d, w = _randn(g, rows, n), _randn(g, rows, n), _randn(g, n)
    x[1] *= 1e-3                       # eps matters
    x[2] = 0
    x[3, 5] = 3e38                     # the mean of squares overflows
    x[4, 7] = float("inf")
    x[5, 0] = float("nan")
    out = torch.empty_like(x)
    prefill_norm(x, None, w, out, 1e-6)
    assert _same(out, P.rmsnorm(x, w, 1e-6))
    y = x.clone()
    prefill_norm(y, d, w, out, 1e-6)
    assert _same(y, x + d) and _same(out, P.rmsnorm(x + d, w, 1e-6))


@pytest.mark.parametrize("B,S,nq,nkv,pad", [(1, 1, 32, 8, 0), (3, 37, 32, 8, 3), (2, 5, 4, 1, 1),
                                            (1, 300, 8, 2, 0), (4, 2048, 32, 8, 16)])
def test_prefill_qkv(dev, B, S, nq, nkv, pad):
    d = 128
    g = torch.Generator(device=dev).manual_seed(S + nq)
    q, k, v = (_randn(g, B, S, n * d) for n in (nq, nkv, nkv))
    qw, kw, cos, sin = (_randn(g, *s) for s in ((d,), (d,), (S + pad, d), (S + pad, d)))
    kc = _randn(g, 2, B, nkv, S + pad, d)
    vc = _randn(g, 2, B, nkv, S + pad, d)

    def roped(x, w):
        x = P.rmsnorm(x.view(B, S, -1, d), w, 1e-6).transpose(1, 2)
        return x * cos[:S] + P.rotate_half(x) * sin[:S]

    want_q, want_k, want_v = roped(q, qw), kc.clone(), vc.clone()
    want_k[1, :, :, :S] = roped(k, kw)
    want_v[1, :, :, :S] = v.view(B, S, nkv, d).transpose(1, 2)
    prefill_qkv(q, k, v, qw, kw, cos, sin, kc[1], vc[1], 1e-6)
    assert torch.equal(q.view(B, S, nq, d).transpose(1, 2), want_q)
    assert torch.equal(kc, want_k) and torch.equal(vc, want_v)   # and nothing else written


def test_silu_mul2_every_gate(dev):
    bits = torch.arange(65536, device=dev, dtype=torch.int32).to(torch.int16)
    gate = bits.view(BF)
    for up in (torch.ones_like(gate), gate.flip(0).contiguous()):
        want = F.silu(gate) * up
        out = torch.empty_like(gate)
        silu_mul2(gate, up, out)
        assert _same(out, want)
    for n in (8, 2056, 65536):           # in place: one chunk, one past a workgroup, all
        short, up = gate[:n].clone(), gate.flip(0)[:n].contiguous()
        want = F.silu(short) * up
        silu_mul2(short, up, short)
        assert _same(short, want)


@pytest.mark.parametrize("B,S,kw", [(1, 8, {}), (2, 77, {}), (1, 7, {}),
                                    (3, 19, dict(hidden=512, inter=1024, nq=8, nkv=2)),
                                    (2, 9, dict(hidden=192, inter=256, nq=4, nkv=1))])
def test_prefill_row_kernels_keep_the_torch_path_bits(dev, monkeypatch, B, S, kw):
    """Both routes over the same inputs, the widths and row counts that the row
    kernels do not take (fewer than 8 rows, rows of 192) among them; and a layer they
    do not serve (a norm gain that is a strided view) between two that they do."""
    cfg = Qwen3Config(layers=3, vocab=64, **kw)
    w = random_weights(cfg, seed=S, device=dev)
    w["layers"][1]["w_post"] = torch.ones(cfg.hidden, 2, dtype=BF, device=dev)[:, 0]
    prompt = torch.randint(0, cfg.vocab, (B, S), device=dev)
    cos, sin = _randn(None, S + 3, 128), _randn(None, S + 3, 128)

    def once():
        kc = torch.zeros(3, B, cfg.nkv, S + 3, 128, dtype=BF, device=dev)
        vc = torch.zeros_like(kc)
        return (*P.prefill(cfg, w, prompt, kc, vc, cos, sin), kc, vc)

    got = once()
    served = P._rows_served(cfg, w["embed"], B, S, got[2], got[3], cos, sin)
    assert served == (B * S >= 8 and cfg.hidden >= 256)
    monkeypatch.setattr(P, "_rows_served", lambda *a: False)
    for a, b in zip(got, once()):
        assert torch.equal(a, b)


def test_a_traced_prefill_replays_the_forward(dev):
    """torch.jit.trace records torch operations only, so it gets nothing else: a replay on
    other tokens has the eager call's bits."""
    cfg = Qwen3Config(layers=2, vocab=64)
    w = random_weights(cfg, seed=3, device=dev)
    cos, sin = _randn(None, 40, 128), _randn(None, 40, 128)

    def f(prompt, kc, vc):
        kc, vc = kc.clone(), vc.clone()
        return (*P.prefill(cfg, w, prompt, kc, vc, cos, sin), kc, vc)

    kc = torch.zeros(2, 2, cfg.nkv, 40, 128, dtype=BF, device=dev)
    one, other = (torch.randint(0, cfg.vocab, (2, 33), device=dev) for _ in range(2))
    f(one, kc, kc)   # the probes of this device and width, outside the trace
    traced = torch.jit.trace(f, (one, kc, kc), check_trace=False)
    for a, b in zip(traced(other, kc, kc), f(other, kc, kc)):
        assert torch.equal(a, b)
