"""Which calls of the prompt forward its row kernels take. They work by address, so a call
that something records, rewrites or differentiates has to stay with the torch operations. On
the CPU, with stand-ins in place of the kernels that fail, against the torch route."""

import pytest
import torch
import torch.autograd.forward_ad as fad
from torch.fx.experimental.proxy_tensor import make_fx
from torch.utils.flop_counter import FlopCounterMode

import kernel_optim_amd.prefill as P
from kernel_optim_amd.model import Qwen3Config, random_weights

BF = torch.bfloat16
B, S, CAP = 2, 8, 16
CFG = Qwen3Config(layers=2, vocab=64, hidden=256, inter=512, nq=4, nkv=1)


class RowKernel(Exception):
    pass


@pytest.fixture
def rows(monkeypatch):
    """The route decision as on the GPU, where a row kernel raises RowKernel."""
    def stand_in(*a):
        raise RowKernel
    for name in ("prefill_norm", "prefill_qkv", "silu_mul2"):
        monkeypatch.setattr(P, name, stand_in)
    monkeypatch.setattr(P, "_on_gpu", lambda dev: True)
    monkeypatch.setattr(P, "_row_sums_exact", lambda dev, n: True)


def _inputs(seed=1):
    w = random_weights(CFG, seed=seed)
    g = torch.Generator().manual_seed(seed)
    kc, vc = (torch.zeros(CFG.layers, B, CFG.nkv, CAP, 128, dtype=BF) for _ in range(2))
    cos, sin = (torch.randn(CAP, 128, generator=g).to(BF) for _ in range(2))
    return w, torch.randint(0, CFG.vocab, (B, S), generator=g), kc, vc, cos, sin


def _call(w, prompt, kc, vc, cos, sin):
    ids, logits = P.prefill(CFG, w, prompt, kc, vc, cos, sin)
    return ids, logits, kc, vc


def _torch_route(args):
    w, prompt, kc, vc, cos, sin = args
    x = torch.nn.functional.embedding(prompt, w["embed"])
    kc, vc = kc.clone(), vc.clone()
    gqa = P.gqa_exact(prompt.device)
    for i, lw in enumerate(w["layers"]):
        x = P._layer_torch(CFG, lw, x, kc[i], vc[i], cos, sin, gqa)
    x = P.rmsnorm(x[:, -1:], w["final_norm"], CFG.eps)
    logits = torch.nn.functional.linear(x, w["lm_head"])[:, -1]
    return logits.argmax(-1), logits, kc, vc


def _same(got, want):
    for a, b in zip(got, want):
        assert torch.equal(a, b)


def test_a_plain_call_takes_the_row_kernels(rows):
    with pytest.raises(RowKernel):
        _call(*_inputs())
    with pytest.raises(RowKernel), torch.device("cpu"):   # a default device rewrites nothing
        _call(*_inputs())
    with pytest.raises(RowKernel), torch.inference_mode():
        _call(*_inputs())


@pytest.mark.parametrize("how", ["jit", "make_fx", "make_fx_pre_dispatch"])
def test_a_traced_call_records_the_whole_forward(rows, how):
    w, prompt, kc, vc, cos, sin = _inputs()
    P.gqa_exact(prompt.device)   # its own probe runs once per device, not in the trace

    def f(prompt, kc, vc):
        return _call(w, prompt, kc.clone(), vc.clone(), cos, sin)

    if how == "jit":
        traced = torch.jit.trace(f, (prompt, kc, vc), check_trace=False)
    else:
        traced = make_fx(f, pre_dispatch="pre" in how)(prompt, kc, vc)
    other = prompt.flip(0).roll(3, 1)
    _same(traced(other, kc, vc), _torch_route((w, other, kc, vc, cos, sin)))


def test_a_transformed_call_stays_with_the_torch_operations(rows):
    args = _inputs()
    w, prompt, kc, vc, cos, sin = args
    want = _torch_route(args)

    def f(prompt, kc, vc):
        return _call(w, prompt, kc, vc, cos, sin)

    _same(torch.func.functionalize(f)(prompt, kc.clone(), vc.clone()), want)
    with FlopCounterMode(display=False) as counter:
        _same(f(prompt, kc.clone(), vc.clone()), want)
    assert counter.get_total_flops() > 0
    two = [torch.stack([t, t]) for t in (prompt, kc, vc)]
    for got in zip(*torch.vmap(f)(*two)):
        for a, b in zip(got, want):
            torch.testing.assert_close(a, b, rtol=2e-2, atol=2e-2)   # batched products


def test_forward_mode_keeps_the_tangents(rows):
    w, prompt, kc, vc, cos, sin = _inputs()
    with fad.dual_level():
        w["final_norm"] = fad.make_dual(w["final_norm"], torch.ones_like(w["final_norm"]))
        logits = P.prefill(CFG, w, prompt, kc, vc, cos, sin)[1]
        assert fad.unpack_dual(logits).tangent is not None


class Logged(torch.Tensor):
    """A subclass whose operations return it, as a wrapper or a distributed tensor does."""


@pytest.mark.parametrize("name", ["prompt", "k_cache", "v_cache", "cos", "sin", "embed", "w_in",
                                  "w_post", "q_norm", "k_norm", "qkv", "o", "gu", "down"])
def test_tensor_subclasses_keep_the_torch_operations(rows, name):
    """In any argument, and in the first layer (whose output then is one too)."""
    args = list(_inputs())
    want = _torch_route(args)
    at = ("w", "prompt", "k_cache", "v_cache", "cos", "sin")
    if name in at:
        args[at.index(name)] = args[at.index(name)].as_subclass(Logged)
    elif name == "embed":
        args[0]["embed"] = args[0]["embed"].as_subclass(Logged)
    else:
        args[0]["layers"][0][name] = args[0]["layers"][0][name].as_subclass(Logged)
    if name in at or name == "embed":
        _same([t.as_subclass(torch.Tensor) for t in _call(*args)], want)
        return
    reached = []
    plain = P._layer_torch
    P._layer_torch = lambda *a: reached.append(plain(*a)) or reached[-1]
    try:
        # the norms' results are subclasses, but the products of plain weights are too: the
        # second layer's input decides
        _same([t.as_subclass(torch.Tensor) for t in _call(*args)], want)
    finally:
        P._layer_torch = plain
    assert len(reached) == 2 and type(reached[0]) is Logged
