"""GEMV layout 5 (up to 64 rows per weight pass) against the oracle, at the edges of its
row tiles, column groups and slices, and its chained form against the plain one."""

import pytest
import torch

from kernel_optim_amd.kernels import gemv
from oracle import ops as O
from tests.bf16util import assert_bf16_close, assert_resid_close, one_ulp_at

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _g(dev, seed):
    return torch.Generator(device=dev).manual_seed(seed)


def _w(dev, rows, K, seed):
    return (torch.randn(rows, K, device=dev, generator=_g(dev, seed)) * 0.02).to(BF)


# one row, part-filled and full row tiles, a second weight pass of one row
ROWS = [1, 2, 15, 16, 17, 33, 48, 49, 64, 65]


# N: the model's width; fewer tiles than a group; a part-filled last tile and group
@pytest.mark.parametrize("M,N", [(m, 6144) for m in ROWS] + [(20, 16), (64, 200), (5, 1000)])
def test_norm_projections(dev, M, N):
    K = 2560
    g = _g(dev, M + N)
    x = torch.randn(M, K, device=dev, generator=g).to(BF)
    nw = (1 + 0.1 * torch.randn(K, device=dev, generator=g)).to(BF)
    ss = x.float().pow(2).sum(-1)
    W = _w(dev, N, K, 3)
    Wt = gemv.tile_weights(W)
    want = O.gemv(x.cpu(), W.cpu(), O.EPI_F32, nw=nw.cpu(), ss=ss.cpu())
    op = gemv.Gemv(M, N, K, gemv.EPI_F32, norm=True)
    assert M == 1 or (5, 2, 1) in op.candidates()
    for given in (None, ss):
        y = torch.empty(M, N, device=dev)
        op(x, Wt, y=y, nw=nw, ss=given, cfg=(5, 2, 1))
        torch.testing.assert_close(y.cpu(), want, rtol=2e-3, atol=2e-3)
    y = torch.empty(M, N, device=dev, dtype=BF)
    gemv.Gemv(M, N, K, gemv.EPI_BF16, norm=True)(x, Wt, y=y, nw=nw, cfg=(5, 2, 1))
    assert_bf16_close(y.cpu(), want.to(BF), max_frac=0.02, atol=one_ulp_at(want))
    for cfg in ((5, 6, 1), (5, 4, 1)):
        op = gemv.Gemv(M, N, K, gemv.EPI_ARGMAX, norm=True)
        ids = torch.full((M,), -1, device=dev, dtype=torch.int64)
        lg = torch.empty(M, N, device=dev, dtype=BF)
        op(x, Wt, y=lg, nw=nw, ids=ids, cfg=cfg)
        assert torch.equal(lg, y)
        assert torch.equal(ids.cpu(), O.argmax_first(lg.cpu()))


@pytest.mark.parametrize("M,N", [(m, 9728) for m in (2, 16, 17, 48, 64, 70)] + [(33, 200)])
def test_swiglu(dev, M, N):
    K = 2560
    g = _g(dev, M)
    x = torch.randn(M, K, device=dev, generator=g).to(BF)
    nw = (1 + 0.1 * torch.randn(K, device=dev, generator=g)).to(BF)
    W = _w(dev, 2 * N, K, 4)
    y = torch.empty(M, N, device=dev, dtype=BF)
    op = gemv.Gemv(M, N, K, gemv.EPI_SWIGLU, norm=True)
    op(x, gemv.tile_weights(W, swiglu=True), y=y, nw=nw, cfg=(5, 3, 1))
    want = O.gemv(x.cpu(), W.cpu(), O.EPI_SWIGLU, nw=nw.cpu(), ss=x.cpu().float().pow(2).sum(-1))
    # 4 ulp: a rounding tie of the gate (tests/test_gpu_ops.py, two row tiles)
    assert_bf16_close(y.cpu(), want, max_ulp=4, max_frac=0.03, atol=one_ulp_at(want))


@pytest.mark.parametrize("M,N", [(m, 2560) for m in ROWS] + [(20, 8), (64, 196), (9, 8192)])
@pytest.mark.parametrize("K,cfg", [(4096, (5, 3, 4)), (9728, (5, 3, 4))])
def test_residual_projections(dev, M, N, K, cfg):
    g = _g(dev, M + N + K)
    x = torch.randn(M, K, device=dev, generator=g).to(BF)
    W = _w(dev, N, K, 5)
    Wt = gemv.tile_weights(W)
    h0 = torch.randn(M, N, device=dev, generator=g).to(BF)
    want, ssr = O.gemv(x.cpu(), W.cpu(), O.EPI_RESID, h=h0.cpu())
    op = gemv.Gemv(M, N, K, gemv.EPI_RESID, norm=False)
    h, ss_out = h0.clone(), torch.full((M,), 5.0, device=dev)
    op(x, Wt, h=h, ss_out=ss_out, cfg=cfg)
    assert_resid_close(h.cpu(), want, O.gemv(x.cpu(), W.cpu(), O.EPI_F32))
    torch.testing.assert_close(ss_out.cpu(), ssr + 5.0, rtol=1e-3, atol=1e-2)
    # h as rows of a larger buffer, 2 bytes off: the same bits
    off = torch.empty(M * N + 1, dtype=BF, device=dev)[1:].view(M, N)
    off.copy_(h0)
    op(x, Wt, h=off, cfg=cfg)
    assert torch.equal(off, h)


@pytest.mark.parametrize("M", [2, 16, 31, 64])
def test_chained_projections_keep_the_plain_bits(dev, M):
    """o -> gate/up and down -> qkv with the normalised input left by the residual
    projection, over graph replays, against each projection's own norm."""
    H, I, NQ = 2560, 9728, 6144
    g = _g(dev, M)
    a = torch.randn(M, 4096, device=dev, generator=g).to(BF)
    h0 = torch.randn(M, H, device=dev, generator=g).to(BF)
    n1, n2 = ((1 + 0.1 * torch.randn(H, device=dev, generator=g)).to(BF) for _ in range(2))
    wo, wg, wd, wq = (gemv.tile_weights(_w(dev, r, k, s), swiglu=s == 7)
                      for r, k, s in ((H, 4096, 6), (2 * I, H, 7), (H, I, 8), (NQ, H, 9)))
    o = gemv.Gemv(M, H, 4096, gemv.EPI_RESID, norm=False)
    gu = gemv.Gemv(M, I, H, gemv.EPI_SWIGLU, norm=True)
    dn = gemv.Gemv(M, H, I, gemv.EPI_RESID, norm=False)
    qkv = gemv.Gemv(M, NQ, H, gemv.EPI_BF16, norm=True)
    o.cfg, gu.cfg, dn.cfg, qkv.cfg = (5, 3, 4), (5, 3, 1), (5, 3, 4), (5, 2, 1)

    def run(h, act, y, chained):
        h.copy_(h0)
        bg, bq = (gu.xn_buffer(h.device), qkv.xn_buffer(h.device)) if chained else (None, None)
        o(a, wo, h=h, nxt=(n1, bg) if chained else None)
        gu(h, wg, y=act, nw=n1, xn=bg)
        dn(act, wd, h=h, nxt=(n2, bq) if chained else None)
        qkv(h, wq, y=y, nw=n2, xn=bq)

    def bufs():
        return (torch.zeros(M, H, device=dev, dtype=BF), torch.zeros(M, I, device=dev, dtype=BF),
                torch.zeros(M, NQ, device=dev, dtype=BF))

    want, got = bufs(), bufs()
    run(*want, False)
    run(*got, True)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run(*got, True)
    for _ in range(3):
        for t in got:
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        for p, q in zip(want, got):
            assert torch.equal(p, q)
        run(*bufs(), False)   # eager work between the replays


def test_chaining_refuses_what_it_does_not_serve(dev):
    o = gemv.Gemv(65, 2560, 4096, gemv.EPI_RESID, norm=False)
    gu = gemv.Gemv(16, 9728, 2560, gemv.EPI_SWIGLU, norm=True)
    a = torch.zeros(65, 4096, device=dev, dtype=BF)
    h = torch.zeros(65, 2560, device=dev, dtype=BF)
    w = gemv.tile_weights(torch.zeros(2560, 4096, device=dev, dtype=BF))
    nw = torch.ones(2560, device=dev, dtype=BF)
    with pytest.raises(ValueError, match="up to 64 rows"):
        o(a, w, h=h, cfg=(5, 3, 4), nxt=(nw, gu.xn_buffer(h.device)))
    with pytest.raises(ValueError, match="layout 5"):
        gu(h[:16], gemv.tile_weights(torch.zeros(19456, 2560, device=dev, dtype=BF), swiglu=True),
           y=torch.zeros(16, 9728, device=dev, dtype=BF), nw=nw, cfg=(2, 1, 0),
           xn=gu.xn_buffer(h.device))


def test_layouts_of_one_projection_may_alternate(dev):
    """Layout 5's sums and layout 4's arrival counters do not share scratch: a Gemv that has
    run one layout runs the other correctly (as tune does)."""
    M, N, K = 8, 2560, 9728
    g = _g(dev, 1)
    x = torch.randn(M, K, device=dev, generator=g).to(BF)
    W = _w(dev, N, K, 5)
    Wt = gemv.tile_weights(W)
    h0 = torch.randn(M, N, device=dev, generator=g).to(BF)
    want, _ = O.gemv(x.cpu(), W.cpu(), O.EPI_RESID, h=h0.cpu())
    y = O.gemv(x.cpu(), W.cpu(), O.EPI_F32)
    op = gemv.Gemv(M, N, K, gemv.EPI_RESID, norm=False)
    for cfg in [(5, 3, 4), (4, 10, 0), (5, 3, 4), (3, 4, 0), (5, 3, 4), (4, 10, 0)]:
        h = h0.clone()
        op(x, Wt, h=h, cfg=cfg)
        assert_resid_close(h.cpu(), want, y)


@pytest.mark.parametrize("K", [2560, 4096])
@pytest.mark.parametrize("M", [1, 2, 3, 5, 8, 13, 15, 16])
def test_layout_2_takes_x_in_row_runs(dev, M, K):
    """Layout 2 loads a wavefront's slice of x as runs of its rows and only as many loads as
    the rows hold; rows past M (poisoned here) reach no output."""
    N = 1000
    g = _g(dev, M)
    buf = torch.full((M + 1, K), float("nan"), device=dev, dtype=BF)
    x = buf[:M]
    x.copy_(torch.randn(M, K, device=dev, generator=g))
    nw = (1 + 0.1 * torch.randn(K, device=dev, generator=g)).to(BF)
    W = _w(dev, N, K, 3)
    Wt = gemv.tile_weights(W)
    for norm in (False, True):
        kw = dict(nw=nw, ss=None) if norm else {}
        y = torch.empty(M, N, device=dev)
        gemv.Gemv(M, N, K, gemv.EPI_F32, norm=norm)(x, Wt, y=y, cfg=(2, 1, 0), **kw)
        ref = dict(nw=nw.cpu(), ss=x.cpu().float().pow(2).sum(-1)) if norm else {}
        want = O.gemv(x.cpu(), W.cpu(), O.EPI_F32, **ref)
        torch.testing.assert_close(y.cpu(), want, rtol=2e-3, atol=2e-3)
