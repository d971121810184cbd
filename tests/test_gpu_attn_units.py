"""One-token attention at the edges of its unit rules."""

import pytest
import torch

from kernel_optim_amd.kernels.fused import DecodeAttention
from oracle import attention as A

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _case(dev, B, cap, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    q = torch.randn(B, 32 * 128, device=dev, generator=g).to(BF)
    k, v = (torch.randn(B, 8, cap, 128, device=dev, generator=g).to(BF) for _ in range(2))
    return q, k, v


@pytest.mark.parametrize("unit", [64, 32, 16, 1024])
def test_a_pair_of_one_unit_keeps_the_merged_bits(dev, unit):
    """Sequences of no key, of one unit (which writes its output itself) and of more in one
    launch, against the two-launch form (which merges every pair) and the oracle."""
    cap = 2 * unit + 7
    lens = [0, 1, 15, 16, unit - 1, unit, unit + 1, cap]
    q, k, v = _case(dev, len(lens), cap, unit)
    n = torch.tensor(lens, dtype=torch.int32, device=dev)
    outs = []
    # one launch asked for, two launches, one by the op's rule
    for kw in (dict(fused_combine=True), dict(two_launches=True), {}):
        op = DecodeAttention(len(lens), 1, cap, 32, 8, 128, dev, unit=unit, **kw)
        assert op.one_launch == ("two_launches" not in kw)
        out = torch.full_like(q, float("nan"))
        for _ in range(2):   # the counters are left at zero
            op.with_lengths(q, k, v, n, out)
        for c in (op.counters, op._own_counters):
            assert c is None or int(c.abs().sum()) == 0
        outs.append(out)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[2], outs[1])
    assert int(outs[0][0].float().abs().sum()) == 0   # no key: zeros
    want = A.decode_attention(q[1:].cpu(), k[1:].cpu(), v[1:].cpu(), lens[1:])
    torch.testing.assert_close(outs[0][1:].cpu().double(), want, atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("split,unit", [(1, 64), (2, None), (3, 320), (5, 128), (10, None)])
def test_per_sequence_units(dev, split, unit):
    """decode_qkv cutting each sequence by its own length: lengths on both sides of the
    one that is left whole (2.5 units), of the smallest unit and of whole units."""
    u = unit or 64
    lens = [1, 63, 64, 65, (5 * u - 1) // 2, 5 * u // 2, 5 * u // 2 + 1, u * split, u * split + 1,
            2 * u * split + 3]
    B, cap = len(lens), -(-max(lens) // 16) * 16
    q, k, v = _case(dev, B, cap, split)
    g = torch.Generator(device=dev).manual_seed(7)
    qkv = torch.randn(B, 48 * 128, device=dev, generator=g).to(BF)
    ones = torch.ones(128, dtype=BF, device=dev)
    cos, sin = torch.ones(cap, 128, dtype=BF, device=dev), torch.zeros(cap, 128, dtype=BF, device=dev)
    pos = torch.tensor(lens, dtype=torch.int32, device=dev) - 1
    op = DecodeAttention(B, 1, cap, 32, 8, 128, dev, unit=unit, fused_combine=True,
                         units_per_seq=split)
    out = torch.zeros_like(q)
    for _ in range(2):
        op.decode_qkv(qkv, ones, ones, cos, sin, pos, k, v, out, 1e-6)
    assert int(op.counters.abs().sum()) == 0
    from kernel_optim_amd.prefill import rmsnorm   # cos = 1, sin = 0: the norm alone
    qn = rmsnorm(qkv[:, :32 * 128].view(B, 32, 128), ones, 1e-6).view(B, -1)
    want = A.decode_attention(qn.cpu(), k.cpu(), v.cpu(), lens)
    torch.testing.assert_close(out.cpu().double(), want, atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("B,split,lens,parts", [
    (12, 5, [1, 319, 320, 321, 400, 511, 512, 513, 640, 641, 800, 1500],
     [1, 1, 2, 2, 2, 2, 4, 5, 5, 4, 5, 5]),
    (4, 8, [159, 160, 255, 256], [1, 3, 4, 4]),          # one round: 8 units, of at least 64
    (17, 3, [799, 800, 1279, 1280] * 4 + [1], [1, 3, 3, 3] * 4 + [1])])   # one unit a round
def test_units_that_a_sequence_is_cut_into(dev, B, split, lens, parts):
    """Counted by the partials that it leaves (a whole sequence leaves none). More units than
    one round of the CUs are taken from 4 smallest units on."""
    cap = -(-max(lens) // 16) * 16
    q, k, v = _case(dev, B, cap, split)
    g = torch.Generator(device=dev).manual_seed(7)
    qkv = torch.randn(B, 48 * 128, device=dev, generator=g).to(BF)
    ones = torch.ones(128, dtype=BF, device=dev)
    cos, sin = torch.ones(cap, 128, dtype=BF, device=dev), torch.zeros(cap, 128, dtype=BF, device=dev)
    pos = torch.tensor(lens, dtype=torch.int32, device=dev) - 1
    op = DecodeAttention(B, 1, cap, 32, 8, 128, dev, fused_combine=True, units_per_seq=split)
    op.ml.fill_(float("nan"))
    out = torch.zeros_like(q)
    op.decode_qkv(qkv, ones, ones, cos, sin, pos, k, v, out, 1e-6)
    n = (~op.ml.view(B, 32, op.max_units, 2)[..., 0].isnan()).sum(-1)
    assert torch.equal(n, n[:, :1].expand(-1, 32))
    assert n[:, 0].tolist() == [p if p > 1 else 0 for p in parts]
    from kernel_optim_amd.prefill import rmsnorm
    qn = rmsnorm(qkv[:, :32 * 128].view(B, 32, 128), ones, 1e-6).view(B, -1)
    want = A.decode_attention(qn.cpu(), k.cpu(), v.cpu(), lens)
    torch.testing.assert_close(out.cpu().double(), want, atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("B,lens", [(1, [0]), (70, [0, 5] * 35)])
def test_sequences_without_keys_give_zeros(dev, B, lens):
    """One sequence, and more than 64 (whose lengths are read in chunks)."""
    q, k, v = _case(dev, B, 16, B)
    n = torch.tensor(lens, dtype=torch.int32, device=dev)
    outs = []
    for two in (False, True):
        op = DecodeAttention(B, 1, 16, 32, 8, 128, dev, unit=16, two_launches=two)
        assert op.one_launch != two
        out = torch.full_like(q, float("nan"))
        op.with_lengths(q, k, v, n, out)
        outs.append(out)
    assert torch.equal(outs[0], outs[1])
    assert int(outs[0][0].float().abs().sum()) == 0


def test_bad_arguments_are_named(dev):
    q, k, v = _case(dev, 2, 32, 1)
    n = torch.tensor([3, 4], dtype=torch.int32, device=dev)
    op = DecodeAttention(2, 1, 32, 32, 8, 128, dev)
    out = torch.zeros_like(q)
    bad = [("q must have shape", (q[:1], k, v, n, out)), ("out must be torch.bf", (q, k, v, n, out.float())),
           ("must share strides", (q, k, v.transpose(0, 1).contiguous().transpose(0, 1), n, out)),
           ("must have shape", (q, k[:, :, :16], v, n, out)), ("int32", (q, k, v, n.long(), out)),
           ("must be contiguous", (q, k, v, n, torch.zeros(4096, 2, dtype=BF, device=dev).t())),
           ("on the GPU", (q.cpu(), k, v, n, out)), ("must be a tensor", (None, k, v, n, out)),
           ("bf16 GPU", (q, k.float(), v.float(), n, out))]
    for text, args in bad:
        with pytest.raises(ValueError, match=text):
            op.with_lengths(*args)


def test_first_call_on_another_stream_than_the_objects(dev):
    """The arrival counters are zero for every stream: the constructor waits for the fill,
    here behind work on its own stream and over memory that held other words."""
    q, k, v = _case(dev, 2, 512, 3)
    n = torch.tensor([512, 300], dtype=torch.int32, device=dev)
    want = A.decode_attention(q.cpu(), k.cpu(), v.cpu(), [512, 300])
    out = torch.full_like(q, float("nan"))
    torch.cuda.synchronize()
    mine, other = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(mine):
        size = DecodeAttention(2, 1, 512, 32, 8, 128, dev).sync.untyped_storage().nbytes()
        old = torch.full((size // 4,), 7, dtype=torch.int32, device=dev)
        del old
        torch.cuda._sleep(20_000_000)
        op = DecodeAttention(2, 1, 512, 32, 8, 128, dev)
    assert op.one_launch
    with torch.cuda.stream(other):
        op.with_lengths(q, k, v, n, out)
    torch.cuda.synchronize()
    torch.testing.assert_close(out.cpu().double(), want, atol=2e-2, rtol=2e-2)


def test_an_object_made_under_capture_takes_two_launches(dev):
    """Its counters would be zeroed by the replays only."""
    q, k, v = _case(dev, 2, 512, 4)
    n = torch.tensor([512, 300], dtype=torch.int32, device=dev)
    want = A.decode_attention(q.cpu(), k.cpu(), v.cpu(), [512, 300])
    out, eager = torch.full_like(q, float("nan")), torch.full_like(q, float("nan"))
    DecodeAttention(2, 1, 512, 32, 8, 128, dev, two_launches=True).with_lengths(q, k, v, n, out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        op = DecodeAttention(2, 1, 512, 32, 8, 128, dev)
        op.with_lengths(q, k, v, n, out)
    assert not op.one_launch
    op.with_lengths(q, k, v, n, eager)   # before any replay
    for _ in range(3):
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
    torch.testing.assert_close(out.cpu().double(), want, atol=2e-2, rtol=2e-2)
