"""Host logic of speculative decoding (CPU): prompt-lookup drafts and the
acceptance rule of the verify step (engine/engine.py:48-93, 477-484). The
expected drafts are worked out by hand from the lookup's definition: the
latest earlier occurrence of the last 3, else 2, else 1 tokens proposes what
followed it, a continuation that reaches the end reads the draft itself, and no
occurrence repeats the last token."""

import pytest
import torch

from kernel_optim_amd.engine import HostCopies, NgramIndex, accept, draft_len
from kernel_optim_amd.model import Qwen3Config


def test_draft_follows_latest_trigram():
    # (1, 2, 3) occurred at 0..2 and was followed by 4, 1, 2
    assert NgramIndex([1, 2, 3, 4, 1, 2, 3]).draft(3) == [4, 1, 2]


def test_draft_runs_into_itself():
    # only (7,) occurred before, followed by 8, 7 and then the draft's own 8
    assert NgramIndex([7, 8, 7]).draft(3) == [8, 7, 8]
    assert NgramIndex([7, 8, 7]).draft(5) == [8, 7, 8, 7, 8]


def test_draft_latest_occurrence_wins():
    # (1,) occurred at 0 (-> 2) and at 2 (-> 3): the later one proposes 3, 1, then itself
    assert NgramIndex([1, 2, 1, 3, 1]).draft(3) == [3, 1, 3]


def test_draft_prefers_longer_match():
    # bigram (5, 6) was followed by 9; unigram (6,) latest by 7
    seq = [5, 6, 9, 6, 7, 5, 6]
    assert NgramIndex(seq).draft(2) == [9, 6]


def test_draft_without_match_repeats_last():
    assert NgramIndex([42]).draft(4) == [42, 42, 42, 42]
    assert NgramIndex([1, 2, 3]).draft(2) == [3, 3]


def test_extend_is_incremental():
    a = NgramIndex([1, 2, 3, 4])
    a.extend([1, 2, 3])
    b = NgramIndex([1, 2, 3, 4, 1, 2, 3])
    assert a.seq == b.seq and a.after == b.after and a.draft(4) == b.draft(4)


def test_accept_prefix_and_next_token():
    # verify input [last, d1, d2, d3]; greedy ids after each input position
    assert accept([5, 1, 2, 3], [1, 2, 3, 8]) == [1, 2, 3, 8]   # all drafts + the next
    assert accept([5, 1, 2, 3], [1, 2, 9, 4]) == [1, 2, 9]      # stops at the first miss
    assert accept([5, 1, 2, 3], [7, 2, 3, 4]) == [7]            # no draft accepted
    assert accept([5], [6]) == [6]                              # K = 0


def test_draft_len_by_batch():
    assert [draft_len(b) for b in (1, 4, 5, 16, 17, 32, 33)] == [6, 6, 4, 4, 2, 2, 0]


@pytest.mark.parametrize("tune", [True, False])
def test_auto_takes_the_fused_graph_where_its_gemvs_read_the_weights_once(monkeypatch, tune):
    """Up to 32 sequences at any width; up to 64 where layout 5 serves the widths, which is
    not taken with tuning off."""
    from kernel_optim_amd import engine
    monkeypatch.setattr(engine, "TUNE", tune)
    small = Qwen3Config(layers=2, vocab=64, hidden=512, inter=1024, nq=8, nkv=2)
    assert engine.rows_served(Qwen3Config()) and not engine.rows_served(small)
    for cfg, most in ((Qwen3Config(), 64 if tune else 32), (small, 32)):
        for B in (1, 32, 33, 64, 65):
            assert engine.auto_graph(cfg, B) == ("fused" if B <= most else "hipblaslt")


def test_attention_units_per_sequence_fill_the_cus():
    """One round of the 256 CUs where that fills them, else the cut that fills its rounds
    best; fixed units for one or two sequences and above 64."""
    from kernel_optim_amd.engine import attn_units_per_seq
    assert [attn_units_per_seq(B, 8) for B in (1, 2, 3, 4, 8, 10, 16, 32, 64, 65)] == \
        [0, 0, 10, 8, 4, 3, 2, 1, 1, 0]
    assert [attn_units_per_seq(B, 8) for B in (11, 12, 13, 17, 21, 22, 24, 33, 42, 43, 48, 49)] == \
        [5, 5, 2, 3, 3, 1, 1, 3, 3, 2, 2, 1]
    for nkv in (1, 2, 8):
        for B in range(3, 65):
            u = attn_units_per_seq(B, nkv)
            assert u >= 1 and B * nkv * u <= 1024


@torch.inference_mode()
def test_host_copies_are_pinned_while_few_are_held():
    pins = []

    def empty(*a, pin_memory, **kw):
        pins.append(pin_memory)
        return torch.empty(*a, **kw)

    copies = HostCopies(4000, empty)
    ids, logits = torch.arange(10), torch.randn(10, 90).bfloat16()   # 80 + 1800 bytes
    for _ in range(5):   # dropped at once: the next call may pin again
        got = copies((ids, logits))
        assert torch.equal(got[0], ids) and torch.equal(got[1], logits)
        del got
    assert pins == [True] * 10
    kept = []
    for i in range(4):
        kept.append([t[1:3] for t in copies((ids, logits))])   # views hold the whole
    assert pins[10:] == [True] * 4 + [False] * 4
    assert all(torch.equal(a, ids[1:3]) and torch.equal(b, logits[1:3]) for a, b in kept)
    del kept[0]
    copies((ids, logits))
    assert pins[18:] == [True] * 2
    huge = torch.zeros(4001, dtype=torch.uint8)
    assert torch.equal(copies((huge,))[0], huge) and pins[-1] is False
