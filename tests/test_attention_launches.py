"""Which launches DecodeAttention makes; the decision is made on the host."""

import pytest

from kernel_optim_amd.kernels.fused import DecodeAttention


def _op(B, cap, **kw):
    return DecodeAttention(B, 1, cap, 32, 8, 128, "cpu", **kw)


@pytest.mark.parametrize("B,cap,units,one", [
    (1, 512, 8, True), (1, 1536, 24, True), (1, 1537, 25, False), (1, 4096, 64, False),
    (1, 8192, 64, False), (2, 2048, 32, False), (2, 2560, 20, True), (2, 16384, 32, False),
    (4, 8192, 16, True), (16, 8192, 2, True), (64, 16384, 4, False)])
def test_one_launch_only_where_few_units_meet_in_a_pair(B, cap, units, one):
    """One workgroup merges a pair's units in turn: past 24 of them the second launch, with
    a wavefront per row, is faster (and with several rounds of the grid, B = 64)."""
    op = _op(B, cap)
    assert op.max_units == units
    assert op.one_launch == one and op.counters is None
    assert _op(B, cap, fused_combine=True).one_launch


def test_two_launches_can_be_asked_for():
    """The reference's form, which a comparison of the two has to name."""
    for B, cap in ((16, 8192), (1, 512), (64, 16384)):
        assert not _op(B, cap, two_launches=True).one_launch
    with pytest.raises(ValueError, match="two_launches"):
        _op(1, 512, two_launches=True, fused_combine=True)
    with pytest.raises(ValueError, match="two_launches"):
        DecodeAttention(2, 3, 512, 32, 8, 128, "cpu", two_launches=True, fused_combine=True,
                        token_rows=True)
