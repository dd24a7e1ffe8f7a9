"""The dense decode's split count for batches of more workgroups than are
resident at once (256 CUs, a group of 8 waves a CU for paired heads, two of 4
for single ones)."""

from __future__ import annotations

import pytest

from latentserve_amd.kernels.hip import paged_decode_hip as pdh


def _plain(batch, heads, pages, int8):
    """Units for the CUs, no split under MIN_SPLIT_PAGES pages."""
    units = pdh.UNITS_PER_4_CUS["int8" if int8 else "fp16"] * 64
    return max(1, min(-(-units // (batch * heads)), pages // pdh.MIN_SPLIT_PAGES))


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("heads", [1, 2, 3, 4, 8])
def test_more_groups_than_are_resident(int8, heads):
    """A split is added only where the launch deals the groups, and for sequences
    long enough to gain: elsewhere it is a second set of groups (up to 1.8 times
    the time)."""
    for batch in (60, 100, 129, 200, 256, 257, 300, 513, 1000):
        groups, fit = (batch * heads // 2, 256) if heads % 2 == 0 else (batch * heads, 512)
        if groups <= fit:
            continue
        for pages in (1, 16, 19, 47, 95, 96, 500, 4096):
            got = pdh.choose_splits(batch, heads, pages, None, int8=int8)
            if batch > 256 or pages < 96:
                assert got == _plain(batch, heads, pages, int8), (batch, pages)
            else:                                # whole rounds, no more than one split added
                assert got == -(-(-(-groups // fit) * fit) // groups) <= 2, (batch, pages)


@pytest.mark.parametrize("batch,heads,pages,one,two", [
    (13, 8, 384, 4, 9), (17, 8, 288, 3, 7), (22, 8, 192, 2, 5), (33, 8, 96, 1, 3), (50, 8, 96, 1, 1),
    (129, 1, 288, 3, 7),
])
def test_list_walks_of_long_splits_take_two_rounds(batch, heads, pages, one, two):
    """The page-subset walk's launch deals nothing: where whole rounds round the
    count down, a long sequence's few groups would run on alone.  (Two rounds of
    twice the count are no finer than one.)"""
    from latentserve_amd.kernels.hip import paged_sparse as ps

    def count(n, **kw):
        return pdh.choose_splits(batch, heads, n, None, dealt=False, **kw)

    rounds = ps.LIST_ROUND_PAGES
    assert count(pages, round_pages=rounds) == count(pages) == one
    assert count(pages + 1, round_pages=rounds) == two
    assert count(pages + 1) == one                     # selecting walks: one round


@pytest.mark.parametrize("batch,heads", [(1, 2), (8, 2), (16, 8), (65, 8), (200, 4)])
def test_list_walks_elsewhere_as_without_the_rule(batch, heads):
    for pages in (1, 60, 500, 8192):
        assert pdh.choose_splits(batch, heads, pages, None, dealt=False, round_pages=64) == \
            pdh.choose_splits(batch, heads, pages, None, dealt=False)
