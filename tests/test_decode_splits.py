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
