"""Which launches sparse_attention makes, on the CPU: the library is replaced by
a recorder, so the operands can be CPU tensors and nothing runs."""

from __future__ import annotations

import pytest
import torch

from latentserve_amd import _lib
from latentserve_amd.kernels.hip import paged_decode_hip as pdh
from latentserve_amd.kernels.hip import paged_sparse as ps

H, NREP, D = 2, 6, 128


class _Recorder:
    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        if name.endswith("_bytes") or name.endswith("_ints"):
            return lambda *a: 64
        return lambda *a: self.calls.append((name, a)) or 0


@pytest.fixture
def library(monkeypatch):
    rec = _Recorder()
    monkeypatch.setattr(_lib, "lib", lambda: rec)
    monkeypatch.setattr(_lib, "stream_of", lambda device: 1)
    monkeypatch.setattr(pdh, "ineligible_reason", lambda *a: None)
    return rec


def _attend(width, bound_blocks=None, blocks=32, batch=2, heads=H, ratio=0.5, **kw):
    half = dict(dtype=torch.float16)
    bounds = [torch.zeros(blocks if bound_blocks is None else bound_blocks, heads, D, **half)
              for _ in range(2)]
    pool = torch.zeros(blocks, 16, heads, D, **half)
    ps.sparse_attention(torch.zeros(batch, heads, NREP, D, **half), pool, pool,
                        torch.zeros(batch, width, dtype=torch.int32),
                        torch.full((batch,), 16 * width, dtype=torch.int32), *bounds, ratio=ratio,
                        **kw)


@pytest.mark.parametrize("width", [40, 2048, 2049, 8192])
@pytest.mark.parametrize("bound_blocks", [31, 32, 33])
def test_one_launch_only_with_bounds_of_every_pool_block(library, width, bound_blocks):
    """The one-launch path has one block count for pools and bounds: with bounds
    of fewer blocks it would read past their end, whatever the row's length."""
    _attend(width, bound_blocks)
    names = [name for name, _ in library.calls]
    if bound_blocks == 32:
        assert names == ["ls_sparse_attention_bounds_fp16" if width <= ps.COOP_MAX_PAGES
                         else "ls_sparse_attention_bounds_long_fp16"]
    else:
        assert names == ["ls_page_scores", "ls_sparse_attention_fp16"]
        assert library.calls[0][1][5] == bound_blocks


def test_every_row_width_counts_in_a_buffer_of_its_own(library):
    """A row's count of scored shares is the word behind its scores, all ones at
    rest: widths that share a buffer leave scores in each other's counts."""
    for width in (40, 41, 42, 43, 44):
        _attend(width)
    one = "ls_sparse_attention_bounds_fp16"
    buffers = [args[13] for name, args in library.calls if name == one]
    assert len(set(buffers)) == 5
    for width in (40, 43):                      # and the same one again
        _attend(width)
    again = [args[13] for name, args in library.calls if name == one][5:]
    assert again == [buffers[0], buffers[3]]


@pytest.mark.parametrize("batch,heads,width,one", [
    (2, 2, 2048, True), (2, 2, 8192, True),           # 64 groups a row: 128 pages each
    (8, 8, 2048, True), (8, 8, 2049, False),          # 64 rows, four groups each
    (13, 5, 480, True), (13, 5, 616, False),          # 65 rows, three groups each
    (13, 5, 615, True), (17, 8, 294, True),           # under 40000 pages in all
    (16, 8, 320, True), (16, 8, 321, False),
    (17, 8, 160, True), (17, 8, 295, False),          # a group a row
    (33, 8, 160, True), (33, 8, 161, False), (200, 8, 161, False),
    (25, 6, 6250, False),                             # more than a group a row needed
])
def test_one_launch_while_a_groups_share_of_the_scoring_is_a_batch(library, batch, heads, width, one):
    """Past it a long row's few groups score while the chip idles, and where not
    every group is resident they wait for groups that have not started."""
    _attend(width, batch=batch, heads=heads, ratio=0.25)
    names = [name for name, _ in library.calls]
    if one:
        assert names == ["ls_sparse_attention_bounds_fp16" if width <= ps.COOP_MAX_PAGES
                         else "ls_sparse_attention_bounds_long_fp16"]
    else:
        assert names == ["ls_page_scores", "ls_sparse_attention_fp16"]


@pytest.mark.parametrize("scoring", ["bounds", "mass"])
@pytest.mark.parametrize("batch,heads,width,splits", [
    (16, 8, 1000, 2), (17, 8, 632, 1), (17, 8, 640, 3), (25, 6, 6250, 3), (170, 1, 640, 3),
    (171, 1, 640, 1), (25, 8, 4375, 2), (32, 8, 2000, 1), (33, 8, 2000, 1),
    (12, 8, 1276, 2), (12, 8, 1280, 5), (9, 8, 1920, 7), (8, 8, 8192, 4), (13, 8, 4000, 2),
])
def test_splits_of_the_two_launch_path(library, scoring, batch, heads, width, splits):
    """Where the whole groups a row that are resident leave CUs idle (129 to 170
    rows: one), long lists take two rounds of an odd count; a list longer than a
    group's table has as many as it needs."""
    _attend(width, batch=batch, heads=heads, ratio=0.25, scoring=scoring)
    name, args = library.calls[-1]
    assert name == "ls_sparse_attention_fp16"
    assert args[-4] == splits
    library.calls.clear()
    _attend(width, batch=batch, heads=heads, ratio=0.25, scoring=scoring, num_splits=4)
    assert library.calls[-1][1][-4] == 4              # as asked
