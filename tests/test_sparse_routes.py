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


def _attend(width, bound_blocks=None, blocks=32, batch=2):
    half = dict(dtype=torch.float16)
    bounds = [torch.zeros(blocks if bound_blocks is None else bound_blocks, H, D, **half)
              for _ in range(2)]
    pool = torch.zeros(blocks, 16, H, D, **half)
    ps.sparse_attention(torch.zeros(batch, H, NREP, D, **half), pool, pool,
                        torch.zeros(batch, width, dtype=torch.int32),
                        torch.full((batch,), 16 * width, dtype=torch.int32), *bounds, ratio=0.5)


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
