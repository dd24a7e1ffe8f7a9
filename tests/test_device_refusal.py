"""CPU tensors never reach a HIP launch: every entry point that takes its stream
from its operands' device refuses them.  The library is replaced by a recorder,
so nothing is launched here whatever the entry points do, with or without a
GPU."""

from __future__ import annotations

import pytest
import torch

from latentserve_amd import _lib
from latentserve_amd.kernels.hip import int8_write as iw
from latentserve_amd.kernels.hip import paged_gather as pg
from latentserve_amd.kernels.hip import paged_sparse as ps
from latentserve_amd.runtime.kv_cache import KVCacheSpec, PagedKVCache

B, H, NB, PAGES, D = 2, 2, 8, 4, 128


class _Recorder:
    def __init__(self):
        self.launched = []

    def __getattr__(self, name):
        if name.endswith("_bytes") or name.endswith("_ints"):
            return lambda *a: 64
        return lambda *a: self.launched.append(name) or 0


@pytest.fixture
def library(monkeypatch):
    rec = _Recorder()
    monkeypatch.setattr(_lib, "lib", lambda: rec)
    # a GPU host's stream lookup: the current device when none is named
    monkeypatch.setattr(_lib, "_raw_stream", lambda index: 1)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    return rec


def _half(*shape):
    return torch.zeros(*shape, dtype=torch.float16)


def _cache():
    c = PagedKVCache(KVCacheSpec(num_layers=1, num_kv_heads=H, head_dim=D, max_batch_size=B,
                                 max_seq_len=64, device="cpu"))
    c.advance(20)
    return c


def _tables():
    return torch.zeros(B, PAGES, dtype=torch.int32), torch.full((B,), 20, dtype=torch.int32)


def _finalize():
    iw.finalize_blocks(_half(1, 16, H, D), torch.zeros(1, dtype=torch.long),
                       torch.zeros(NB, 16, H, D, dtype=torch.int8), torch.zeros(NB, H, D),
                       asym=False, eps=1e-8, qmax=127.0, levels=255.0, offset=128.0)


CALLS = {
    "cache read": lambda: _cache().read(0, B),
    "cache page bounds": lambda: _cache().enable_page_bounds(),
    "gather": lambda: pg.gather(_half(NB, 16, H, D), *_tables()),
    "read, unlike pools": lambda: pg.read(_half(NB, 16, H, D), _half(NB + 1, 16, H, D), *_tables()),
    "rebuild_bounds": lambda: ps.rebuild_bounds(_half(NB, 16, H, D), _half(NB, H, D),
                                                _half(NB, H, D)),
    "update_bounds": lambda: ps.update_bounds(_half(B, H, D), torch.zeros(B, dtype=torch.long),
                                              _half(NB, H, D), _half(NB, H, D)),
    "page_scores": lambda: ps.page_scores(_half(B, H, 6, D), _half(NB, H, D), _half(NB, H, D),
                                          *_tables()),
    "page_scores_mass": lambda: ps.page_scores_mass(_half(B, H, 6, D), _half(NB, H, D),
                                                    _half(NB, H, D), *_tables()),
    "index_select": lambda: ps.index_select(_half(B, H, 6, D), _half(NB, H, D), _half(NB, H, D),
                                            *_tables(), 2, 0.5),
    "select": lambda: ps.select(torch.zeros(B, H, PAGES), 2),
    "finalize_blocks": _finalize,
}


@pytest.mark.parametrize("call", CALLS)
def test_cpu_tensors_are_refused(library, call):
    with pytest.raises(ValueError, match="cuda"):
        CALLS[call]()
    assert library.launched == []


def test_stream_of_takes_gpu_devices_only(library):
    assert _lib.stream_of(torch.device("cuda")) == 1
    assert _lib.stream_of(torch.device("cuda", 3)) == 1
    for device in ("cpu", "meta"):
        with pytest.raises(ValueError):
            _lib.stream_of(torch.device(device))
