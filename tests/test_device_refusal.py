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


def _mixed_calls():
    """(entry, the operand left on the CPU) -> a call with every other operand on
    the GPU."""
    half = dict(dtype=torch.float16, device="cuda")
    zeros = torch.zeros

    def gather(name):
        ops = dict(pool=zeros(NB, 16, H, D, **half), t=_tables()[0].cuda(), l=_tables()[1].cuda())
        ops[name] = ops[name].cpu()
        return pg.gather(ops["pool"], ops["t"], ops["l"])

    def read(name):
        ops = dict(k=zeros(NB, 16, H, D, **half), v=zeros(NB, 16, H, D, **half),
                   t=_tables()[0].cuda(), l=_tables()[1].cuda())
        ops[name] = ops[name].cpu()
        return pg.read(ops["k"], ops["v"], ops["t"], ops["l"])

    def finalize(name):
        ops = dict(data=zeros(3, 16, H, D, **half), ids=zeros(2, dtype=torch.long, device="cuda"),
                   rows=zeros(2, dtype=torch.long, device="cuda"),
                   k_pool=zeros(NB, 16, H, D, dtype=torch.int8, device="cuda"),
                   k_scale=zeros(NB, H, D, device="cuda"), k_zero=zeros(NB, H, D, device="cuda"))
        ops[name] = ops[name].cpu()
        return iw.finalize_blocks(ops["data"], ops["ids"], ops["k_pool"], ops["k_scale"],
                                  ops["k_zero"], rows=ops["rows"], asym=True, eps=1e-8, qmax=127.0,
                                  levels=255.0, offset=128.0)

    def prefill(name):
        ops = dict(k=zeros(B, H, 5, D, **half), v=zeros(B, H, 5, D, **half),
                   slots=zeros(B, 5, dtype=torch.long, device="cuda"),
                   rows=zeros(B, dtype=torch.long, device="cuda"),
                   k_pool=zeros(NB, 16, H, D, dtype=torch.int8, device="cuda"),
                   k_scale=zeros(NB, H, D, device="cuda"), k_zero=zeros(NB, H, D, device="cuda"),
                   v_pool=zeros(NB, 16, H, D, dtype=torch.int8, device="cuda"),
                   v_scale=zeros(NB, 16, H, device="cuda"), v_zero=zeros(NB, 16, H, device="cuda"),
                   k_res=zeros(B, 16, H, D, **half))
        if name is not None:
            ops[name] = ops[name].cpu()
        quant = (1e-8, 127.0, 255.0, 128.0)
        return iw.prefill_write(*ops.values(), asym=True, k_quant=quant, v_quant=quant)

    return {(fn, name): (lambda fn=fn, name=name: fn(name)) for fn, names in (
        (gather, ("pool", "t", "l")), (read, ("k", "t", "l")),
        (finalize, ("data", "ids", "rows", "k_pool", "k_scale", "k_zero")),
        (prefill, ("k", "v", "slots", "rows", "k_pool", "k_scale", "k_zero", "v_pool", "v_scale",
                   "v_zero", "k_res"))) for name in names}, lambda: prefill(None)


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
def test_one_operand_on_the_cpu_is_refused(library):
    """A CPU operand among GPU ones (the recorder takes the launch's place)."""
    calls, whole = _mixed_calls()
    for (fn, name), call in calls.items():
        with pytest.raises(ValueError):
            call()
        assert library.launched == [], (fn.__name__, name)
    whole()
    assert library.launched == ["ls_int8_prefill_write"]


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
@pytest.mark.parametrize("before", [0, 3, 39, 40, -5])
def test_paged_write_leaves_rows_that_meet_the_pool(library, before):
    """Rows that start inside a pool, or before it and run into it, are not the
    kernel's (it reads and stores in no defined order); rows that end where it
    starts are.  (The recorder takes the launch's place.)"""
    from latentserve_amd.kernels.hip import paged_write as pw
    n = 40                                               # rows of k; `before` of them before the pool
    buf = torch.zeros(n + NB * 16, 1, D, dtype=torch.float16, device="cuda")
    k = buf[n - before:2 * n - before].view(1, n, 1, D).transpose(1, 2)
    k_pool, v_pool = buf[n:].view(NB, 16, 1, D), torch.zeros_like(buf[n:]).view(NB, 16, 1, D)
    slots = torch.arange(n, device="cuda")
    other = torch.zeros_like(k)
    for args in ((k, other, slots, k_pool, v_pool), (other, k, slots, k_pool, v_pool),
                 (k, other, slots, v_pool, k_pool), (other, k, slots, v_pool, k_pool)):
        library.launched.clear()
        assert pw.write(*args) is (before == n)
        assert library.launched == (["ls_paged_write"] if before == n else [])
