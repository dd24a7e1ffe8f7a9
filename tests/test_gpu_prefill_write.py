"""A prefill chunk's K/V write and read-back, on an MI355X.

* fp16 / fp32 caches: the one-launch write puts every row at its slot bit for
  bit whatever the strides of k and v (rows the kernel cannot load take the
  indexed store), touches nothing else, and the one-launch read of both pools
  equals a gather of each.
* INT8: after chunks that start and end everywhere in a page, the codes, steps
  and residual equal the oracle's quantizers (bit for bit), K rows before a
  chunk in its first page coming from the residual.
"""

from __future__ import annotations

import numpy as np
import pytest

import oracle

torch = pytest.importorskip("torch")

pytestmark = [
    pytest.mark.gpu,
    pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU"),
]

BS = 16


def _layout(x, how):
    """The same values [B, H, n, D] in other memory."""
    if how == "token-major":                       # a projection's [B, n, H, D]
        return x.transpose(1, 2).contiguous().transpose(1, 2)
    if how == "slice":                             # part of a wider fused row
        wide = torch.zeros(*x.shape[:-1], x.shape[-1] + 64, dtype=x.dtype, device=x.device)
        wide[..., 32:32 + x.shape[-1]] = x
        return wide[..., 32:32 + x.shape[-1]]
    if how == "misaligned":                        # rows 2 elements off 16 bytes
        flat = torch.zeros(x.numel() + 2, dtype=x.dtype, device=x.device)
        flat[2:] = x.reshape(-1)
        return flat[2:].view(x.shape)
    if how == "strided":                           # channels not adjacent
        return x.transpose(2, 3).contiguous().transpose(2, 3)
    return x.contiguous()


LAYOUTS = ("head-major", "token-major", "slice", "misaligned", "strided")


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("h,d", [(2, 128), (3, 64)])
def test_write_and_read_are_bit_exact(dtype, layout, h, d):
    from latentserve_amd.kernels.hip import paged_gather as pg
    from latentserve_amd.runtime.kv_cache import KVCacheSpec, PagedKVCache
    c = PagedKVCache(KVCacheSpec(num_layers=1, num_kv_heads=h, head_dim=d, max_batch_size=3,
                                 max_seq_len=300, dtype=dtype, device="cuda"))
    g = torch.Generator(device="cuda").manual_seed(3)
    hist = [[], []]
    for n in (1, 2, 14, 33, 1, 129):               # starts 0, 1, 3, 17, 50, 51
        c.advance(n, slots=[0, 2])
        k, v = (torch.randn(2, h, n, d, generator=g, device="cuda").to(dtype) for _ in range(2))
        c.write(0, _layout(k, layout), _layout(v, layout))
        hist[0].append(k)
        hist[1].append(v)
    want = [torch.cat(x, dim=2) for x in hist]
    total = want[0].shape[2]
    got = c.read(0, 2)
    for z, pool in enumerate((c.k_pool[0], c.v_pool[0])):
        assert torch.equal(got[z], want[z])
        assert torch.equal(pg.gather(pool, c.block_tables_tensor(2), c.seq_lens_tensor(2),
                                     total), want[z])
        used = torch.zeros(pool.shape[0] * BS, dtype=torch.bool, device="cuda")
        for s in (0, 2):
            used[torch.tensor(c.tables[s].slots(0, total), device="cuda")] = True
        assert not pool.view(-1, h, d)[~used].any()


@pytest.mark.parametrize("asym", [False, True])
@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("chunks", [(2, 13, 2, 31, 16, 33), (16, 17, 15, 32), (15, 130, 2),
                                    (1, 15, 48, 1, 1, 3)])
@pytest.mark.parametrize("h", [1, 3])
def test_int8_chunks_equal_the_oracle(asym, layout, chunks, h):
    from latentserve_amd.runtime.int8_cache import Int8PagedKVCache
    from latentserve_amd.runtime.kv_cache import KVCacheSpec
    c = Int8PagedKVCache(KVCacheSpec(num_layers=1, num_kv_heads=h, head_dim=128,
                                     max_batch_size=4, max_seq_len=256, device="cuda"),
                         asymmetric=asym)
    g = torch.Generator(device="cuda").manual_seed(5)
    slots = [3, 1]
    c.advance(5, slots=[2])                        # another sequence's page first
    hist = [[], []]
    for n in chunks:
        c.advance(n, slots=slots)
        k, v = (torch.randn(2, h, n, 128, generator=g, device="cuda").half() for _ in range(2))
        v[0, 0, 0] = 0                             # a row at the scale's floor
        if n == 1:                                 # the decode write takes unit-stride rows
            c.write(0, k, v)
        else:
            c.write(0, _layout(k, layout), _layout(v, layout))
        hist[0].append(k)
        hist[1].append(v)
    k_all, v_all = (torch.cat(x, dim=2).transpose(1, 2).cpu().numpy() for x in hist)
    total = k_all.shape[1]
    last = (total - 1) // BS
    for i, s in enumerate(slots):
        t = c.tables[s]
        at = np.array(t.slots(0, total))
        codes, step, zero = oracle.quantize_v(np.ascontiguousarray(v_all[i]), asym=asym,
                                              recip=True)
        assert np.array_equal(c.v_pool[0].cpu().numpy().reshape(-1, h, 128)[at], codes)
        assert np.array_equal(c.v_scale_pool[0].cpu().numpy().reshape(-1, h)[at], step)
        if asym:
            assert np.array_equal(c.v_zero_pool[0].cpu().numpy().reshape(-1, h)[at], zero)
        if last:
            pages = np.ascontiguousarray(k_all[i, :last * BS]).reshape(last, BS, h, 128)
            codes, step, zero = oracle.quantize_k(pages, asym=asym, recip=True)
            blk = t.blocks[:last]
            assert np.array_equal(c.k_pool[0].cpu().numpy()[blk], codes)
            assert np.array_equal(c.k_scale_pool[0].cpu().numpy()[blk], step)
            if asym:
                assert np.array_equal(c.k_zero_pool[0].cpu().numpy()[blk], zero)
        res = c.residual(0)[s].cpu().numpy()
        assert np.array_equal(res[:total - last * BS], k_all[i, last * BS:])
        assert c.pooled_pages(s) == last


@pytest.mark.parametrize("asym", [False, True])
def test_int8_chunk_takes_ks_and_vs_own_eps(asym):
    """K's and V's quantizer constants apart, eps included: rows below V's floor
    but above K's, and the other way round."""
    from latentserve_amd.kernels.hip import int8_write as iw
    h, n, nb = 2, 40, 5
    g = torch.Generator(device="cuda").manual_seed(9)
    k, v = ((torch.randn(1, h, n, 128, generator=g, device="cuda") * 0.01).half()
            for _ in range(2))
    pool = lambda *shape, dtype=torch.float32: torch.zeros(*shape, dtype=dtype, device="cuda")
    kp, vp = (pool(nb, BS, h, 128, dtype=torch.int8) for _ in range(2))
    ks, kz, vs, vz = pool(nb, h, 128), pool(nb, h, 128), pool(nb, BS, h), pool(nb, BS, h)
    for k_eps, v_eps in ((1e-8, 0.5), (0.5, 1e-8)):
        iw.prefill_write(k, v, torch.arange(n, device="cuda").view(1, n),
                         torch.zeros(1, dtype=torch.long, device="cuda"), kp, ks, kz, vp, vs, vz,
                         pool(1, BS, h, 128, dtype=torch.float16), asym=asym,
                         k_quant=(k_eps, 127.0, 255.0, 128.0), v_quant=(v_eps, 7.0, 15.0, 8.0))
        rows = np.ascontiguousarray(v[0].transpose(0, 1).cpu().numpy())
        codes, step, zero = oracle.quantize_v(rows, asym=asym, eps=v_eps, bits=4, recip=True)
        assert np.array_equal(vp.view(-1, h, 128)[:n].cpu().numpy(), codes)
        assert np.array_equal(vs.view(-1, h)[:n].cpu().numpy(), step)
        pages = np.ascontiguousarray(k[0].transpose(0, 1)[:2 * BS].cpu().numpy())
        codes, step, kzero = oracle.quantize_k(pages.reshape(2, BS, h, 128), asym=asym, eps=k_eps,
                                               recip=True)
        assert np.array_equal(kp[:2].cpu().numpy(), codes)
        assert np.array_equal(ks[:2].cpu().numpy(), step)
        if asym:
            assert np.array_equal(vz.view(-1, h)[:n].cpu().numpy(), zero)
            assert np.array_equal(kz[:2].cpu().numpy(), kzero)


@pytest.mark.parametrize("which", ["k", "v"])
@pytest.mark.parametrize("first", [0, 16, 24])
def test_int8_chunk_read_from_the_residual(monkeypatch, which, first):
    """k or v that lies in the residual pool the launch stores to: a copy of it
    is what the kernel reads (the pointers that reach the library say so), and
    the result is that of the values as they were."""
    from latentserve_amd import _lib
    from latentserve_amd.kernels.hip import int8_write as iw
    h, n, nb, nr = 2, 37, 4, 4
    g = torch.Generator(device="cuda").manual_seed(first)
    # (the buffer: 16 rows, then the residual pool; the chunk starts at row `first`)
    buf = torch.randn((nr + 1) * BS, h, 128, generator=g, device="cuda").half()
    other = torch.randn(1, h, n, 128, generator=g, device="cuda").half()
    real, seen = _lib.lib(), []

    class Library:
        def __getattr__(self, name):
            def call(*args):
                seen.append((args[0], args[2]))
                return getattr(real, name)(*args)
            return call

    def run(apart):
        buf_ = buf.clone()
        chunk, res = buf_[first:first + n].transpose(0, 1)[None], buf_[BS:].view(nr, BS, h, 128)
        if apart:
            chunk = chunk.clone()
        k, v = (chunk, other) if which == "k" else (other, chunk)
        pool = lambda *shape, dtype=torch.float32: torch.zeros(*shape, dtype=dtype, device="cuda")
        out = [pool(nb, BS, h, 128, dtype=torch.int8), pool(nb, h, 128), None,
               pool(nb, BS, h, 128, dtype=torch.int8), pool(nb, BS, h), None, res]
        quant = (1e-8, 127.0, 255.0, 128.0)
        iw.prefill_write(k, v, torch.arange(5, 5 + n, device="cuda").view(1, n),
                         torch.ones(1, dtype=torch.long, device="cuda"), *out, asym=False,
                         k_quant=quant, v_quant=quant)
        lo, hi = res.data_ptr(), res.data_ptr() + res.numel() * 2
        return [t for t in out if t is not None], lo, hi

    want, _, _ = run(True)
    monkeypatch.setattr(_lib, "lib", lambda: Library())
    got, lo, hi = run(False)
    assert all(p >= hi or p + n * h * 256 <= lo for p in seen[-1]), "read where it stores"
    assert all(torch.equal(a, b) for a, b in zip(got, want))
