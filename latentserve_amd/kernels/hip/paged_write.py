"""New K and V rows scattered to their paged slots on a HIP kernel.

The write side of the fp16 paged cache (PagedKVCache.write,
cache/paged_cache.py: a transposed copy and an indexed store for K, again for
V): one launch that reads k and v where the projection left them, whatever
their batch, head and token strides, and stores each 16-byte piece at its slot.
"""

from __future__ import annotations

from typing import Optional, Tuple

import torch

from latentserve_amd import _lib

PAGE = 16


def write(k: torch.Tensor, v: torch.Tensor, slots: torch.Tensor, k_pool: torch.Tensor,
          v_pool: torch.Tensor,
          bounds: Optional[Tuple[torch.Tensor, torch.Tensor]] = None) -> bool:
    """k, v [B, H, n, D] to flat token slots [B * n] int64 of the contiguous
    pools [nb, 16, H, D]: a bit-exact copy.  With bounds (kmin, kmax [nb, H,
    128]), every block's K bounds are rebuilt after it (rebuild_bounds).

    False, with nothing done, where the kernel does not apply: CPU tensors,
    another type than the pools', rows that do not start on 16 bytes or whose
    channels are not adjacent, gradients to record, or rows whose span
    meets the pools (the order of the kernel's reads and stores is not
    defined)."""
    shape, pshape = k.shape, k_pool.shape
    b, h, n, d = shape
    size = k.element_size()
    ks, vs, ps = k.stride(), v.stride(), k_pool.stride()
    kp, vp, kpp, vpp = k.data_ptr(), v.data_ptr(), k_pool.data_ptr(), v_pool.data_ptr()
    pool_bytes = k_pool.numel() * size
    # (the bytes that k and v span, gaps between their rows included)
    k_end = kp + ((b - 1) * ks[0] + (h - 1) * ks[1] + (n - 1) * ks[2] + d) * size
    v_end = vp + ((b - 1) * vs[0] + (h - 1) * vs[1] + (n - 1) * vs[2] + d) * size
    k_pool_end, v_pool_end = kpp + pool_bytes, vpp + pool_bytes
    dev = k.device
    if not (dev.type == "cuda" and dev == v.device == k_pool.device == v_pool.device
            and k.dtype == v.dtype == k_pool.dtype == v_pool.dtype and size in (1, 2, 4)
            and shape == v.shape and pshape == v_pool.shape
            and ps == (PAGE * h * d, h * d, d, 1) == v_pool.stride()
            and pshape[1:] == (PAGE, h, d) and 0 < b <= 65535 and n > 0
            and ks[3] == 1 == vs[3]
            and not ((ks[0] | ks[1] | ks[2] | vs[0] | vs[1] | vs[2] | d) * size
                     | kp | vp | kpp | vpp) & 15
            and (kp >= k_pool_end or k_end <= kpp) and (kp >= v_pool_end or k_end <= vpp)
            and (vp >= k_pool_end or v_end <= kpp) and (vp >= v_pool_end or v_end <= vpp)
            and not (torch.is_grad_enabled() and (k.requires_grad or v.requires_grad))):
        return False
    if slots.dtype != torch.int64 or slots.shape != (b * n,) or slots.stride(0) != 1 \
            or slots.device != dev:
        raise ValueError(f"slots must be {b * n} unit-stride int64 values on k's device")
    kmin = kmax = bst = None
    if bounds is not None:
        lo, hi = bounds
        if k.dtype != torch.float16 or lo.dtype != torch.float16 or hi.dtype != torch.float16 \
                or lo.shape != (pshape[0], h, d) or hi.shape != lo.shape or lo.stride(-1) != 1 \
                or hi.stride() != lo.stride() or lo.device != dev or hi.device != dev:
            raise ValueError(f"bounds must be matching float16 [{pshape[0]}, {h}, {d}] tensors "
                             "with unit last stride")
        kmin, kmax, bst = lo.data_ptr(), hi.data_ptr(), _lib.strides(lo, 2)
    S = _lib.strides
    rc = _lib.lib().ls_paged_write(kp, S(k, 3), vp, S(v, 3), slots.data_ptr(), kpp, vpp,
                                   S(k_pool, 3), pshape[0], size, b, h, n, d, PAGE, kmin, kmax,
                                   bst, _lib.stream_of(dev))
    _lib.check(rc, "ls_paged_write")
    return True
