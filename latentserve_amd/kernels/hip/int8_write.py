"""INT8 KV cache write side on HIP kernels.

Mirrors the reference's kernels/cuda/int8_write.py: ``eligible`` (:53-58) and
``decode_write`` (:61-82), the fused decode-step write (V's per-token
quantize and scatter, K's scatter into the fp16 last-page residual), plus
``finalize_blocks``, the per-block K quantizer of
Int8PagedKVCache._finalize_blocks (cache/int8_paged_cache.py:670-699), so a
completed page is quantized on the GPU too, and ``prefill_write``, a whole
prefill chunk's write in one launch.

Codes and scales are bit-exact with the reference's torch ops.  Torch
divides by a Python number differently on the two devices (GPU: times the
fp32 reciprocal formed on the host; CPU: a true division); ``exact_division``
picks the CPU form, the default is the GPU form, which is what the reference
stores when it runs on a GPU and what its int8_write.cu computes.
"""

from __future__ import annotations

import ctypes
from typing import Optional

import torch

from latentserve_amd import _lib

HEAD_DIM = 128
PAGE = 16
_I64x3 = ctypes.c_int64 * 3


def eligible(k: torch.Tensor, v: torch.Tensor) -> bool:
    """One token per sequence, fp16, head_dim 128, channels unit-stride."""
    return (k.is_cuda and v.is_cuda and k.dtype == v.dtype == torch.float16
            and k.dim() == 4 and v.dim() == 4 and k.shape[2] == 1 and v.shape[2] == 1
            and k.shape[-1] == HEAD_DIM and v.shape[-1] == HEAD_DIM
            and k.stride(-1) == 1 and v.stride(-1) == 1)


def _contig(t: torch.Tensor, name: str) -> None:
    if not t.is_contiguous():
        raise ValueError(f"{name} must be contiguous")


def _on_device(first: torch.Tensor, *others: Optional[torch.Tensor]) -> None:
    dev = first.get_device()
    for t in others:
        if t is not None and t.get_device() != dev:
            raise ValueError(f"all tensors must be on one device, got {first.device} and "
                             f"{t.device}")


def decode_write(k, v, slots, res_idx, flat_v, flat_v_scale, flat_v_zero, k_res, *,
                 asym: bool, eps: float, qmax: float, levels: float, offset: float,
                 exact_division: bool = False) -> None:
    """k, v [B, H, 1, D] fp16; slots, res_idx [B] int64 flat indices;
    flat_v [S, H, D] int8, flat_v_scale / flat_v_zero [S, H] fp32;
    k_res [R, H, D] fp16.  Rows outside [0, S) / [0, R) are skipped."""
    if not eligible(k, v):
        raise ValueError("decode_write: k and v must be fp16 [B, H, 1, 128] GPU tensors")
    b, h, _, d = k.shape
    for t, name in ((slots, "slots"), (res_idx, "res_idx")):
        if t.dtype != torch.int64 or t.dim() != 1 or t.shape[0] < b or t.stride(0) != 1:
            raise ValueError(f"{name} must be a unit-stride int64 [B] tensor")
    if flat_v.dtype != torch.int8 or flat_v.shape[1:] != (h, d):
        raise ValueError("flat_v must be int8 [S, H, D]")
    if flat_v_scale.dtype != torch.float32 or flat_v_scale.shape != flat_v.shape[:2]:
        raise ValueError("flat_v_scale must be fp32 [S, H]")
    if asym and (flat_v_zero is None or flat_v_zero.shape != flat_v_scale.shape
                 or flat_v_zero.dtype != torch.float32):
        raise ValueError("asymmetric quantization needs flat_v_zero fp32 [S, H]")
    if k_res.dtype != torch.float16 or k_res.shape[1:] != (h, d):
        raise ValueError("k_res must be fp16 [R, H, D]")
    for t, name in ((flat_v, "flat_v"), (flat_v_scale, "flat_v_scale"), (k_res, "k_res")):
        _contig(t, name)
    if asym:
        _contig(flat_v_zero, "flat_v_zero")
    P, S = _lib.ptr, _lib.strides
    k2, v2 = k[:, :, 0], v[:, :, 0]
    rc = _lib.lib().ls_int8_decode_write(
        P(k2), S(k2, 2), P(v2), S(v2, 2), P(slots), P(res_idx), P(flat_v), P(flat_v_scale),
        P(flat_v_zero) if asym else None, P(k_res), flat_v.shape[0], k_res.shape[0], b, h, d,
        int(bool(asym)), float(eps), float(qmax), float(levels), float(offset),
        0 if exact_division else 1, _lib.stream_of(k.device))
    _lib.check(rc, "ls_int8_decode_write")


def finalize_blocks(data: torch.Tensor, ids: torch.Tensor, k_pool: torch.Tensor,
                    k_scale: torch.Tensor, k_zero: Optional[torch.Tensor] = None, *,
                    asym: bool, eps: float, qmax: float, levels: float, offset: float,
                    exact_division: bool = False, rows: Optional[torch.Tensor] = None) -> None:
    """Quantize data [N, 16, H, D] fp16 into k_pool blocks ids [N] (int64):
    one step per (block, head, channel), written to k_scale [nb, H, D] (and
    the zero point to k_zero when asym).  Ids outside the pool are skipped.
    With rows (int64, one an id), item i is data[rows[i]]."""
    if data.dtype != torch.float16 or data.dim() != 4 or data.shape[1] != PAGE \
            or data.shape[-1] != HEAD_DIM or data.stride(-1) != 1:
        raise ValueError("data must be fp16 [N, 16, H, 128] with unit channel stride")
    _, _, h, d = data.shape
    n = data.shape[0] if rows is None else ids.shape[0]
    if rows is not None and (rows.dtype != torch.int64 or rows.shape != (n,)
                             or rows.stride(0) != 1):
        raise ValueError("rows must be a unit-stride int64 tensor, one an id")
    if ids.dtype != torch.int64 or ids.dim() != 1 or ids.shape[0] != n or ids.stride(0) != 1:
        raise ValueError("ids must be a unit-stride int64 [N] tensor")
    if k_pool.dtype != torch.int8 or k_pool.shape[1:] != (PAGE, h, d) or k_pool.stride(-1) != 1:
        raise ValueError("k_pool must be int8 [nb, 16, H, D]")
    nb = k_pool.shape[0]
    if k_scale.dtype != torch.float32 or k_scale.shape != (nb, h, d) or k_scale.stride(-1) != 1:
        raise ValueError("k_scale must be fp32 [nb, H, D]")
    if asym and (k_zero is None or k_zero.shape != k_scale.shape
                 or k_zero.stride() != k_scale.stride() or k_zero.dtype != torch.float32):
        raise ValueError("asymmetric quantization needs k_zero shaped and strided as k_scale")
    _on_device(data, ids, k_pool, k_scale, k_zero if asym else None, rows)
    P, S = _lib.ptr, _lib.strides
    src = (P(data), S(data, 3)) if rows is None else (P(data), S(data, 3), P(rows), data.shape[0])
    L = _lib.lib()
    rc = (L.ls_int8_finalize_blocks if rows is None else L.ls_int8_finalize_rows)(
        *src, P(ids), n, P(k_pool), S(k_pool, 3), P(k_scale),
        P(k_zero) if asym else None, S(k_scale, 2), nb, h, d, PAGE, int(bool(asym)), float(eps),
        float(qmax), float(levels), float(offset), 0 if exact_division else 1,
        _lib.stream_of(data.device))
    _lib.check(rc, "ls_int8_finalize_blocks" if rows is None else "ls_int8_finalize_rows")


def prefill_write(k, v, slots, rows, k_pool, k_scale, k_zero, v_pool, v_scale, v_zero, k_res, *,
                  asym: bool, k_quant, v_quant, exact_division: bool = False) -> None:
    """A chunk's k, v [B, H, n, 128] fp16 at flat slots [B, n] int64 (each
    sequence's in token order): V quantized into v_pool [nb, 16, H, D] /
    v_scale [nb, 16, H]; K's complete pages into k_pool / k_scale [nb, H, D],
    its last page to row rows[b] (int64 [B]) of k_res [R, 16, H, D] (where the
    rows before the chunk in its first page are).  k_quant, v_quant: (eps,
    qmax, levels, offset).  One launch."""
    shape = k.shape
    b, h, n, d = shape
    dev = k.get_device()                      # (-1: not on a GPU)
    if dev < 0 or v.get_device() != dev or k.dtype != torch.float16 or v.dtype != torch.float16 \
            or d != HEAD_DIM or v.shape != shape:
        raise ValueError("prefill_write: k and v must be fp16 [B, H, n, 128] GPU tensors")
    if slots.dtype != torch.int64 or slots.shape != (b, n) or not slots.is_contiguous() \
            or slots.get_device() != dev:
        raise ValueError("slots must be a contiguous int64 [B, n] tensor on k's device")
    if rows.dtype != torch.int64 or rows.dim() != 1 or rows.numel() < b or rows.stride() != (1,) \
            or rows.get_device() != dev:
        raise ValueError("rows must be a unit-stride int64 [B] tensor on k's device")
    nb, nr = k_pool.shape[0], k_res.shape[0]
    i8, f32 = torch.int8, torch.float32
    pools = [(k_pool, "k_pool", i8, (nb, PAGE, h, d)), (v_pool, "v_pool", i8, (nb, PAGE, h, d)),
             (k_scale, "k_scale", f32, (nb, h, d)), (v_scale, "v_scale", f32, (nb, PAGE, h)),
             (k_res, "k_res", torch.float16, (nr, PAGE, h, d))]
    if asym:
        if k_zero is None or v_zero is None:
            raise ValueError("asymmetric quantization needs k_zero and v_zero")
        pools += [(k_zero, "k_zero", f32, (nb, h, d)), (v_zero, "v_zero", f32, (nb, PAGE, h))]
    for t, name, dt, like in pools:
        if t.dtype != dt or t.shape != like or not t.is_contiguous() or t.get_device() != dev:
            raise ValueError(f"{name} must be contiguous {dt} {like} on k's device")
    res = k_res.data_ptr()
    res_end = res + 2 * nr * PAGE * h * d
    k, ks = _loadable(k, shape, 4, res, res_end)
    v, vs = _loadable(v, shape, 16, res, res_end)
    eps, qmax, levels, offset = k_quant
    v_eps, v_qmax, v_levels, v_offset = v_quant
    rc = _lib.lib().ls_int8_prefill_write(
        k.data_ptr(), ks, v.data_ptr(), vs, slots.data_ptr(), rows.data_ptr(),
        k_pool.data_ptr(), k_scale.data_ptr(), k_zero.data_ptr() if asym else None,
        v_pool.data_ptr(), v_scale.data_ptr(), v_zero.data_ptr() if asym else None,
        res, nb, nr, b, h, n, d, PAGE, int(bool(asym)), eps, qmax, levels, offset,
        0 if exact_division else 1, v_eps, v_qmax, v_levels, v_offset, _lib.stream_of(k.device))
    _lib.check(rc, "ls_int8_prefill_write")


def _loadable(t: torch.Tensor, shape, nbytes: int, lo: int, hi: int):
    """t, or a contiguous copy where its rows are not unit-stride and aligned to
    the kernel's loads or its span meets the bytes [lo, hi) that the launch
    stores to; and its first three strides."""
    sb, sh, st, sd = t.stride()
    p = t.data_ptr()
    b, h, n, d = shape
    if sd != 1 or (p | 2 * (sb | sh | st)) % nbytes \
            or p < hi and lo < p + 2 * ((b - 1) * sb + (h - 1) * sh + (n - 1) * st + d):
        t = t.clone(memory_format=torch.contiguous_format)
        sb, sh, st, _ = t.stride()
    return t, _I64x3(sb, sh, st)
