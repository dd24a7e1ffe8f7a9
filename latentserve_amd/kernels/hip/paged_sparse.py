"""Sparse (page-subset) decode attention on the HIP kernels.

Mirrors the reference's kernels/cuda/paged_sparse.py: ``budget`` (:74-78),
``rebuild_bounds`` (:81-84), ``update_bounds`` (:86-101), ``page_scores``
(:104-123), ``select`` (:164-168), ``budgets`` (:171-182), ``sparse_decode``
(:185-219) and ``sparse_attention`` (:222-251), all on HIP kernels.

Per layer per decode step ``sparse_attention`` with bounds scoring is one
launch (ls_sparse_attention_bounds_fp16, past COOP_MAX_PAGES pages a row
ls_sparse_attention_bounds_long_fp16): the page-subset decode's workgroups
score their shares of their sequence's pages, exchange the scores, and each
selects its own list by the selection kernel's rule (the same lists and
partition as index + select + sparse_decode).  Mass scoring, and bounds
scoring of more than COOP_MAX_NREP query rows a KV head or of many long rows
(_one_launch), are two launches (the scores, then ls_sparse_attention_fp16);
``fused=False`` runs the three (index, select, decode).  Nothing syncs with
the host, so the step is capturable in a HIP graph.
"""

from __future__ import annotations

import ctypes
import math
from typing import Optional

import torch

from latentserve_amd import _lib
from latentserve_amd.kernels.gqa import _scratch as scratch
from latentserve_amd.kernels.hip import paged_decode_hip as pdh

PAGE = pdh.PAGE
SELECT_MAX_PAGES = 8192
_LINE_FLOATS = 32          # one 128-byte line of fp32 scores per index group


def _check_bounds(kmin: torch.Tensor, kmax: torch.Tensor, device) -> None:
    if kmin.dtype != torch.float16 or kmax.dtype != torch.float16:
        raise ValueError("kmin/kmax must be float16 [num_blocks, H_kv, head_dim]")
    if kmin.dim() != 3 or kmin.shape != kmax.shape or kmin.stride() != kmax.stride() \
            or kmin.stride(-1) != 1:
        raise ValueError("kmin/kmax must match, [num_blocks, H_kv, head_dim], unit last stride")
    if kmin.device != device or kmax.device != device:
        raise ValueError("kmin/kmax must be on q's device")


def _score_buffer(b: int, h: int, max_pages: int, device) -> torch.Tensor:
    """Persistent [B, H, max_pages] fp32 view whose rows start on 128-byte
    lines (the fused index+select kernel's requirement)."""
    width = -(-max(1, max_pages) // _LINE_FLOATS) * _LINE_FLOATS
    buf = scratch("sparse_scores", (b, h, width), torch.float32, device)
    return buf[:, :, :max_pages]


def kernel_resources(device: Optional[torch.device] = None, n_rep: int = 6,
                     kv_heads: int = 2) -> dict:
    """Registers, private (spill) memory and LDS of each loaded page-subset
    kernel, by name (kernels/cuda/paged_sparse.py:254-265; the reference's
    four names plus this build's selection and one-launch kernels)."""
    names = ("page_bounds_update", "page_index", "page_index_heads", "paged_sparse_fp16",
             "page_mass", "page_select", "page_bounds_rebuild")
    # the selecting decodes: four score keys a thread, or (by the row's length)
    # two, eight or sixteen; the 4-wave form of many short rows
    names += tuple(f"{n}{keys}" for n in ("sparse_attention_fp16", "sparse_attention_bounds_fp16")
                   for keys in ("", "_4waves", "_keys2", "_keys8", "_keys16"))
    return {n: _lib.kernel_resources(n, device, kv_heads=kv_heads, n_rep=n_rep) for n in names}


def rebuild_bounds(k_pool: torch.Tensor, kmin: torch.Tensor, kmax: torch.Tensor) -> None:
    """Every block's per-channel K bounds from the pool, over all PAGE rows."""
    _check_bounds(kmin, kmax, k_pool.device)
    if k_pool.dtype != torch.float16 or k_pool.stride(-1) != 1:
        raise ValueError("k_pool must be float16 with unit last stride")
    nb, page, h, d = k_pool.shape
    if kmin.shape != (nb, h, d):
        raise ValueError(f"kmin/kmax must be [{nb}, {h}, {d}]")
    P, S = _lib.ptr, _lib.strides
    rc = _lib.lib().ls_page_bounds_rebuild(P(k_pool), S(k_pool, 3), nb, P(kmin), P(kmax),
                                           S(kmin, 2), h, d, page, _lib.stream_of(k_pool.device))
    _lib.check(rc, "ls_page_bounds_rebuild")


def update_bounds(k_new: torch.Tensor, slots: torch.Tensor, kmin: torch.Tensor,
                  kmax: torch.Tensor, page: int = 16) -> None:
    """k_new [B, H, D] (or [B, H, 1, D]) just written at flat `slots` [B]."""
    k = k_new.reshape(k_new.shape[0], k_new.shape[1], k_new.shape[-1])
    _check_bounds(kmin, kmax, k.device)
    if k.dtype != torch.float16 or k.stride(-1) != 1:
        raise ValueError("k_new must be float16 with unit last stride")
    if slots.dtype != torch.int64 or slots.dim() != 1 or slots.shape[0] != k.shape[0] \
            or slots.stride(0) != 1:
        raise ValueError("slots must be a contiguous int64 [B] tensor")
    b, h, d = k.shape
    P, S = _lib.ptr, _lib.strides
    rc = _lib.lib().ls_page_bounds_update(P(k), S(k, 2), P(slots), P(kmin), P(kmax), S(kmin, 2),
                                          kmin.shape[0], b, h, d, page,
                                          _lib.stream_of(k.device))
    _lib.check(rc, "ls_page_bounds_update")


def _check_index_inputs(q, kmin, kmax, block_tables, seq_lens):
    if q.dtype != torch.float16 or q.dim() != 4 or q.stride(-1) != 1:
        raise ValueError("q must be float16 [B, H_kv, n_rep, D] with unit last stride")
    _check_bounds(kmin, kmax, q.device)
    if block_tables.dtype != torch.int32 or seq_lens.dtype != torch.int32 \
            or block_tables.stride(-1) != 1 or seq_lens.stride(-1) != 1:
        raise ValueError("block tables and sequence lengths must be unit-stride int32")


def page_scores(q, kmin, kmax, block_tables, seq_lens, recent: int = 2) -> torch.Tensor:
    """-> [B, H, max_pages] fp32: bound per page, +inf forced, -inf past the end."""
    _check_index_inputs(q, kmin, kmax, block_tables, seq_lens)
    b, h, n_rep, d = q.shape
    max_pages = block_tables.shape[1]
    scores = _score_buffer(b, h, max_pages, q.device)
    P, S = _lib.ptr, _lib.strides
    rc = _lib.lib().ls_page_scores(
        P(q), S(q, 3), P(kmin), P(kmax), S(kmin, 2), kmin.shape[0], P(block_tables),
        block_tables.stride(0), max_pages, P(seq_lens), P(scores), S(scores, 2),
        b, h, n_rep, d, PAGE, int(recent), _lib.stream_of(q.device))
    _lib.check(rc, "ls_page_scores")
    return scores


def page_scores_mass(q, kmin, kmax, block_tables, seq_lens, recent: int = 2,
                     softmax_scale: Optional[float] = None, page: int = PAGE) -> torch.Tensor:
    """Summed-mass scores -> [B, H, max_pages] fp32 (kernels/cuda/
    paged_sparse.py:126-161): for each query head a softmax over the pages
    of bound * scale + log(tokens in the page), summed over the group; page
    0 and the last `recent` pages +inf, pages past the end -inf.  Two
    launches; the per-head logits go through a persistent workspace."""
    _check_index_inputs(q, kmin, kmax, block_tables, seq_lens)
    if page != PAGE:
        raise ValueError(f"the HIP indexer reads {PAGE}-token pages")
    b, h, n_rep, d = q.shape
    max_pages = block_tables.shape[1]
    scores = _score_buffer(b, h, max_pages, q.device)
    nbytes = _lib.lib().ls_page_mass_workspace_bytes(b, h, n_rep, max_pages)
    work = scratch("sparse_mass_heads", (max(1, nbytes // 4),), torch.float32, q.device)
    scale = softmax_scale if softmax_scale is not None else 1.0 / math.sqrt(d)
    P, S = _lib.ptr, _lib.strides
    rc = _lib.lib().ls_page_scores_mass(
        P(q), S(q, 3), P(kmin), P(kmax), S(kmin, 2), kmin.shape[0], P(block_tables),
        block_tables.stride(0), max_pages, P(seq_lens), P(work), P(scores), S(scores, 2),
        b, h, n_rep, d, PAGE, int(recent), float(scale), _lib.stream_of(q.device))
    _lib.check(rc, "ls_page_scores_mass")
    return scores


def select(scores: torch.Tensor, k: int, sorted: bool = False,
           seq_lens: Optional[torch.Tensor] = None, ratio: Optional[float] = None,
           recent: int = 2) -> torch.Tensor:
    """Top-k pages per (sequence, head) -> int32 [B, H, k].

    Ties between equal scores go to the lower page. ``sorted``: best first
    (forced +inf pages first, then by score). Unsorted, the pages come in
    page order; given ``seq_lens`` and ``ratio``, the first n_b entries of
    sequence b are then its own budget's best pages (what sparse_decode
    attends with that ratio) and the remaining k - n_b follow.
    """
    if scores.dtype != torch.float32 or scores.dim() != 3 or scores.stride(-1) != 1:
        raise ValueError("scores must be float32 [B, H, P] with unit last stride")
    b, h, p = scores.shape
    k = int(k)
    if not 0 <= k <= p:
        raise ValueError(f"k={k} out of range for {p} pages")
    if p > SELECT_MAX_PAGES:
        raise ValueError(f"select supports up to {SELECT_MAX_PAGES} pages, got {p}")
    use_ratio = ratio is not None and not sorted
    if use_ratio and (seq_lens is None or seq_lens.dtype != torch.int32):
        raise ValueError("a ratio needs int32 seq_lens")
    if k == 0 or b == 0:
        return torch.empty(b, h, k, dtype=torch.int32, device=scores.device)
    sel = scratch("sparse_select", (b, h, k), torch.int32, scores.device)
    P, S = _lib.ptr, _lib.strides
    rc = _lib.lib().ls_page_select(
        P(scores), S(scores, 2), P(seq_lens) if use_ratio else None, b, h, p, k,
        float(ratio) if use_ratio else 0.0, int(recent), 1 if sorted else 0, P(sel),
        (ctypes.c_int64 * 2)(*sel.stride()[:2]), _lib.stream_of(scores.device))
    _lib.check(rc, "ls_page_select")
    return sel


def index_select(q, kmin, kmax, block_tables, seq_lens, k: int, ratio: float,
                 recent: int = 2) -> torch.Tensor:
    """page_scores + select(ratio=...) -> int32 [B, H, k] (two launches)."""
    _check_index_inputs(q, kmin, kmax, block_tables, seq_lens)
    b, h, n_rep, d = q.shape
    max_pages = block_tables.shape[1]
    if max_pages > SELECT_MAX_PAGES:
        raise ValueError(f"selection supports up to {SELECT_MAX_PAGES} pages, got {max_pages}")
    k = int(k)
    if not 1 <= k <= max_pages:
        raise ValueError(f"k={k} out of range for {max_pages} pages")
    scores = _score_buffer(b, h, max_pages, q.device)
    sel = scratch("sparse_index_sel", (b, h, k), torch.int32, q.device)
    P, S = _lib.ptr, _lib.strides
    rc = _lib.lib().ls_sparse_index(
        P(q), S(q, 3), P(kmin), P(kmax), S(kmin, 2), kmin.shape[0], P(block_tables),
        block_tables.stride(0), max_pages, P(seq_lens), P(scores), S(scores, 2), None, k,
        float(ratio), int(recent), P(sel), S(sel, 2), b, h, n_rep, d, PAGE,
        _lib.stream_of(q.device))
    _lib.check(rc, "ls_sparse_index")
    return sel


def budget(ratio: float, max_pages: int, recent: int = 2) -> int:
    """List width for a context of max_pages pages: ceil(ratio x pages),
    never fewer than page 0 plus the `recent` forced pages, never more than
    the pages there are (paged_sparse.py:74-78)."""
    if ratio >= 1.0:
        return max_pages
    return min(max_pages, max(recent + 1, math.ceil(ratio * max_pages)))


def budgets(seq_lens: torch.Tensor, ratio: float, recent: int = 2, page: int = 16) -> torch.Tensor:
    """int32 [B]: how many pages each sequence attends at its present
    length (paged_sparse.py:171-182).  The same product the kernels form in
    fp32 with ceilf, so host and device agree on every length; raised to
    recent + 1, cut to the sequence's pages.  The kernels compute it
    themselves: this is for callers and tests."""
    pages = (seq_lens.to(torch.int64) + page - 1) // page
    if ratio >= 1.0:
        return pages.to(torch.int32)
    prod = torch.tensor(ratio, dtype=torch.float32, device=pages.device) * pages.to(torch.float32)
    n = torch.ceil(prod).to(torch.int64).clamp(min=recent + 1)
    return torch.minimum(n, pages).to(torch.int32)


# Pages a split of the list walk up to which its groups are one round: over equal
# lengths one is the fastest, over ragged ones a long sequence's few groups run
# on alone, and two rounds of smaller groups lose little to either.  (us, full /
# ragged lengths, one round -> two, with the count by the CUs alone, a round and a
# few groups more, in parentheses: B17 x 8 heads, 500 pages 94 / 56 -> 99 / 45 (126 /
# 49), B40 x 8, 250 pages 114 / 88 -> 115 / 69 (135 / 72), B70 x 4, 125 pages 55 /
# 47 -> 58 / 40 (69 / 40); 79 to 83 pages a split: B33 x 8 34 / 29 -> 39 / 28 (47 /
# 30), B17 x 8 49 / 40 -> 53 / 40 (67 / 36).)
LIST_ROUND_PAGES = 96


def sparse_decode(q, k_pool, v_pool, block_tables, seq_lens, sel,
                  num_splits: Optional[int] = None,
                  softmax_scale: Optional[float] = None,
                  ratio: Optional[float] = None, recent: int = 2,
                  out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Attention over the pages in `sel` [B, H, K] only -> [B, H, n_rep, D]
    (into `out` when given, as paged_decode_hip).

    With `ratio`, each sequence attends the first max(recent+1,
    ceil(ratio*pages)) entries of its (score-sorted) list for its current
    length, counted on the device; entries past a sequence's end are skipped.
    """
    reason = pdh.ineligible_reason(q, k_pool)
    if reason is None and k_pool.dtype != torch.float16:
        reason = "the page-subset kernel reads fp16 pools"
    if reason is not None:
        raise ValueError(f"sparse_decode: {reason}")
    pdh._check_common(q, k_pool, v_pool, block_tables, seq_lens)
    if sel.dtype != torch.int32 or sel.dim() != 3 or sel.stride(-1) != 1:
        raise ValueError("sel must be an int32 [B, H, K] tensor with unit last stride")
    b, h, n_rep, d = q.shape
    num_sel = sel.shape[-1]
    splits = num_splits or pdh.choose_splits(b, h, num_sel, q.device, dealt=False,
                                             round_pages=LIST_ROUND_PAGES)
    splits = max(1, min(splits, max(1, num_sel), pdh.MAX_SPLITS))
    scale = softmax_scale if softmax_scale is not None else 1.0 / math.sqrt(d)
    buf, work, cnt = pdh._buffers("sparse", b, h, splits, n_rep, q.device)
    target = buf if out is None else pdh.check_out(out, q)
    P, S = _lib.ptr, _lib.strides
    rc = _lib.lib().ls_paged_sparse_fp16(
        P(q), S(q, 3), P(k_pool), P(v_pool), S(k_pool, 3), k_pool.shape[0],
        P(block_tables), block_tables.stride(0), block_tables.shape[1], P(seq_lens),
        P(sel), S(sel, 2), num_sel, 0.0 if ratio is None else float(ratio), int(recent),
        P(target), S(target, 3), P(work), P(cnt), b, h, n_rep, d, k_pool.shape[1],
        splits, 0, float(scale), _lib.stream_of(q.device))
    _lib.check(rc, "ls_paged_sparse_fp16")
    return buf[:, :, :n_rep] if out is None else out


SELECT_SPLIT_ENTRIES = 1024    # list entries a selecting group keeps (a split's share)
# the one-launch bounds path: bounds of as many blocks as the pools and at most
# this many query rows a KV head (else the index kernel, then the selecting
# decode); past this many pages a row, its entry for long rows
COOP_MAX_PAGES = 2048
COOP_MAX_NREP = 8
# A selecting group a CU.  In one launch a row's scores are the work of its own
# groups, 160 pages in one batch of loads; in two the index kernel spreads every
# row over the chip, which a short row's groups would leave idle.  So one launch
# up to a batch a group, and up to COOP_MAX_PAGES where the rows are few enough
# that the launch it saves counts.  (us, ratio 0.25, full / ragged lengths, one
# launch -> two: B12 x 8 heads to 8000 34.1 / 29.6 -> 32.4 / 27.2, B17 x 8 to
# 5000 34.0 / 31.6 -> 30.2 / 27.2, to 32000 176 / 134 -> 142 / 99, B32 x 8 to
# 16000 121 / 89 -> 116 / 82, B8 x 8 to 100K 190 / 127 -> 180 / 109; under a
# batch, B16 x 8 to 1500 15.6 / 14.4 -> 17.0 / 16.1, B24 x 8 to 2500 22.8 / 20.5 ->
# 23.3 / 20.4, B32 x 8 to 2500 25.2 / 21.4 -> 26.5 / 21.7.)
# The second launch is 12 us of host work, which calls outside a graph spend: only
# with pages enough in all rows to take longer than that on the GPU.
SELECT_GROUPS = 256
SCORE_BATCH = 160
FEW_ROWS = 64
TWO_LAUNCH_MIN_PAGES = 40000
# In two launches the groups need not be resident together: where the whole groups
# a row that are leave CUs idle (129 to 170 rows: one, on up to half of them), two
# rounds of an odd count fill them, from this many selected pages a group on (us,
# full / ragged lengths, B17 x 8 heads, one -> three groups: 125 pages 43.1 /
# 37.6 -> 47.5 / 36.0, 250 79.5 / 68.0 -> 75.9 / 60.5, 500 142 / 99 -> 136 / 71;
# B12 x 8, two -> five: 625 pages 118 / 97 -> 121 / 86).
TWO_ROUNDS_MIN_PAGES = 160


def _one_launch(rows: int, width: int) -> bool:
    """Whether the groups of `rows` (sequence, KV head) rows of `width` pages score
    the pages themselves."""
    share = -(-width // max(1, SELECT_GROUPS // max(1, rows)))
    return (share <= SCORE_BATCH or rows * width < TWO_LAUNCH_MIN_PAGES
            or (rows <= FEW_ROWS and width <= COOP_MAX_PAGES))


def _two_rounds(rows: int, k: int) -> int:
    """Splits of the two-launch path's lists of k pages in two rounds of groups, 0
    where one round is as good."""
    fit, two = (n * SELECT_GROUPS // max(1, rows) for n in (1, 2))
    return two if 1 <= fit < 4 and two > 2 * fit and k >= TWO_ROUNDS_MIN_PAGES * fit else 0


def sparse_attention(q, k_pool, v_pool, block_tables, seq_lens, kmin, kmax,
                     ratio: float = 0.25, recent: int = 2,
                     num_splits: Optional[int] = None, max_seq_len: Optional[int] = None,
                     softmax_scale: Optional[float] = None,
                     scoring: str = "bounds",
                     out: Optional[torch.Tensor] = None, fused: bool = True) -> torch.Tensor:
    """Index, select, attend. The list width k follows `max_seq_len` (the
    context) when given, else the table's width; each sequence then attends
    its own budget for its current length.  Fused, bounds scoring is one
    launch (the decode's workgroups score, select and attend), or two as mass
    scoring (the scores, then a decode that selects); ``fused=False``
    runs index, select and decode as three."""
    if scoring not in ("bounds", "mass"):
        raise ValueError(f"unknown scoring {scoring!r} (bounds or mass)")
    page = k_pool.shape[1]
    pages = block_tables.shape[1] if max_seq_len is None else min(
        block_tables.shape[1], -(-int(max_seq_len) // page))
    k = budget(ratio, pages, recent)
    if not fused:
        if scoring == "mass":
            mass = page_scores_mass(q, kmin, kmax, block_tables, seq_lens, recent, softmax_scale)
            sel = select(mass, k, seq_lens=seq_lens, ratio=ratio, recent=recent)
        else:
            sel = index_select(q, kmin, kmax, block_tables, seq_lens, k, ratio, recent)
        return sparse_decode(q, k_pool, v_pool, block_tables, seq_lens, sel, num_splits,
                             softmax_scale, ratio=ratio, recent=recent, out=out)
    reason = pdh.ineligible_reason(q, k_pool)
    if reason is None and k_pool.dtype != torch.float16:
        reason = "the page-subset kernel reads fp16 pools"
    if reason is not None:
        raise ValueError(f"sparse_attention: {reason}")
    pdh._check_common(q, k_pool, v_pool, block_tables, seq_lens)
    if block_tables.shape[1] > SELECT_MAX_PAGES:
        raise ValueError(f"selection supports up to {SELECT_MAX_PAGES} pages, "
                         f"got {block_tables.shape[1]}")
    b, h, n_rep, d = q.shape
    # (a selecting group serves one head: as many groups as a pair of heads makes
    # elsewhere, so the count is asked for twice the heads)
    splits = num_splits or pdh.choose_splits(b, 2 * h, k, q.device, dealt=False)
    splits = max(1, min(splits, max(1, k), pdh.MAX_SPLITS))
    # (bounds that cover another number of blocks than the pools: the index
    # kernel, which takes the bounds' own count; the one launch has one count
    # for both, and would read past the end of shorter bounds)
    one = (scoring == "bounds" and n_rep <= COOP_MAX_NREP and kmin.shape[0] == k_pool.shape[0]
           and _one_launch(b * h, block_tables.shape[1]))
    if not num_splits and not one:
        splits = max(splits, _two_rounds(b * h, k))
    splits = max(splits, -(-k // SELECT_SPLIT_ENTRIES))
    scale = softmax_scale if softmax_scale is not None else 1.0 / math.sqrt(d)
    buf, work, cnt = pdh._buffers("sparse", b, h, splits, n_rep, q.device)
    target = buf if out is None else pdh.check_out(out, q)
    P, S = _lib.ptr, _lib.strides
    short = block_tables.shape[1] <= COOP_MAX_PAGES
    if one:
        # one launch: the decode's workgroups score the pages themselves,
        # exchanging the scores through a buffer whose count words are all
        # ones at rest
        _check_bounds(kmin, kmax, q.device)
        # (each row is followed by one word: the count of its scored shares; rows
        # padded to 16 bytes, so a row starts 16-byte aligned.  A buffer a width:
        # in one of several widths, the word one counts in holds a score of
        # another)
        width = block_tables.shape[1]
        ws = scratch(("sparse_coop_scores", width), (b, h, (width + 4) // 4 * 4), torch.int32,
                     q.device, init=-1)
        entry = "ls_sparse_attention_bounds_fp16" if short else "ls_sparse_attention_bounds_long_fp16"
        rc = getattr(_lib.lib(), entry)(
            P(q), S(q, 3), P(k_pool), P(v_pool), S(k_pool, 3), k_pool.shape[0],
            P(block_tables), block_tables.stride(0), block_tables.shape[1], P(seq_lens),
            P(kmin), P(kmax), S(kmin, 2), P(ws), S(ws, 2), k, float(ratio), int(recent),
            P(target), S(target, 3), P(work), P(cnt), b, h, n_rep, d, page,
            splits, 0, float(scale), _lib.stream_of(q.device))
        _lib.check(rc, entry)
        return buf[:, :, :n_rep] if out is None else out
    if scoring == "mass":
        scores = page_scores_mass(q, kmin, kmax, block_tables, seq_lens, recent, softmax_scale)
    else:
        scores = page_scores(q, kmin, kmax, block_tables, seq_lens, recent)
    rc = _lib.lib().ls_sparse_attention_fp16(
        P(q), S(q, 3), P(k_pool), P(v_pool), S(k_pool, 3), k_pool.shape[0],
        P(block_tables), block_tables.stride(0), block_tables.shape[1], P(seq_lens),
        P(scores), S(scores, 2), scores.shape[2], k, float(ratio), int(recent),
        P(target), S(target, 3), P(work), P(cnt), b, h, n_rep, d, page,
        splits, 0, float(scale), _lib.stream_of(q.device))
    _lib.check(rc, "ls_sparse_attention_fp16")
    return buf[:, :, :n_rep] if out is None else out
