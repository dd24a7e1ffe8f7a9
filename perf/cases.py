"""The measured cases: what a serving program has this framework do.

A case is a dict of plain values.  ``listed()`` names twelve that span the
range, ``draw(rng)`` gives more of the same ranges, ``prepare`` makes what the
program holds before the call, ``run`` is one pass through the public entry
points, ``exact`` the same result in 64 bits by plain torch.  Kinds of work:

attention   one decode step's paged attention over every layer's pool (fp16,
            symmetric INT8, or asymmetric INT8 with the token's quantized
            write before it), replayed from a HIP graph as the serving loop
            replays it
sparse      the same step attending a page budget (score, select, attend)
prefill     a prompt's K/V written to the paged cache in two chunks, all
            layers (fp16 with page bounds kept and the cache read back, or
            quantized to INT8)
layer       a decoder layer's products, norms and RoPE at decode batch sizes
rows        the fused elementwise ops over a prompt's rows
step        a whole captured decode step of the 28-layer decoder

Sequences sit on scattered pages (a seeded permutation of the pool), as after
some time of serving.
"""

from __future__ import annotations

import math

import torch

from latentserve_amd.kernels import decode_gemm as dg
from latentserve_amd.kernels import fused_elementwise as fe
from latentserve_amd.kernels.gqa.paged_decode import choose_num_splits
from latentserve_amd.kernels.hip import int8_write as iw
from latentserve_amd.kernels.hip import paged_decode_hip as pdh
from latentserve_amd.kernels.hip import paged_sparse as ps
from latentserve_amd.runtime.hip_graph import CapturedDecode
from latentserve_amd.runtime.int8_cache import Int8PagedKVCache
from latentserve_amd.runtime.kv_cache import KVCacheSpec, PagedKVCache
from latentserve_amd.runtime.qwen_decoder import HIP_GEMM_MAX_ROWS, DecoderConfig, QwenDecoder

PAGE, D = 16, 128
EPS = 1e-8          # floor of an INT8 scale
NORM_EPS = 1e-6
DEV = "cuda"


def listed():
    return [
        # one user's chat at a short context: launches and latency
        dict(name="fp16 b1 2k", kind="attention", kv="fp16", batch=1, ctx=2048, ragged=False,
             kv_heads=2, n_rep=6, layers=28),
        # the repository's headline workload
        dict(name="fp16 b16 16k", kind="attention", kv="fp16", batch=16, ctx=16384, ragged=False,
             kv_heads=2, n_rep=6, layers=28),
        # a busy server's chats: many short sequences of all lengths, wider KV
        dict(name="fp16 b48 ragged 1.5k", kind="attention", kv="fp16", batch=48, ctx=1531,
             ragged=True, kv_heads=8, n_rep=4, layers=16),
        # the INT8 cache at the headline shape, the token's write included
        dict(name="int8 b16 16k", kind="attention", kv="int8", batch=16, ctx=16384, ragged=False,
             kv_heads=2, n_rep=6, layers=28),
        # asymmetric INT8, a few documents of different lengths
        dict(name="int8z b5 ragged 11k", kind="attention", kv="int8z", batch=5, ctx=11003,
             ragged=True, kv_heads=4, n_rep=7, layers=28),
        # half of the pages at the longest context bucket
        dict(name="sparse b8 32k", kind="sparse", batch=8, ctx=32768, ragged=False, kv_heads=2,
             n_rep=6, layers=28, ratio=0.5, scoring="bounds"),
        # a quarter of the pages (the default ratio) of very long documents
        dict(name="sparse b2 100k", kind="sparse", batch=2, ctx=100003, ragged=False, kv_heads=2,
             n_rep=6, layers=16, ratio=0.25, scoring="bounds"),
        # prompts arriving: a batch of four, bounds kept for sparse decoding
        dict(name="prefill fp16 4x2048", kind="prefill", kv="fp16", batch=4, tokens=2048,
             chunk=1024, kv_heads=2, layers=28, bounds=True),
        # one odd prompt into the INT8 cache, its second chunk starting in a page
        dict(name="prefill int8 1x1021", kind="prefill", kv="int8", batch=1, tokens=1021,
             chunk=517, kv_heads=2, layers=28, bounds=False),
        # the products of a layer for a batch of 48 tokens
        dict(name="layer m48", kind="layer", rows=48, hidden=1536, inter=8960, q_heads=12,
             kv_heads=2, layers=8),
        # the elementwise ops of one layer over a prompt
        dict(name="rows 4099", kind="rows", rows=4099, hidden=1536, inter=8960, q_heads=12,
             kv_heads=2),
        # the whole decode step of the reference's full-step configuration
        dict(name="step b16 8k", kind="step", batch=16, ctx=8192, layers=28),
    ]


GEOMETRIES = ((2, 6), (2, 6), (4, 7), (8, 4), (1, 8), (2, 7), (3, 5))
# one step's K and V bytes over all layers at most (the headline's)
MAX_STEP_BYTES = 28 * 16 * 16384 * 2 * 2 * D * 2


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("attention", "attention", "attention", "sparse", "sparse", "prefill",
                       "prefill", "layer", "layer", "rows", "step"))
    if kind in ("attention", "sparse"):
        kv_heads, n_rep = rng.choice(GEOMETRIES)
        case = dict(kind=kind, ragged=rng.random() < 0.6, kv_heads=kv_heads, n_rep=n_rep)
        if kind == "attention":
            case["kv"] = rng.choice(("fp16", "fp16", "int8", "int8z"))
            case["batch"] = _log_int(rng, 1, 128)
            most = min(32768, 262144 * 2 // (case["batch"] * kv_heads))
            case["ctx"] = _log_int(rng, min(100, most // 2), most)
        else:
            case["ratio"] = rng.choice((0.125, 0.25, 0.5))
            case["scoring"] = rng.choice(("bounds", "bounds", "mass"))
            case["batch"] = _log_int(rng, 1, 32)
            most = min(131072, 262144 * 2 // (case["batch"] * kv_heads))
            case["ctx"] = _log_int(rng, 1000, most)
        layer = case["batch"] * case["ctx"] * kv_heads * D * 4
        case["layers"] = max(1, min(28, MAX_STEP_BYTES // (2 * layer)))
        return case
    if kind == "prefill":
        batch = rng.choice((1, 1, 1, 2, 3, 5, 8))
        tokens = _log_int(rng, 40, 8192 // batch)
        return dict(kind=kind, kv=rng.choice(("fp16", "int8", "int8z")), batch=batch,
                    tokens=tokens, chunk=rng.randint(tokens // 3 + 1, tokens - 2),
                    kv_heads=rng.choice((2, 2, 4, 8)), layers=rng.choice((8, 16, 28)),
                    bounds=rng.random() < 0.4)
    if kind == "layer":
        hidden, inter, q_heads, kv_heads = rng.choice(
            ((1536, 8960, 12, 2), (1024, 2816, 8, 4), (2048, 5632, 16, 2), (896, 4864, 7, 1)))
        return dict(kind=kind, rows=_log_int(rng, 1, 64), hidden=hidden, inter=inter,
                    q_heads=q_heads, kv_heads=kv_heads, layers=8)
    if kind == "rows":
        hidden, inter, q_heads, kv_heads = rng.choice(
            ((1536, 8960, 12, 2), (1024, 2816, 8, 4), (3584, 18944, 28, 4), (2048, 5632, 16, 2)))
        return dict(kind=kind, rows=_log_int(rng, 70, 8192), hidden=hidden, inter=inter,
                    q_heads=q_heads, kv_heads=kv_heads)
    batch = _log_int(rng, 1, 48)
    return dict(kind="step", batch=batch, ctx=_log_int(rng, 200, min(8192, 131072 // batch)),
                layers=28)


# ---------------------------------------------------------------------------
# inputs (plain torch, shared by prepare and exact)
# ---------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape, dtype=torch.float16, std=1.0):
    t = torch.empty(*shape, dtype=dtype, device=DEV)
    t.normal_(0.0, std, generator=g)
    return t


def _lengths(case):
    """Each sequence's tokens: the context, or spread over [ctx / 32, ctx]
    with the longest at the context (fixed by the case, so work() knows them)."""
    b, ctx = case["batch"], case["ctx"]
    if not case.get("ragged"):
        return [ctx] * b
    g = torch.Generator().manual_seed(1000003 * b + ctx)
    lens = torch.randint(max(1, ctx // 32), ctx + 1, (b,), generator=g).tolist()
    lens[int(torch.randint(0, b, (1,), generator=g))] = ctx
    return lens


def _pages(n):
    return -(-n // PAGE)


def _fit_sym(x, dim):
    s = x.abs().amax(dim=dim, keepdim=True).clamp_min(EPS) * torch.tensor(
        1.0 / 127, dtype=x.dtype, device=x.device)
    return torch.clamp(torch.round(x / s), -127, 127).to(torch.int8), s, None


def _fit_asym(x, dim):
    lo, hi = x.amin(dim=dim, keepdim=True), x.amax(dim=dim, keepdim=True)
    s = ((hi - lo) * torch.tensor(1.0 / 255, dtype=x.dtype, device=x.device)).clamp_min(EPS)
    u = torch.clamp(torch.round((x - lo) / s), 0, 255) - 128
    return u.to(torch.int8), s, lo + 128 * s


def _kv_inputs(case, seed):
    """Pools, tables, lengths and queries of an attention or sparse case.  Keys
    carry a per-channel offset, as trained models' keys do."""
    b, h, r, layers = case["batch"], case["kv_heads"], case["n_rep"], case["layers"]
    lens = _lengths(case)
    width = _pages(case["ctx"])
    pages = [_pages(n) for n in lens]
    nb = sum(pages) + 3
    g = _gen(seed)
    ids = torch.randperm(nb, device=DEV, generator=g)[:sum(pages)].to(torch.int32)
    tables = torch.zeros(b, width, dtype=torch.int32, device=DEV)
    at = 0
    for i, p in enumerate(pages):
        tables[i, :p] = ids[at:at + p]
        at += p
    kv = case.get("kv", "fp16")
    s = {"lens": lens, "tables": tables, "q": _randn(g, layers, b, h, r, D), "nb": nb,
         "seq": torch.tensor(lens, dtype=torch.int32, device=DEV)}
    offset = _randn(g, layers, h, D)
    int8 = kv != "fp16"
    dt = torch.int8 if int8 else torch.float16
    s["k"] = torch.empty(layers, nb, PAGE, h, D, dtype=dt, device=DEV)
    s["v"] = torch.empty_like(s["k"])
    if int8:
        s["ks"] = torch.empty(layers, nb, h, D, device=DEV)
        s["vs"] = torch.empty(layers, nb, PAGE, h, device=DEV)
        s["kz"] = torch.empty_like(s["ks"]) if kv == "int8z" else None
        s["vz"] = torch.empty_like(s["vs"]) if kv == "int8z" else None
        s["res"] = torch.empty(layers, b, PAGE, h, D, dtype=torch.float16, device=DEV)
        s["k_new"] = _randn(g, layers, b, h, 1, D)
        s["v_new"] = _randn(g, layers, b, h, 1, D)
        fit = _fit_asym if kv == "int8z" else _fit_sym
        last = tables[torch.arange(b, device=DEV), torch.tensor(pages, device=DEV) - 1].long()
    for li in range(layers):
        k = _randn(g, nb, PAGE, h, D)
        k += offset[li]
        v = _randn(g, nb, PAGE, h, D)
        if not int8:
            s["k"][li], s["v"][li] = k, v
            continue
        s["res"][li] = k[last]
        for x, dim, name in ((k, 1, "k"), (v, 3, "v")):
            code, step, zero = fit(x.float(), dim)
            s[name][li] = code
            s[name + "s"][li] = step.squeeze(dim)
            if zero is not None:
                s[name + "z"][li] = zero.squeeze(dim)
    if int8:
        pos = torch.tensor([n - 1 for n in lens], device=DEV)
        s["slots"] = last * PAGE + pos % PAGE
        s["res_idx"] = torch.arange(b, device=DEV) * PAGE + pos % PAGE
        s["res_rows"] = torch.arange(b, dtype=torch.int32, device=DEV)
    return s


def _captured(step):
    """`step` recorded in a HIP graph (warmed up first, on a side stream)."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    return graph


# ---------------------------------------------------------------------------
# attention and sparse
# ---------------------------------------------------------------------------


def _prepare_attention(case, seed):
    s = _kv_inputs(case, seed)
    layers, ctx = case["layers"], case["ctx"]
    s["out"] = torch.empty_like(s["q"])
    if case["kind"] == "sparse":
        s["kmin"] = torch.empty(layers, s["nb"], case["kv_heads"], D, dtype=torch.float16,
                                device=DEV)
        s["kmax"] = torch.empty_like(s["kmin"])
        for li in range(layers):
            ps.rebuild_bounds(s["k"][li], s["kmin"][li], s["kmax"][li])

        def step():
            for li in range(layers):
                ps.sparse_attention(s["q"][li], s["k"][li], s["v"][li], s["tables"], s["seq"],
                                    s["kmin"][li], s["kmax"][li], ratio=case["ratio"],
                                    max_seq_len=ctx, scoring=case["scoring"], out=s["out"][li])
    elif case["kv"] == "fp16":
        def step():
            for li in range(layers):
                pdh.paged_decode_hip(s["q"][li], s["k"][li], s["v"][li], s["tables"], s["seq"],
                                     ctx, out=s["out"][li])
    else:
        asym, h = case["kv"] == "int8z", case["kv_heads"]

        def step():
            for li in range(layers):
                kz = s["kz"][li] if asym else None
                vz = s["vz"][li] if asym else None
                iw.decode_write(s["k_new"][li], s["v_new"][li], s["slots"], s["res_idx"],
                                s["v"][li].view(-1, h, D), s["vs"][li].view(-1, h),
                                vz.view(-1, h) if asym else None, s["res"][li].view(-1, h, D),
                                asym=asym, eps=EPS, qmax=127.0, levels=255.0, offset=128.0)
                pdh.paged_decode_hip(s["q"][li], s["k"][li], s["v"][li], s["tables"], s["seq"],
                                     ctx, k_scale=s["ks"][li], v_scale=s["vs"][li], k_zero=kz,
                                     v_zero=vz, k_residual=s["res"][li], res_rows=s["res_rows"],
                                     out=s["out"][li])
    s["graph"] = _captured(step)
    return s


def _run_attention(case, s):
    s["graph"].replay()
    if case.get("kv", "fp16") == "fp16":
        return s["out"]
    written = [s["out"], s["v"], s["vs"], s["res"]]
    return written + [s["vz"]] if case["kv"] == "int8z" else written


def _kept_pages(case, s, li, i, pages, scores):
    """The pages sequence i attends per head: its budget's best by score, page
    0 and the last two always among them."""
    n = min(pages, max(3, int(math.ceil(float(torch.tensor(case["ratio"], dtype=torch.float32)
                                              * pages)))))
    scores = scores.clone()
    scores[:, 0] = math.inf
    scores[:, max(0, pages - 2):] = math.inf
    return torch.sort(scores, dim=1, descending=True, stable=True).indices[:, :n]


def _page_scores(case, s, li, i, blocks, length):
    k = s["k"][li][blocks].double()                                    # [P, 16, H, D]
    lo, hi = k.amin(dim=1), k.amax(dim=1)
    q = s["q"][li][i].double()                                         # [H, R, D]
    up = torch.matmul(q.clamp(min=0), hi.permute(1, 2, 0).contiguous()) \
        + torch.matmul(q.clamp(max=0), lo.permute(1, 2, 0).contiguous())      # [H, R, P]
    if case["scoring"] == "bounds":
        return up.amax(dim=1)
    tokens = torch.full((len(blocks),), float(PAGE), dtype=torch.float64, device=DEV)
    tokens[-1] = length - PAGE * (len(blocks) - 1)
    return torch.softmax(up / math.sqrt(D) + tokens.log(), dim=-1).sum(dim=1)


def _exact_attention(case, seed):
    s = _kv_inputs(case, seed)
    b, layers = case["batch"], case["layers"]
    kv = case.get("kv", "fp16")
    if kv != "fp16":
        fit = _fit_asym if kv == "int8z" else _fit_sym
        h = case["kv_heads"]
        s["vs"], s["res"] = s["vs"].double(), s["res"].double()
        for li in range(layers):
            x = s["v_new"][li].float().squeeze(2)
            code, _, _ = fit(x, 2)
            _, step, zero = fit(x.double(), 2)
            s["v"][li].view(-1, h, D)[s["slots"]] = code
            s["vs"][li].view(-1, h)[s["slots"]] = step.squeeze(2)
            if zero is not None:
                if s["vz"].dtype != torch.float64:
                    s["vz"] = s["vz"].double()
                s["vz"][li].view(-1, h)[s["slots"]] = zero.squeeze(2)
            s["res"][li].view(-1, h, D)[s["res_idx"]] = s["k_new"][li].double().squeeze(2)
    out = torch.empty(s["q"].shape, dtype=torch.float64, device=DEV)
    for li in range(layers):
        for i in range(b):
            length = s["lens"][i]
            blocks = s["tables"][i, :_pages(length)].long()
            k, v = s["k"][li][blocks].double(), s["v"][li][blocks].double()
            if kv != "fp16":
                k *= s["ks"][li][blocks].double()[:, None]
                v *= s["vs"][li][blocks][..., None]
                if kv == "int8z":
                    k += s["kz"][li][blocks].double()[:, None]
                    v += s["vz"][li][blocks][..., None]
                k[-1] = s["res"][li][i]
            q = s["q"][li][i].double()
            k = k.flatten(0, 1)[:length].permute(1, 2, 0).contiguous()      # [H, D, L]
            w = torch.matmul(q, k) / math.sqrt(D)
            if case["kind"] == "sparse":
                scores = _page_scores(case, s, li, i, blocks, length)
                keep = torch.zeros(scores.shape, dtype=torch.bool, device=DEV)
                keep.scatter_(1, _kept_pages(case, s, li, i, len(blocks), scores), True)
                dead = ~keep.repeat_interleave(PAGE, dim=1)[:, None, :length]
                w.masked_fill_(dead, -math.inf)
            out[li, i] = torch.matmul(torch.softmax(w, dim=-1),
                                      v.flatten(0, 1)[:length].transpose(0, 1).contiguous())
    if kv == "fp16":
        return out
    written = [out, None, s["vs"], s["res"]]
    return written + [s["vz"]] if kv == "int8z" else written


def _work_attention(case):
    lens = _lengths(case)
    b, h, r, layers = case["batch"], case["kv_heads"], case["n_rep"], case["layers"]
    tokens = sum(lens)
    full = sum(_pages(n) for n in lens)
    kv = case.get("kv", "fp16")
    if case["kind"] == "sparse":
        kept = sum(min(_pages(n), max(3, math.ceil(case["ratio"] * _pages(n)))) for n in lens)
        data = kept * PAGE * h * D * 4 + full * h * D * 4
        tokens = kept * PAGE
    elif kv == "fp16":
        data = tokens * h * D * 4
    else:
        zeros = 2 if kv == "int8z" else 1
        data = tokens * h * D * 2 + zeros * ((full - b) * h * D * 4 + tokens * h * 4) \
            + b * PAGE * h * D + b * h * D * 8
    return {"bytes": layers * (data + 2 * b * h * r * D * 2 + full * 4 + b * 4),
            "flops": layers * tokens * h * r * D * 4}


# ---------------------------------------------------------------------------
# prefill
# ---------------------------------------------------------------------------


def _prefill_inputs(case, seed):
    g = _gen(seed)
    shape = (case["layers"], case["batch"], case["tokens"], case["kv_heads"], D)
    # as the projections leave them: [B, n, H, D], seen as [B, H, n, D]
    k, v = _randn(g, *shape), _randn(g, *shape)
    k += _randn(g, case["layers"], 1, 1, case["kv_heads"], D)
    return k, v


def _prepare_prefill(case, seed):
    k, v = _prefill_inputs(case, seed)
    spec = KVCacheSpec(num_layers=case["layers"], num_kv_heads=case["kv_heads"], head_dim=D,
                       max_batch_size=case["batch"], max_seq_len=case["tokens"] + 64, device=DEV)
    if case["kv"] == "fp16":
        cache = PagedKVCache(spec)
        if case["bounds"]:
            cache.enable_page_bounds()
    else:
        cache = Int8PagedKVCache(spec, asymmetric=case["kv"] == "int8z")
    cut = case["chunk"]
    chunks = [(n, [(kk[:, a:a + n].transpose(1, 2), vv[:, a:a + n].transpose(1, 2))
                   for kk, vv in zip(k, v)])
              for a, n in ((0, cut), (cut, case["tokens"] - cut))]
    return {"cache": cache, "chunks": chunks, "slots": list(range(case["batch"])),
            "int8": case["kv"] != "fp16"}


def _run_prefill(case, s):
    cache = s["cache"]
    cache.reset()
    read = None
    for n, layers in s["chunks"]:
        cache.advance(n, slots=s["slots"])
        for li, (k, v) in enumerate(layers):
            cache.write(li, k, v)
            if not s["int8"]:
                # what the chunk's attention reads: the sequence so far
                read = cache.read(li, case["batch"])
    if s["int8"]:
        last = case["layers"] - 1
        got = [cache.k_pool[0], cache.v_pool[0], cache.k_scale_pool[0], cache.v_scale_pool[0],
               cache.residual(0), cache.k_pool[last], cache.v_pool[last],
               cache.k_scale_pool[last], cache.v_scale_pool[last], cache.residual(last)]
        if cache.asymmetric:
            got += [cache.k_zero_pool[last], cache.v_zero_pool[last]]
        return got
    got = [read[0], read[1], cache.k_pool[0], cache.v_pool[0]]
    if case["bounds"]:
        got += list(cache.page_bounds(case["layers"] - 1))
    return got


def _exact_prefill(case, seed):
    k, v = _prefill_inputs(case, seed)
    b, n, h = case["batch"], case["tokens"], case["kv_heads"]
    if case["kv"] == "fp16":
        last = [x[-1].double().transpose(1, 2) for x in (k, v)]
        return last + [None] * (4 if case["bounds"] else 2)
    # the pools' scales: pages are handed out in order, chunk by chunk
    fit = _fit_asym if case["kv"] == "int8z" else _fit_sym
    cap = _pages(n + 64) * b
    first, pages = _pages(case["chunk"]), _pages(n)
    ids = torch.tensor([[i * first + p if p < first
                         else b * first + i * (pages - first) + p - first for p in range(pages)]
                        for i in range(b)], device=DEV)
    got = []
    for li in (0, case["layers"] - 1):
        ks = torch.ones(cap, h, D, dtype=torch.float64, device=DEV)
        vs = torch.ones(cap, PAGE, h, dtype=torch.float64, device=DEV)
        res = torch.zeros(b, PAGE, h, D, dtype=torch.float64, device=DEV)
        kz, vz = torch.zeros_like(ks), torch.zeros_like(vs)
        for i in range(b):
            whole = pages - 1                            # the last page stays in the residual
            kk = k[li, i].double()
            if whole:
                _, step, zero = fit(kk[:whole * PAGE].view(whole, PAGE, h, D), 1)
                ks[ids[i, :whole]] = step.squeeze(1)
                if zero is not None:
                    kz[ids[i, :whole]] = zero.squeeze(1)
            res[i, :n - whole * PAGE] = kk[whole * PAGE:]
            _, step, zero = fit(v[li, i].double(), 2)
            slots = (ids[i].view(-1, 1) * PAGE + torch.arange(PAGE, device=DEV)).view(-1)[:n]
            vs.view(-1, h)[slots] = step.squeeze(2)
            if zero is not None:
                vz.view(-1, h)[slots] = zero.squeeze(2)
        got += [None, None, ks, vs, res]
    return got + ([kz, vz] if case["kv"] == "int8z" else [])


def _work_prefill(case):
    rows = case["layers"] * case["batch"] * case["tokens"] * case["kv_heads"]
    if case["kv"] == "fp16":
        # read and write the new rows; read the cache back after each chunk
        chunks = case["chunk"] + case["tokens"]
        back = 2 * rows * chunks / case["tokens"]
        bounds = rows / PAGE * D * 4 if case["bounds"] else 0
        return {"bytes": (2 * rows + back) * D * 4 + bounds, "flops": 0}
    z = 2 if case["kv"] == "int8z" else 1
    return {"bytes": rows * D * 4 + rows * D * 2 + z * (rows // PAGE * D * 4 + rows * 4),
            "flops": 0}


# ---------------------------------------------------------------------------
# a decoder layer's products, and the elementwise ops over a prompt
# ---------------------------------------------------------------------------


def _layer_inputs(case, seed):
    g = _gen(seed)
    m, hid, inter, hq, hk = (case[n] for n in ("rows", "hidden", "inter", "q_heads", "kv_heads"))
    layers = []
    for _ in range(case["layers"]):
        layers.append({
            "x": _randn(g, m, hid), "res": _randn(g, m, hid), "attn": _randn(g, m, hq * D),
            "w_qkv": _randn(g, (hq + 2 * hk) * D, hid, std=0.02),
            "b_qkv": _randn(g, (hq + 2 * hk) * D), "w_o": _randn(g, hid, hq * D, std=0.02),
            "w_gu": _randn(g, 2 * inter, hid, std=0.02), "w_down": _randn(g, hid, inter, std=0.02),
            "n1": 1 + _randn(g, hid, std=0.1), "n2": 1 + _randn(g, hid, std=0.1),
            "k": torch.zeros(m, PAGE, hk, D, dtype=torch.float16, device=DEV),
            "v": torch.zeros(m, PAGE, hk, D, dtype=torch.float16, device=DEV)})
    perm = torch.randperm(m, device=DEV, generator=g)
    return {"layers": layers, "slots": perm * PAGE + 5,
            "pos": torch.randint(0, 4096, (m,), device=DEV, generator=g),
            "angle": _angles(4096)}


def _angles(n):
    """fp16 cos and sin of the rotary angles of n positions (theta 1e6)."""
    inv = 1.0 / (1e6 ** (torch.arange(0, D, 2, device=DEV).float() / D))
    a = torch.outer(torch.arange(n, device=DEV).float(), inv)
    a = torch.cat([a, a], dim=-1)
    return a.cos().half(), a.sin().half()


def _prepare_layer(case, seed):
    s = _layer_inputs(case, seed)
    hq, hk = case["q_heads"], case["kv_heads"]
    cos, sin = s["angle"]
    # weights packed once at up to 16 rows (the decoder's own rule); above, as
    # a torch Linear holds them
    packed = case["rows"] <= HIP_GEMM_MAX_ROWS
    for y in s["layers"]:
        y["p_qkv"] = dg.PackedWeight(y["w_qkv"], "qkv", D) if packed else y["w_qkv"]
        y["p_o"] = dg.PackedWeight(y["w_o"]) if packed else y["w_o"]
        y["p_gu"] = dg.PackedWeight(y["w_gu"], "gate_up") if packed else y["w_gu"]
        y["p_down"] = dg.PackedWeight(y["w_down"]) if packed else y["w_down"]

    def step():
        s["got"] = []
        for y in s["layers"]:
            h, r = fe.fused_add_rms_norm(y["x"], y["res"], y["n1"], NORM_EPS)
            q = dg.qkv_rope_write(h, y["p_qkv"], y["b_qkv"], s["pos"], cos, sin, s["slots"],
                                  y["k"], y["v"], hq, hk)
            o = dg.linear(y["attn"], y["p_o"])
            h, r = fe.fused_add_rms_norm(o, r, y["n2"], NORM_EPS)
            x = dg.linear(dg.gate_up_silu(h, y["p_gu"]), y["p_down"])
            s["got"].append((q, y["k"], y["v"], r, x))

    s["graph"] = _captured(step)
    return s


def _run_layer(case, s):
    s["graph"].replay()
    return s["got"]


def _norm64(x, w):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + NORM_EPS) * w


def _rope64(x, c, s):
    half = D // 2
    return x * c + torch.cat([-x[..., half:], x[..., :half]], dim=-1) * s


def _exact_layer(case, seed):
    s = _layer_inputs(case, seed)
    m, hq, hk, inter = case["rows"], case["q_heads"], case["kv_heads"], case["inter"]
    cos, sin = (t.double()[s["pos"]][:, None] for t in s["angle"])
    got = []
    for y in s["layers"]:
        y = {n: t.double() for n, t in y.items()}
        r = y["x"] + y["res"]
        h = _norm64(r, y["n1"])
        qkv = (h @ y["w_qkv"].t() + y["b_qkv"]).view(m, hq + 2 * hk, D)
        q, k, v = qkv[:, :hq], qkv[:, hq:hq + hk], qkv[:, hq + hk:]
        q = _rope64(q, cos, sin).reshape(m, hk, hq // hk, D)
        y["k"].view(-1, hk, D)[s["slots"]] = _rope64(k, cos, sin)
        y["v"].view(-1, hk, D)[s["slots"]] = v
        r = y["attn"] @ y["w_o"].t() + r
        h = _norm64(r, y["n2"])
        gu = h @ y["w_gu"].t()
        gate, up = gu[:, :inter], gu[:, inter:]
        x = (gate * torch.sigmoid(gate) * up) @ y["w_down"].t()
        got.append((q, y["k"], y["v"], r, x))
    return got


def _work_layer(case):
    m, hid, inter, hq, hk = (case[n] for n in ("rows", "hidden", "inter", "q_heads", "kv_heads"))
    weights = (2 * hq + 2 * hk) * D * hid + 3 * inter * hid
    acts = m * (5 * hid + (2 * hq + 2 * hk) * D)
    return {"bytes": case["layers"] * 2 * (weights + acts),
            "flops": case["layers"] * 2 * m * weights}


def _rows_inputs(case, seed):
    g = _gen(seed)
    n, hid, inter, hq, hk = (case[x] for x in ("rows", "hidden", "inter", "q_heads", "kv_heads"))
    cos, sin = _angles(n)
    qkv = _randn(g, 1, n, (hq + 2 * hk) * D)               # q and k are slices of it
    return {"x": _randn(g, 1, n, hid), "res": _randn(g, 1, n, hid),
            "w": 1 + _randn(g, hid, std=0.1), "qkv": qkv, "gu": _randn(g, 1, n, 2 * inter),
            "cos": cos.view(1, 1, n, D), "sin": sin.view(1, 1, n, D)}


def _run_rows(case, s):
    hq, hk = case["q_heads"], case["kv_heads"]
    h, r = fe.fused_add_rms_norm(s["x"], s["res"], s["w"], NORM_EPS)
    q, k = fe.rope_qk(s["qkv"][..., :hq * D], s["qkv"][..., hq * D:(hq + hk) * D], s["cos"],
                      s["sin"], hq, hk, D)
    return h, r, q, k, fe.silu_and_mul(s["gu"])


def _exact_rows(case, seed):
    s = {n: t.double() for n, t in _rows_inputs(case, seed).items()}
    hq, hk, n, inter = case["q_heads"], case["kv_heads"], case["rows"], case["inter"]
    r = s["x"] + s["res"]
    c, sn = s["cos"].view(1, n, 1, D), s["sin"].view(1, n, 1, D)
    q = _rope64(s["qkv"][..., :hq * D].reshape(1, n, hq, D), c, sn)
    k = _rope64(s["qkv"][..., hq * D:(hq + hk) * D].reshape(1, n, hk, D), c, sn)
    gate, up = s["gu"][..., :inter], s["gu"][..., inter:]
    return (_norm64(r, s["w"]), r, q.reshape(1, n, hq * D), k.reshape(1, n, hk * D),
            gate * torch.sigmoid(gate) * up)


def _work_rows(case):
    n, hid, inter, hq, hk = (case[x] for x in ("rows", "hidden", "inter", "q_heads", "kv_heads"))
    return {"bytes": 2 * n * (4 * hid + 2 * (hq + hk) * D + 2 * D + 3 * inter), "flops": 0}


# ---------------------------------------------------------------------------
# a whole decode step
# ---------------------------------------------------------------------------

STD = 0.02


def _step_inputs(case, seed):
    g = _gen(int(seed) + 1)
    cfg = DecoderConfig(num_layers=case["layers"])
    ids = torch.randint(0, cfg.vocab_size, (case["batch"], 1), device=DEV, generator=g)
    pools = (case["layers"], case["batch"] * _pages(case["ctx"]), PAGE, cfg.num_kv_heads, D)
    return cfg, ids, _randn(g, *pools), _randn(g, *pools)


def _prepare_step(case, seed):
    cfg, ids, k, v = _step_inputs(case, seed)
    b, ctx = case["batch"], case["ctx"]
    model = QwenDecoder(cfg, device=DEV, seed=int(seed), std=STD)
    cache = model.allocate_cache(b, ctx)
    slots = list(range(b))
    if ctx > 1:
        cache.advance(ctx - 1, slots=slots)
    for li in range(cfg.num_layers):
        cache.k_pool[li].copy_(k[li])
        cache.v_pool[li].copy_(v[li])
    cache.advance(1, slots=slots)
    splits = choose_num_splits(b, cfg.num_kv_heads, ctx, PAGE, model.device)
    step = CapturedDecode(model, b, ctx, splits)
    step.set_inputs(ids, torch.full_like(ids, ctx - 1))
    step.record()
    return {"step": step, "ids": ids, "pos": torch.full_like(ids, ctx - 1), "cache": cache}


def _run_step(case, s):
    s["step"].set_inputs(s["ids"], s["pos"])
    logits = s["step"].replay()
    return logits, s["cache"].k_pool[-1], s["cache"].v_pool[-1]


def _exact_step(case, seed):
    cfg, ids, k_all, v_all = _step_inputs(case, seed)
    b, ctx, hq, hk = case["batch"], case["ctx"], cfg.num_heads, cfg.num_kv_heads
    g = _gen(seed)                          # the model's own weights, in its order
    half = torch.float16

    def weight(*shape):
        return (torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32)
                * STD).to(half).double()

    embed = (torch.randn(cfg.vocab_size, cfg.hidden_size, generator=g, device=DEV)
             * STD).to(half)
    inv = 1.0 / (cfg.rope_theta ** (torch.arange(0, D, 2).float() / D))
    a = torch.tensor(float(ctx - 1)) * inv
    a = torch.cat([a, a])
    cos, sin = a.cos().half().double().to(DEV), a.sin().half().double().to(DEV)
    x = embed[ids.view(-1)].double()
    pages = _pages(ctx)
    # pages are handed out in order: all of each prompt's, then the new token's
    done = _pages(ctx - 1)
    ids_of = torch.tensor([[i * done + p if p < done else b * done + i for p in range(pages)]
                           for i in range(b)], device=DEV)
    for li in range(cfg.num_layers):
        w_qkv = weight((hq + 2 * hk) * D, cfg.hidden_size)
        b_qkv = weight((hq + 2 * hk) * D)
        w_o = weight(cfg.hidden_size, hq * D)
        w_gu = weight(2 * cfg.intermediate_size, cfg.hidden_size)
        w_down = weight(cfg.hidden_size, cfg.intermediate_size)
        qkv = (_norm64(x, 1.0) @ w_qkv.t() + b_qkv).view(b, hq + 2 * hk, D)
        q = _rope64(qkv[:, :hq], cos, sin).reshape(b, hk, hq // hk, D)
        attn = torch.empty_like(q)
        for i in range(b):
            k = k_all[li][ids_of[i]].double().flatten(0, 1)[:ctx]
            v = v_all[li][ids_of[i]].double().flatten(0, 1)[:ctx]
            k[ctx - 1] = _rope64(qkv[i, hq:hq + hk], cos, sin)
            v[ctx - 1] = qkv[i, hq + hk:]
            w = torch.matmul(q[i], k.permute(1, 2, 0).contiguous()) / math.sqrt(D)
            attn[i] = torch.matmul(torch.softmax(w, dim=-1), v.transpose(0, 1).contiguous())
        x = x + attn.view(b, hq * D) @ w_o.t()
        gu = _norm64(x, 1.0) @ w_gu.t()
        gate, up = gu.chunk(2, dim=-1)
        x = x + (gate * torch.sigmoid(gate) * up) @ w_down.t()
    h = _norm64(x, 1.0)
    logits = torch.cat([h @ part.double().t() for part in embed.split(16384)], dim=-1)
    return logits.view(b, 1, -1), None, None


def _work_step(case):
    cfg = DecoderConfig(num_layers=case["layers"])
    b, hid, inter = case["batch"], cfg.hidden_size, cfg.intermediate_size
    per_layer = (2 * cfg.num_heads + 2 * cfg.num_kv_heads) * D * hid + 3 * inter * hid
    weights = case["layers"] * per_layer + cfg.vocab_size * hid
    kv = case["layers"] * b * case["ctx"] * cfg.num_kv_heads * D * 2
    return {"bytes": 2 * (weights + kv + b * cfg.vocab_size),
            "flops": 2 * b * weights + 2 * kv * cfg.num_heads // cfg.num_kv_heads}


# ---------------------------------------------------------------------------

_KINDS = {
    "attention": (_prepare_attention, _run_attention, _exact_attention, _work_attention),
    "sparse": (_prepare_attention, _run_attention, _exact_attention, _work_attention),
    "prefill": (_prepare_prefill, _run_prefill, _exact_prefill, _work_prefill),
    "layer": (_prepare_layer, _run_layer, _exact_layer, _work_layer),
    "rows": (_rows_inputs, _run_rows, _exact_rows, _work_rows),
    "step": (_prepare_step, _run_step, _exact_step, _work_step),
}


def prepare(case, seed):
    state = _KINDS[case["kind"]][0](case, seed)
    state["case"] = dict(case)
    return state


def run(state):
    case = state["case"]
    return _KINDS[case["kind"]][1](case, state)


def exact(case, seed):
    return _KINDS[case["kind"]][2](case, seed)


def work(case):
    return _KINDS[case["kind"]][3](case)


def tolerance(case):
    """About four times what the path shows against ``exact`` (relative error
    over the output 2.5e-4 fp16, 5.2e-4 INT8 attention; 8e-4 down to 3e-4 a
    layer's products; 4e-4 the elementwise ops; 4.8e-3 the logits after 28
    layers in fp16; 2e-3 to 3.6e-3 the sparse output, where pages whose scores
    nearly tie at the budget's edge are picked differently)."""
    kind = case["kind"]
    if kind == "prefill":
        return "exact"                       # copies and bit-exact quantizers
    if kind == "step":
        return {"rel": 2e-2, "max": 0.1}
    if kind == "sparse":
        return {"rel": 1e-2, "max": 0.5}
    if kind == "layer":
        return {"rel": 3e-3, "max": 0.03}
    return {"rel": 2e-3, "max": 0.02}
