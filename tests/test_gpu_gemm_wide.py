"""The decode GEMM's walk, on an MI355X: row counts at the edges of its 16-row
column blocks (1 to 4 of them), widths that end inside a tile and leave a
workgroup one, two or three tiles, K of one step, of chunks
shorter than a wave's steps and split over workgroups, both weight layouts,
and the fused epilogues bit-equal to the launches they replace."""

from __future__ import annotations

import pytest

torch = pytest.importorskip("torch")

pytestmark = [
    pytest.mark.gpu,
    pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU"),
]


def dg():
    from latentserve_amd.kernels import decode_gemm
    return decode_gemm


def fe():
    from latentserve_amd.kernels import fused_elementwise
    return fused_elementwise


def _operands(m, n, k):
    gen = torch.Generator(device="cuda").manual_seed(m + 3 * n + 7 * k)
    x = torch.randn(m, k, device="cuda", generator=gen).half()
    w = (torch.randn(n, k, device="cuda", generator=gen) * k**-0.5).half()
    return x, w, torch.randn(n, device="cuda", generator=gen).half()


@pytest.mark.parametrize("m", [1, 16, 17, 32, 33, 48, 49, 64])
@pytest.mark.parametrize("n,k", [(16, 32), (5, 96), (100, 1024), (4100, 288), (8200, 1120),
                                 (12300, 1536), (300, 2048), (50, 2080), (1536, 8960),
                                 (2000, 4864), (40, 480), (5000, 512), (47, 544)])
def test_product(m, n, k):
    x, w, b = _operands(m, n, k)
    want = x.double() @ w.double().t() + b.double()
    ys = [dg().linear(x, wk, b) for wk in (w, dg().PackedWeight(w), w)]
    torch.cuda.synchronize()
    # one fp16 rounding (2^-11 relative, twice that at a binade's edge) and the
    # fp32 sums: at most K products of size |x| |w| rounded at 2^-24 each
    slack = (x.double().abs() @ w.double().abs().t() + b.double().abs()) * k * 2.0**-24
    assert ((ys[0].double() - want).abs() <= want.abs() * 2.0**-10 + slack + 2.0**-24).all()
    assert torch.equal(ys[0], ys[1]) and torch.equal(ys[0], ys[2])


@pytest.mark.parametrize("m", [5, 16, 17, 48, 64])
def test_infinite_and_nan_rows_stay_in_their_rows(m):
    """A row of X with inf or NaN, and a chunk shorter than the wave's steps:
    the other rows' outputs are those of the finite product."""
    x, w, b = _operands(m, 40, 224)
    clean = dg().linear(x, w, b)
    x2 = x.clone()
    x2[3, 5], x2[m - 1, 100] = float("inf"), float("nan")
    got = dg().linear(x2, w, b)
    keep = torch.ones(m, dtype=torch.bool, device="cuda")
    keep[3] = keep[m - 1] = False
    assert torch.equal(got[keep], clean[keep])
    assert got[m - 1].isnan().all() and torch.equal(got[3], (x2[3:4].float() @ w.float().t()
                                                             + b.float()).half()[0])


@pytest.mark.parametrize("m", [17, 40, 64])
@pytest.mark.parametrize("inter,k", [(8960, 1536), (100, 64), (36, 896), (1500, 2048),
                                     (300, 4096)])
@pytest.mark.parametrize("bias", [False, True])
def test_gate_up_silu(m, inter, k, bias):
    x, w, b = _operands(m, 2 * inter, k)
    b = b if bias else None
    got = dg().gate_up_silu(x, w, b)
    assert torch.equal(got, fe().silu_and_mul(dg().linear(x, w, b)))


@pytest.mark.parametrize("m", [17, 40, 64])
@pytest.mark.parametrize("hq,hk,d,k", [(12, 2, 128, 1536), (7, 1, 128, 896), (4, 4, 64, 4096)])
@pytest.mark.parametrize("bounds", [False, True])
def test_qkv_rope_write(m, hq, hk, d, k, bounds):
    x, w, b = _operands(m, (hq + 2 * hk) * d, k)
    gen = torch.Generator(device="cuda").manual_seed(m)
    nb, page = 70, 16
    ang = torch.rand(300, d // 2, device="cuda", generator=gen) * 6
    cos, sin = torch.cat([ang, ang], -1).cos().half(), torch.cat([ang, ang], -1).sin().half()
    pos = torch.randint(0, 400, (m,), device="cuda", generator=gen)
    slots = torch.randperm(nb, device="cuda", generator=gen)[:m] * page
    slots += torch.randint(0, 2, (m,), device="cuda", generator=gen) * 5
    slots[0], slots[2] = -1, nb * page + 3
    outs = []
    for fused in (True, False):
        kp, vp = (torch.full((nb, page, hk, d), 2.0, device="cuda").half() for _ in range(2))
        mn, mx = (torch.full((nb, hk, d), s, device="cuda").half() for s in (-0.5, 0.5))
        kw = dict(kmin=mn, kmax=mx) if bounds else {}
        if fused:
            q = dg().qkv_rope_write(x, w, b, pos, cos, sin, slots, kp, vp, hq, hk, **kw)
        else:
            q = fe().rope_write_decode(dg().linear(x, w, b), pos, cos, sin, slots, kp, vp, hq, hk,
                                       **kw)
        outs.append((q, kp, vp, mn, mx))
    for a, c in zip(*outs):
        assert torch.equal(a, c)


@pytest.mark.parametrize("k", [32, 64, 96, 448])
def test_weight_rows_far_apart_with_empty_chunks(k):
    """Rows past 32-bit offsets and a K of fewer steps than the waves: the waves
    without a chunk read within the rows (the last row ends the allocation)."""
    n, ld = 16, (1 << 26) + 8
    x, w, b = _operands(16, n, k)
    store = torch.empty((n - 1) * ld + k, dtype=torch.float16, device="cuda")
    far = store.as_strided((n, k), (ld, 1))
    far.copy_(w)
    assert torch.equal(dg().linear(x, far, b), dg().linear(x, w, b))


def test_split_product_in_a_graph_replays_exactly():
    x, w, _ = _operands(48, 1536, 8960)
    assert dg().workspace_bytes(48, 1536, 8960) > 0
    want = dg().linear(x, w)
    out = torch.empty_like(want)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        dg().linear(x, w, out=out)
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        dg().linear(x[:20], w)                     # eager work between replays


@pytest.mark.parametrize("m", [3, 64])
def test_weight_rows_far_apart(m):
    """Row-major weights whose rows lie 2^27 bytes apart: a tile's rows are
    past 32-bit offsets from its first (64-bit addresses, the same results)."""
    n, k, ld = 20, 224, 2**26 + 8
    store = torch.empty((n - 1) * ld + k, dtype=torch.float16, device="cuda")
    far = store.as_strided((n, k), (ld, 1))
    x, w, b = _operands(m, n, k)
    far.copy_(w)
    assert torch.equal(dg().linear(x, far, b), dg().linear(x, w, b))
    assert torch.equal(dg().gate_up_silu(x, far), dg().gate_up_silu(x, w))


@pytest.mark.parametrize("m,k", [(3, 96), (16, 1536), (40, 1536), (64, 2048)])
@pytest.mark.parametrize("off", ["table", "bias", "rows", "none"])
def test_qkv_rope_write_off_the_wide_loads(m, k, off):
    """The q/k/v epilogue where its early 8-byte loads or its 8-byte stores do
    not apply (tables or a bias off 4 bytes, an odd table stride; rows of q and
    the pools off 8 bytes) and where they do, without a bias in between, over
    pages of 12 tokens: the bits of linear followed by rope_write_decode."""
    gen = torch.Generator(device="cuda").manual_seed(m + k)
    hq, hk, d, nb, page = 4, 2, 64, 70, 12
    n = (hq + 2 * hk) * d
    x = torch.randn(m, k, device="cuda", generator=gen).half()
    w = (torch.randn(n, k, device="cuda", generator=gen) * k**-0.5).half()
    bias = torch.randn(n + 1, device="cuda", generator=gen).half()
    b = {"bias": bias[1:], "none": bias[:n]}.get(off)
    wide = torch.randn(2, 50, d + 1, device="cuda", generator=gen).half()
    cos, sin = (wide[0, :, 1:], wide[1, :, 1:]) if off == "table" else \
        (wide[0, :, :d].contiguous(), wide[1, :, :d].contiguous())
    pos = torch.randint(0, 60, (m,), device="cuda", generator=gen)
    slots = torch.randperm(nb, device="cuda", generator=gen)[:m] * page \
        + torch.randint(0, page, (m,), device="cuda", generator=gen)
    slots[0] = nb * page                                 # past the pool: not stored
    extra = 1 if off == "rows" else 0
    outs = []
    for fused in (True, False):
        g = torch.Generator(device="cuda").manual_seed(7)
        pools = [torch.randn(nb, page, hk, d + extra, device="cuda", generator=g).half()[..., extra:]
                 for _ in range(2)]
        q = torch.zeros(m, hk, hq // hk, d + extra, device="cuda").half()[..., extra:]
        args = (pos, cos, sin, slots, *pools, hq, hk)
        if fused:
            dg().qkv_rope_write(x, w, b, *args, q_out=q)
        else:
            fe().rope_write_decode(dg().linear(x, w, b), *args, q_out=q)
        outs.append((q, *pools))
    torch.cuda.synchronize()
    for a, c in zip(*outs):
        assert torch.equal(a, c)
