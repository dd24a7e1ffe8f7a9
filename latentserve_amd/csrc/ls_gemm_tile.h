// Device code shared by the decode GEMM kernels: the weight rows of an output
// tile, and the epilogues of a tile's fp32 sums (plain, gate/up + SiLU, and
// RoPE + K/V store), so every kernel finishes a product with the same
// rounding.
#pragma once

#include "ls_common.h"
#include "ls_gemm.h"

#pragma clang fp contract(off)

namespace ls {

// Device-coherent (write-through, sc1) 16-byte store: the workgroup that
// sums a tile's partials may run on another XCD, whose L2 does not see this
// one's.
__device__ __forceinline__ void store_through4(float* p, f4 v) {
    asm volatile("global_store_dwordx4 %0, %1, off sc1" : : "v"(p), "v"(v) : "memory");
}

// Stores one lane's four outputs y[m][nc .. nc + 3] (fewer at the right
// edge of a width-n output).
__device__ __forceinline__ void store_out(const GemmParams& a, int m, int nc, int n,
                                          const half_t* v) {
    half_t* yp = (half_t*)a.y + (int64_t)m * a.ldy + nc;
    if (a.vec_y && nc + 3 < n) {
        h4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = v[e];
        *(h4*)yp = o;
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (nc + e < n) yp[e] = v[e];
    }
}

// W row of output-tile row r: plain tiles hold 16 consecutive rows; gate/up
// tiles hold gate rows 8T .. 8T + 7 and the up rows I + 8T .. (rows past the
// edge clamped to a valid one: their outputs are not stored); RoPE tiles
// hold 8 channels of a head's first half and their rotate-half partners,
// head T / (d / 16), channels 8 (T % (d / 16)) + [0, 8) and + d / 2.
template <int EPI>
__device__ __forceinline__ int w_row_of(int N, int d, int tile, int r, bool& real) {
    if (EPI == GEMM_GLU) {
        const int half_n = N / 2, j0 = 8 * tile + (r & 7), j = j0 < half_n ? j0 : half_n - 1;
        real = j0 < half_n;
        return r < 8 ? j : half_n + j;
    }
    int n;
    if (EPI == GEMM_ROPE) {
        const int tph = d / 16, head = tile / tph, i = 8 * (tile % tph) + (r & 7);
        n = head * d + i + (r < 8 ? 0 : d / 2);
    } else {
        n = 16 * tile + r;
    }
    real = n < N;
    return n < N ? n : N - 1;
}
template <int EPI>
__device__ __forceinline__ int w_row(const GemmParams& a, int tile, int r) {
    bool real;
    return w_row_of<EPI>(a.N, a.rope.d, tile, r, real);
}

// The fused q/k/v projection's epilogue for one lane: channels i .. i + 3
// of head `head` (i < d / 2) and their partners i + d / 2 .. for sequence
// m, as x0 / x1 (fp16, bias added); rotated and stored as
// rope_write_decode_kernel stores them (the same rounding, bit-equal).
__device__ __forceinline__ void rope_store(const RopeWriteParams& a, int m, int head, int i,
                                           const half_t* x0, const half_t* x1) {
    const int hd = a.d / 2;
    int64_t p = a.pos[m];
    p = p < 0 ? 0 : (p >= a.tab_rows ? a.tab_rows - 1 : p);
    const half_t* c = (const half_t*)a.cos + p * a.st;
    const half_t* s = (const half_t*)a.sin + p * a.st;
    half_t o0[4], o1[4];
    if (head < a.hq + a.hk) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            o0[e] = rope_h(x0[e], c[i + e], -x1[e], s[i + e]);
            o1[e] = rope_h(x1[e], c[i + hd + e], x0[e], s[i + hd + e]);
        }
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            o0[e] = x0[e];
            o1[e] = x1[e];
        }
    }
    half_t* dst;
    if (head < a.hq) {
        const int n_rep = a.hq / a.hk;
        dst = (half_t*)a.q_out + (int64_t)m * a.sq_b + (int64_t)(head / n_rep) * a.sq_h +
              (int64_t)(head % n_rep) * a.sq_r;
    } else {
        const int64_t slot = a.slots[m];
        if (slot < 0) return;
        const int64_t blk = slot / a.page, off = slot % a.page;
        if (blk >= a.num_blocks) return;
        const bool isk = head < a.hq + a.hk;
        const int h = isk ? head - a.hq : head - a.hq - a.hk;
        dst = (half_t*)(isk ? a.k_pool : a.v_pool) + blk * a.sp_b + off * a.sp_t +
              (int64_t)h * a.sp_h;
        if (isk && a.kmin) {
            // the page's K bounds: its first token resets them (fp16 min /
            // max are exact)
            half_t* mn = (half_t*)a.kmin + blk * a.sb_b + (int64_t)h * a.sb_h;
            half_t* mx = (half_t*)a.kmax + blk * a.sb_b + (int64_t)h * a.sb_h;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (off == 0) {
                    mn[i + e] = o0[e];
                    mx[i + e] = o0[e];
                    mn[i + hd + e] = o1[e];
                    mx[i + hd + e] = o1[e];
                } else {
                    mn[i + e] = (half_t)fminf((float)mn[i + e], (float)o0[e]);
                    mx[i + e] = (half_t)fmaxf((float)mx[i + e], (float)o0[e]);
                    mn[i + hd + e] = (half_t)fminf((float)mn[i + hd + e], (float)o1[e]);
                    mx[i + hd + e] = (half_t)fmaxf((float)mx[i + hd + e], (float)o1[e]);
                }
            }
        }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        dst[i + e] = o0[e];
        dst[i + hd + e] = o1[e];
    }
}

// The plain, gate/up and q/k/v epilogues of one 16 x 16 tile whose K is not
// split over workgroups: lane (r, g) holds the sums of row m = 16 mb + r, tile
// columns 4g .. 4g + 3 (acc).  All lanes of a wave call it together.
template <int EPI>
__device__ __forceinline__ void finish_tile(const GemmParams& a, int tile, int mb, int lane, f4 acc) {
    const int r = lane & 15, g = lane >> 4, m = 16 * mb + r;
    if (EPI == GEMM_PLAIN) {
        const int nc = 16 * tile + 4 * g;              // this lane's 4 output columns
        if (nc >= a.N || m >= a.M) return;
        half_t o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float bv =
                a.bias && nc + e < a.N ? (float)((const half_t*)a.bias)[nc + e] : 0.f;
            o[e] = (half_t)(acc[e] + bv);
        }
        store_out(a, m, nc, a.N, o);
        return;
    }
    // lanes g = 0, 1 hold the first half's columns (gate, or a head's first
    // half) 8 tile + 4g + e, lanes g + 2 the matching second half's
    f4 up;
#pragma unroll
    for (int e = 0; e < 4; ++e) up[e] = __shfl_xor(acc[e], 32);
    if (EPI == GEMM_GLU) {
        const int half_n = a.N / 2, j = 8 * tile + 4 * g;
        if (g >= 2 || m >= a.M || j >= half_n) return;
        half_t o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float gv = acc[e], uv = up[e];
            if (a.bias && j + e < half_n) {
                gv += (float)((const half_t*)a.bias)[j + e];
                uv += (float)((const half_t*)a.bias)[half_n + j + e];
            }
            o[e] = silu_mul_h((half_t)gv, (half_t)uv);
        }
        store_out(a, m, j, half_n, o);
        return;
    }
    const int tph = a.rope.d / 16, head = tile / tph, i = 8 * (tile % tph) + 4 * g;
    if (g >= 2 || m >= a.M || head >= a.rope.hq + 2 * a.rope.hk) return;
    const int n0 = head * a.rope.d + i, n1 = n0 + a.rope.d / 2;
    half_t x0[4], x1[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float v0 = acc[e], v1 = up[e];
        if (a.bias) {
            v0 += (float)((const half_t*)a.bias)[n0 + e];
            v1 += (float)((const half_t*)a.bias)[n1 + e];
        }
        x0[e] = (half_t)v0;
        x1[e] = (half_t)v1;
    }
    rope_store(a.rope, m, head, i, x0, x1);
}

}  // namespace ls
