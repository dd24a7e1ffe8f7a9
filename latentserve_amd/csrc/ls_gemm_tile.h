// Device code shared by the decode GEMM kernels: the weight rows of an output
// tile, and the epilogues of a tile's fp32 sums (plain, gate/up + SiLU, and
// RoPE + K/V store), so every kernel finishes a product with the same
// rounding.
#pragma once

#include "ls_common.h"
#include "ls_gemm.h"

#pragma clang fp contract(off)

namespace ls {

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

// What the q/k/v epilogue reads of a lane's sequence and tile, requested before
// the tile's sums are known: late, the bias, the position, the angles it
// names and the slot were four memory round trips in a chain at the end of the
// launch (M 48, row-major, 2048 x 1536: 8.84 -> 8.43 us; and with no branch an
// element in the epilogue, M 16, packed, with the norm, 7.24 -> 6.92).
struct RopeAhead {
    int64_t pos, slot;                   // of the lane's sequence
    u2 c0, c1, s0, s1;                   // angles of its channels, 4 fp16 each
    u2 b0, b1;                           // their bias
};

__device__ __forceinline__ void rope_unpack(u2 v, half_t* o) {
    const h4 t = as_h4(v.x, v.y);
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = t[e];
}

// The row's position and slot (once a launch).
__device__ __forceinline__ void rope_row(const GemmParams& a, int m, RopeAhead& ra) {
    m = m < a.M ? m : a.M - 1;
    ra.pos = a.rope.pos[m];
    ra.slot = a.rope.slots[m];
}

// The angles and bias of a tile's columns (ROPE_TILE_VM loads), by resources (of no bytes without a
// bias, or where rope.ahead is unset: the epilogue then loads them): no load
// under a branch, which would make the walk's loads wait.
constexpr int ROPE_TILE_VM = 6;
__device__ __forceinline__ void rope_tile(const GemmParams& a, int tile, int lane, RopeAhead& ra) {
    const RopeWriteParams& w = a.rope;
    const int tph = w.d / 16, head = tile / tph, i = 8 * (tile % tph) + 4 * ((lane >> 4) & 1);
    const int64_t p = ra.pos < 0 ? 0 : (ra.pos >= w.tab_rows ? w.tab_rows - 1 : ra.pos);
    const int bytes = w.ahead ? 0x7fffffff : 0;
    const uint32_t at = (uint32_t)((p * w.st + i) * 2);
    const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc((void*)w.cos, 0, bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)w.sin, 0, bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rb =
        __builtin_amdgcn_make_buffer_rsrc((void*)a.bias, 0, a.bias && w.ahead ? a.N * 2 : 0, 0x00020000);
    const uint32_t n0 = (uint32_t)(head * w.d + i) * 2;
    auto ld = [](__amdgpu_buffer_rsrc_t r, uint32_t off) {
        return __builtin_bit_cast(u2, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
    };
    ra.c0 = ld(rc, at);
    ra.c1 = ld(rc, at + w.d);
    ra.s0 = ld(rs, at);
    ra.s1 = ld(rs, at + w.d);
    ra.b0 = ld(rb, n0);
    ra.b1 = ld(rb, n0 + w.d);
}

// The same without rope.ahead (tables past 32-bit offsets, or off 4 bytes), once
// the sums are known.
__device__ __forceinline__ void rope_late(const GemmParams& a, int head, int i, RopeAhead& ra) {
    const RopeWriteParams& w = a.rope;
    const int64_t p = ra.pos < 0 ? 0 : (ra.pos >= w.tab_rows ? w.tab_rows - 1 : ra.pos);
    auto four = [](const void* base, int64_t at) {
        const uint16_t* x = (const uint16_t*)base + at;
        return u2{x[0] | (uint32_t)x[1] << 16, x[2] | (uint32_t)x[3] << 16};
    };
    const int64_t at = p * w.st + i, n0 = (int64_t)head * w.d + i;
    const int hd = w.d / 2;
    ra.c0 = four(w.cos, at);
    ra.c1 = four(w.cos, at + hd);
    ra.s0 = four(w.sin, at);
    ra.s1 = four(w.sin, at + hd);
    if (a.bias) {
        ra.b0 = four(a.bias, n0);
        ra.b1 = four(a.bias, n0 + hd);
    }
}

// The fused q/k/v projection's epilogue for one lane: channels i .. i + 3
// of head `head` (i < d / 2) and their partners i + d / 2 .. for sequence
// m, as x0 / x1 (fp16, bias added); rotated and stored as
// rope_write_decode_kernel stores them (the same rounding, bit-equal).
__device__ __forceinline__ void rope_store(const RopeWriteParams& a, int m, int head, int i,
                                           const half_t* x0, const half_t* x1,
                                           const RopeAhead& ra) {
    const int hd = a.d / 2;
    half_t c0[4], c1[4], s0[4], s1[4];
    rope_unpack(ra.c0, c0);
    rope_unpack(ra.c1, c1);
    rope_unpack(ra.s0, s0);
    rope_unpack(ra.s1, s1);
    const bool rotated = head < a.hq + a.hk;
    half_t o0[4], o1[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const half_t r0 = rope_h(x0[e], c0[e], -x1[e], s0[e]);
        const half_t r1 = rope_h(x1[e], c1[e], x0[e], s1[e]);
        o0[e] = rotated ? r0 : x0[e];
        o1[e] = rotated ? r1 : x1[e];
    }
    half_t* dst;
    if (head < a.hq) {
        const int n_rep = a.hq / a.hk;
        dst = (half_t*)a.q_out + (int64_t)m * a.sq_b + (int64_t)(head / n_rep) * a.sq_h +
              (int64_t)(head % n_rep) * a.sq_r;
    } else {
        const int64_t slot = ra.slot;
        if (slot < 0 || slot >= (int64_t)a.num_blocks * a.page) return;
        // (a 64-bit division is a hundred instructions)
        const int64_t blk = slot >> 32 ? slot / a.page : (unsigned)slot / (unsigned)a.page;
        const int64_t off = slot - blk * a.page;
        const bool isk = head < a.hq + a.hk;
        const int h = isk ? head - a.hq : head - a.hq - a.hk;
        dst = (half_t*)(isk ? a.k_pool : a.v_pool) + blk * a.sp_b + off * a.sp_t +
              (int64_t)h * a.sp_h;
        if (isk && a.kmin) {
            // the page's K bounds: its first token resets them (fp16 min /
            // max are exact)
            half_t* mn = (half_t*)a.kmin + blk * a.sb_b + (int64_t)h * a.sb_h;
            half_t* mx = (half_t*)a.kmax + blk * a.sb_b + (int64_t)h * a.sb_h;
            half_t n0[4], n1[4], m0[4], m1[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                n0[e] = mn[i + e];
                n1[e] = mn[i + hd + e];
                m0[e] = mx[i + e];
                m1[e] = mx[i + hd + e];
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                mn[i + e] = off ? (half_t)fminf((float)n0[e], (float)o0[e]) : o0[e];
                mx[i + e] = off ? (half_t)fmaxf((float)m0[e], (float)o0[e]) : o0[e];
                mn[i + hd + e] = off ? (half_t)fminf((float)n1[e], (float)o1[e]) : o1[e];
                mx[i + hd + e] = off ? (half_t)fmaxf((float)m1[e], (float)o1[e]) : o1[e];
            }
        }
    }
    if (a.vec_out) {
        h4 v0, v1;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v0[e] = o0[e];
            v1[e] = o1[e];
        }
        *(h4*)(dst + i) = v0;
        *(h4*)(dst + i + hd) = v1;
        return;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        dst[i + e] = o0[e];
        dst[i + hd + e] = o1[e];
    }
}

// The plain, gate/up and q/k/v epilogues of one 16 x 16 tile whose K is not
// split over workgroups: lane (r, g) holds the sums of row m = 16 mb + r, tile
// columns 4g .. 4g + 3 (acc); ra is read by the q/k/v epilogue only.  All
// lanes of a wave call it together.
template <int EPI>
__device__ __forceinline__ void finish_tile(const GemmParams& a, int tile, int mb, int lane, f4 acc,
                                            const RopeAhead& ra) {
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
    RopeAhead rt = ra;
    if (!a.rope.ahead) rope_late(a, head, i, rt);
    half_t b0[4], b1[4], x0[4], x1[4];
    rope_unpack(rt.b0, b0);
    rope_unpack(rt.b1, b1);
    const bool biased = a.bias != nullptr;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        x0[e] = (half_t)(biased ? acc[e] + (float)b0[e] : acc[e]);
        x1[e] = (half_t)(biased ? up[e] + (float)b1[e] : up[e]);
    }
    rope_store(a.rope, m, head, i, x0, x1, rt);
}

}  // namespace ls
