// The decode GEMM's kernel (ls_gemm.hip has the host side):
//   Y[M, N] = X[M, K] . W[N, K]^T (+ bias), M <= 64,
// its gate/up form silu(X . Wg^T) * (X . Wu^T) and its q/k/v form, finished
// in the epilogue (ls_gemm_tile.h).
//
// HBM-bound on W: every weight is used once a launch, X stays in the caches.
// The work unit is a 16-row tile of W (16 output features) and every tile
// meets all of X, MB column blocks of 16 rows: up to 4 KiB of X for each KiB
// of W.  So a workgroup reads X once and walks many tiles.  Its 8 waves split
// its range of K, a chunk of at most SPW steps of 32 channels a wave; each
// wave holds its chunk of X in registers and streams the tiles blockIdx.x,
// + gridDim.x, ... through SETS register sets, one tile's weights requested
// as soon as an earlier tile's are consumed.  A tile's 8 partial sums meet in
// LDS (a buffer a set: one barrier a tile), and wave mb finishes column block
// mb.  The grid is one group a CU, each with its share of the tiles.
//
// K beyond 8 waves x 8 steps (2048 channels) is split over workgroups
// (blockIdx.y): fp32 partials through the workspace, the last group of a tile
// to arrive sums them in split order, so the result does not depend on which
// one that is.
//
// The W loads go through a buffer resource: a step past the wave's chunk is
// an offset past its end and a tile past the walk a resource of no bytes,
// zeros without a memory request, so the walk has no load under a branch (the
// compiler would wait for every load in flight at the join).
//
// MFMA v_mfma_f32_16x16x16_f16 with A = 16 rows of W and B = X^T: lane (r, g)
// holds 16 bytes of W row r and of X row r a step, and the two MFMAs of the
// step take elements 0-3 and 4-7 of those, the channel order of both operands
// being the same.  Output lane (r, g) holds Y[r][n0 + 4g .. 4g + 3].
//
// Measured (graph-timed over 1 GB of rotating weights, us before -> now; the
// kernel before gave a group of up to 4 waves one to four tiles, with X read
// again for them, and split K from 512 channels on above 32 rows):
//                      M 16, packed     M 48, row-major    M 64, row-major
//   17920 x 1536      15.5 -> 12.5      42.8 -> 14.1       52.8 -> 16.7
//   1536 x 8960       12.4 -> 9.8       42.7 -> 12.8       53.5 -> 14.5
//   1536 x 1536        4.9 -> 4.0       12.7 ->  6.0       15.2 ->  7.2
//   2048 x 5632       10.8 -> 8.4
//   151936 x 1536     89.0 -> 80.8  (5.8 TB/s)
#pragma once

#include <type_traits>

#include "ls_common.h"
#include "ls_gemm.h"
#include "ls_gemm_tile.h"

#pragma clang fp contract(off)

namespace ls {

namespace {

constexpr int LDS_BYTES = 160 * 1024;
// W is read once, whole lines at a time: nontemporal (M 48, packed weights,
// 17920 x 1536: 14.6 -> 13.9 us, 1536 x 8960: 16.6 -> 15.9; with loads that
// take half of each line it is slower than plain, 15.9 -> 18.4).
constexpr int W_POLICY = 2;
// Register sets of W: tiles in flight a wave.  (Three at one column block,
// whose registers would allow it, are slower: M 16, packed, gate/up 12.8 ->
// 13.6 us, down 10.3 -> 10.6; so are two groups a CU: 12.8 -> 13.4, 10.3 ->
// 10.4.)
constexpr int SETS = 2;

// Split K: the partial sums of split sp of tile t, [column block][lane] f4.
// (A tile's partials are contiguous: stored as rows of [M, N], 64 bytes a row,
// the 1536 x 8960 product at M 48 took 16.1 us in 5 splits and
// 20.8 in 10, against 14.2 and 15.0.)
template <int MB>
__device__ __forceinline__ float* part_tile(const GemmParams& a, int sp, int t) {
    const int tiles = (a.N + 15) / 16;
    return a.part + ((int64_t)sp * tiles + t) * MB * WAVE * 4;
}

// sum += the partial tiles t of every split, in split order: R splits' loads in
// flight together (one past the last rereads it and is not added).
template <int R, int MB>
__device__ __forceinline__ void add_partials(const GemmParams& a, int t, int lane, f4 (&sum)[MB]) {
    for (int sp = 0; sp < a.splits; sp += R) {
        f4 v[R][MB];
#pragma unroll
        for (int e = 0; e < R; ++e) {
            const __amdgpu_buffer_rsrc_t rs = coherent_rsrc(
                wave_uniform(part_tile<MB>(a, sp + e < a.splits ? sp + e : a.splits - 1, t)));
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) v[e][mb] = load_coherent4(rs, (mb * WAVE + lane) * 16);
        }
#pragma unroll
        for (int e = 0; e < R; ++e)
            if (sp + e < a.splits)
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) sum[mb] += v[e][mb];
    }
}

// h = fp16(w * fp16(s * inv)) on 8 channels: the fp32 scale rounded to
// fp16, then the weight product in packed fp16 (exact product, one rounding)
__device__ __forceinline__ u4 norm_row(u4 sv, u4 wv, float inv) {
    // (bit casts take named scalars: this compiler casts an element of a
    // vector lvalue from the vector's first element)
    const uint32_t sw[4] = {sv.x, sv.y, sv.z, sv.w};
    const uint32_t ww[4] = {wv.x, wv.y, wv.z, wv.w};
    uint32_t hw[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const h2 s2 = __builtin_bit_cast(h2, sw[e]);
        const h2 n2 = {(half_t)((float)s2.x * inv), (half_t)((float)s2.y * inv)};
        hw[e] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2, ww[e]) * n2);
    }
    return (u4){hw[0], hw[1], hw[2], hw[3]};
}

// PW: the weight is packed (gemm_packed_bytes).  NRM: X is rms_norm(x + nres)
// (one column block, K in one group, packed).  FAR: row-major weights whose
// rows lie too far apart for 32-bit offsets, by 64-bit addresses.
template <int SPW, int MB, int EPI, bool PW, bool NRM, bool FAR>
__global__ __launch_bounds__(GEMM_WAVES* WAVE) void decode_gemm_kernel(GemmParams a) {
    static_assert(!NRM || (PW && MB == 1), "the norm prologue: one column block, packed weight");
    static_assert(!FAR || !PW, "packed tiles are within reach");
    // X on its way to registers: the group's K range of 16 rows a column block,
    // ROUND blocks at once; and a tile's partial sums (a buffer a set: [wave]
    // [column block][lane]), in the same bytes where both do not fit.
    constexpr int PITCH = SPW * GEMM_WAVES * 64 + 16;      // bytes a row: the reads of 16 rows
                                                           // fall in different banks
    constexpr int XBLOCK = 16 * PITCH;
    constexpr int ROUND = MB * XBLOCK <= LDS_BYTES ? MB : LDS_BYTES / XBLOCK;
    constexpr int PART = GEMM_WAVES * MB * WAVE;           // f4 a buffer
    constexpr bool APART = ROUND * XBLOCK + SETS * PART * 16 <= LDS_BYTES;
    __shared__ __attribute__((aligned(16))) char
        lds[APART ? ROUND * XBLOCK + SETS * PART * 16
                  : (ROUND * XBLOCK > SETS * PART * 16 ? ROUND * XBLOCK : SETS * PART * 16)];
    f4* const part = (f4*)(lds + (APART ? ROUND * XBLOCK : 0));
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE;
    const int r = lane & 15, g = lane >> 4;
    const int steps = a.K >> 5, tiles = (a.N + 15) / 16, G = gridDim.x;
    // Chunk c of splits x 8, in pairs of steps (128 bytes of a weight row): the
    // first chunk_more chunks take a pair more than the others' chunk_pairs.
    // (By the host: as divisions here, 500 instructions of them, they stood
    // before the first load: M 16, packed, with the norm 2048 x 1536 8.0 -> 7.5
    // us, gate/up 13.9 -> 13.4; 1536 x 1536 4.2 -> 3.6.)
    const auto first_step = [&](int c) {
        return 2 * (c * a.chunk_pairs + (c < a.chunk_more ? c : a.chunk_more));
    };
    const int c = blockIdx.y * GEMM_WAVES + wv;
    const int S0 = first_step(blockIdx.y * GEMM_WAVES);      // the group's first
    const int begin = first_step(c), end = first_step(c + 1);
    const int ns = (end < steps ? end : steps) - begin;      // at most SPW (host)
    // (fewer pairs than waves leave the last chunks empty: they stay at the
    // group's first step, so that no address is past the row)
    const int s0 = ns > 0 ? begin : S0;

    // W of a tile.  Packed: a step is 1 KiB in the order the lanes take it.
    // Row-major: lane (r, g) needs 16 bytes of row r a step; so that an
    // instruction reads whole 128-byte lines, lanes r and r ^ 1 load both
    // steps of a pair from row r & ~1, then from row r | 1 (the even lane the
    // first step's bytes, the odd lane the second's), and exchange what the
    // other needs when the tile is consumed (w_pair).
    constexpr uint32_t PAST = 0x80000000u;             // past every resource
    const bool odd = lane & 1;
    u4 wb[SETS][SPW];
    auto load_w = [&](int b, int tile) {
        const int t = tile < tiles ? tile : 0;
        const int bytes = tile < tiles ? 0x7fffffff : 0;
        if constexpr (PW) {
            const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
                (void*)wave_uniform((const half_t*)a.w + ((int64_t)t * steps + s0) * WAVE * 8), 0,
                bytes, 0x00020000);
#pragma unroll
            for (int i = 0; i < SPW; ++i)
                wb[b][i] = __builtin_bit_cast(
                    u4, __builtin_amdgcn_raw_buffer_load_b128(
                            rs, lane * 16 + (i < ns ? (uint32_t)(i * WAVE * 16) : PAST), 0,
                            W_POLICY));
        } else if constexpr (FAR) {
            // (a step past the chunk or a tile past the walk rereads and is
            // dropped)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const half_t* row = (const half_t*)a.w +
                                    (int64_t)w_row<EPI>(a, t, (r & ~1) + h) * a.ldw + 32 * s0 + 8 * g;
#pragma unroll
                for (int q = 0; q < SPW / 2; ++q) {
                    const int st = 2 * q + (odd ? 1 : 0);
                    const u4 v = *(const u4*)(row + 32 * (st < ns ? st : 0));
                    const uint32_t live = st < ns ? ~0u : 0u;
                    wb[b][2 * q + h] = v & (u4){live, live, live, live};
                }
            }
        } else {
            // (the tile's first row is the same in every lane)
            const int row0 = w_row<EPI>(a, t, 0);
            const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
                (void*)wave_uniform((const half_t*)a.w + (int64_t)row0 * a.ldw + 32 * s0), 0, bytes,
                0x00020000);
            const uint32_t piece = 16 * g + (odd ? 64 : 0);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int row = w_row<EPI>(a, t, (r & ~1) + h);
                const uint32_t off = (uint32_t)((int64_t)(row - row0) * a.ldw * 2) + piece;
#pragma unroll
                for (int q = 0; q < SPW / 2; ++q)
                    wb[b][2 * q + h] = __builtin_bit_cast(
                        u4, __builtin_amdgcn_raw_buffer_load_b128(
                                rs, off + (2 * q + (odd ? 1 : 0) < ns ? 128u * q : PAST), 0,
                                W_POLICY));
            }
        }
    };
    // The lane's operands of the steps of pair q.
    auto w_pair = [&](int b, int q, u4& first, u4& second) {
        const u4 x = wb[b][2 * q], y = wb[b][2 * q + 1];
        if constexpr (PW) {
            first = x;
            second = y;
        } else {
            const u4 give = odd ? x : y;
            const uint32_t gw[4] = {give.x, give.y, give.z, give.w};
            uint32_t tw[4];
#pragma unroll
            for (int e = 0; e < 4; ++e)      // lane ^ 1 (quad_perm 1, 0, 3, 2)
                tw[e] = __builtin_amdgcn_update_dpp(0, gw[e], 0xB1, 0xF, 0xF, false);
            const u4 take = {tw[0], tw[1], tw[2], tw[3]};
            first = odd ? take : x;
            second = odd ? y : take;
        }
    };
    // X, in whole rows of the group's K range (1 KiB of one row an instruction,
    // rows past M repeating the last, columns past K the last: neither is used)
    // and back in MFMA order: loaded straight to registers, an instruction
    // covers 64 bytes of each of 16 rows, from every CU at once, and that cost
    // 1.5 us a column block at K 1536.  Groups start at different rows and
    // columns, so that the CUs of an XCD do not ask one L2 channel for the
    // same line together.
    u4 xb[SPW][MB];
    auto stage = [&](int first) {
#pragma unroll
        for (int q = 0; q < ROUND; ++q) {
            const int mb = first + q;
            if (mb >= MB) break;
#pragma unroll
            for (int j = 0; j < SPW; ++j) {
                const int row = 2 * ((wv + blockIdx.x) % 8) + j / (SPW / 2);
                const int piece = (j + blockIdx.x) % (SPW / 2);
                const int m = 16 * mb + row < a.M ? 16 * mb + row : a.M - 1;
                const int col = 32 * S0 + 512 * piece + 8 * lane;
                __builtin_amdgcn_global_load_lds(
                    (const void*)((const half_t*)a.x + (int64_t)m * a.ldx +
                                  (col < a.K - 8 ? col : a.K - 8)),
                    (__attribute__((address_space(3))) void*)(lds + q * XBLOCK + row * PITCH +
                                                              1024 * piece),
                    16, 0, 0);
            }
        }
    };
    auto unstage = [&](int first) {
#pragma unroll
        for (int q = 0; q < ROUND; ++q) {
            const int mb = first + q;
            if (mb >= MB) break;
#pragma unroll
            for (int i = 0; i < SPW; ++i)
                xb[i][mb] = *(const u4*)(lds + q * XBLOCK + r * PITCH +
                                         (s0 - S0 + (i < ns ? i : 0)) * 64 + 16 * g);
        }
    };
    // (the largest kernel has no registers for them and loads them late)
    constexpr bool AHEAD = EPI == GEMM_ROPE && SPW * MB < GEMM_MAX_SPW * GEMM_MAX_M / 16;
    RopeAhead ra;
    if constexpr (AHEAD) {
        rope_row(a, 16 * wv + r, ra);
        __builtin_amdgcn_sched_barrier(0);
    }
    stage(0);
    __builtin_amdgcn_sched_barrier(0);
    // the norm prologue's residual rows and weight: the two rows the wave
    // staged, the lane's 8 channels of each piece
    constexpr int PIECES = SPW / 2;
    const int row2 = 2 * ((wv + blockIdx.x) % 8);
    u4 rv[NRM ? 2 : 1][PIECES], nw[PIECES];
    if constexpr (NRM) {
#pragma unroll
        for (int q = 0; q < PIECES; ++q) {
            const int col = 512 * q + 8 * lane < a.K - 8 ? 512 * q + 8 * lane : a.K - 8;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int m = row2 + h < a.M ? row2 + h : a.M - 1;
                rv[h][q] = *(const u4*)((const half_t*)a.nres + (int64_t)m * a.ldr + col);
            }
            nw[q] = *(const u4*)((const half_t*)a.nw + col);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int u = 0; u < SETS; ++u) load_w(u, blockIdx.x + u * G);
    if constexpr (AHEAD) {
        // (the position is here: only X, the norm's operands and W are after it)
        wait_vm_lds<ROUND * SPW + (NRM ? 3 * PIECES : 0) + SETS * SPW>();
        rope_tile(a, blockIdx.x, lane, ra);
        __builtin_amdgcn_sched_barrier(0);
    }
    wait_vm_lds<SETS * SPW + (AHEAD ? ROPE_TILE_VM : 0)>();  // X has landed, W is on its way
    if constexpr (NRM) {
        // Every group normalises the rows itself, a wave the two it staged.
        // s = res + x in packed fp16 (the fp32 sum of two fp16 values rounds
        // to the same fp16), its squares summed over the row by v_dot2 and a
        // wave reduction, then h = fp16(w * fp16(s / rms)) over the row in
        // LDS: the rounding of Qwen2RMSNorm in fp16.  Group 0 stores s.
        u4 sv[2][PIECES];
        float ss[2] = {0.f, 0.f};
        // (the rows read together, s stored last, the sums by DPP: a read and a
        // branch a piece and exchanges through LDS were a chain of LDS round
        // trips, M 16: gate/up 13.4 -> 12.8 us, q/k/v 7.5 -> 7.2)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int q = 0; q < PIECES; ++q)
                sv[h][q] = *(const u4*)(lds + (row2 + h) * PITCH + 1024 * q + 16 * lane);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int q = 0; q < PIECES; ++q) {
                const u4 x = sv[h][q];
                const bool mine = 512 * q + 8 * lane < a.K;
                const uint32_t xw[4] = {x.x, x.y, x.z, x.w};
                const uint32_t rw[4] = {rv[h][q].x, rv[h][q].y, rv[h][q].z, rv[h][q].w};
                uint32_t sw[4];
                float acc = 0.f;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const h2 t = __builtin_bit_cast(h2, rw[e]) + __builtin_bit_cast(h2, xw[e]);
                    acc = __builtin_amdgcn_fdot2(t, t, acc, false);
                    sw[e] = __builtin_bit_cast(uint32_t, t);
                }
                sv[h][q] = (u4){sw[0], sw[1], sw[2], sw[3]};
                ss[h] += mine ? acc : 0.f;
            }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const float inv = 1.f / sqrtf(wave_sum_dpp(ss[h]) / (float)a.K + a.eps);
#pragma unroll
            for (int q = 0; q < PIECES; ++q)
                *(u4*)(lds + (row2 + h) * PITCH + 1024 * q + 16 * lane) =
                    norm_row(sv[h][q], nw[q], inv);
        }
        if (blockIdx.x == 0)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int q = 0; q < PIECES; ++q)
                    if (512 * q + 8 * lane < a.K && row2 + h < a.M)
                        *(u4*)((half_t*)a.nres_out + (int64_t)(row2 + h) * a.ldro + 512 * q +
                               8 * lane) = sv[h][q];
    }
    __syncthreads();
    unstage(0);
#pragma unroll
    for (int first = ROUND; first < MB; first += ROUND) {
        __syncthreads();
        stage(first);
        wait_vm_lds<0>();
        __syncthreads();
        unstage(first);
    }
    __builtin_amdgcn_sched_barrier(0);
    // (steps past the chunk are zeros, as W's there)
#pragma unroll
    for (int i = 0; i < SPW; ++i) {
        const uint32_t live = i < ns ? ~0u : 0u;
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) xb[i][mb] &= (u4){live, live, live, live};
    }
    if constexpr (!APART) __syncthreads();

    // One tile from register set u; MORE: the tile SETS on is requested into
    // it as soon as its weights are consumed.
    auto do_tile = [&](auto set, auto more, int tile) {
        constexpr int u = decltype(set)::value;
        constexpr bool MORE = decltype(more)::value;
        f4 acc[MB];
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[mb] = (f4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < SPW / 2; ++q) {
            u4 w[2];
            w_pair(u, q, w[0], w[1]);
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) {
                    const u4 x = xb[2 * q + h][mb];
                    acc[mb] = mfma16(as_h4(w[h].x, w[h].y), as_h4(x.x, x.y), acc[mb]);
                    acc[mb] = mfma16(as_h4(w[h].z, w[h].w), as_h4(x.z, x.w), acc[mb]);
                }
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (MORE) load_w(u, tile + SETS * G);
        __builtin_amdgcn_sched_barrier(0);
        f4* const pt = part + u * PART;
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) pt[(wv * MB + mb) * WAVE + lane] = acc[mb];
        __syncthreads();
        // (the next tile's sums go to another buffer; this one is written
        // again only after the next barrier, past these reads)
        if (wv < MB) {
            // (read together, where registers allow: left to the compiler, each
            // read waited for the sum before it; with the tile counts by the
            // host and a barrier less, M 16: gate/up 12.8 -> 12.5 us, q/k/v 6.9
            // -> 6.7)
            f4 v[GEMM_WAVES];
#pragma unroll
            for (int p = 0; p < GEMM_WAVES; ++p) v[p] = pt[(p * MB + wv) * WAVE + lane];
            if constexpr (SPW * MB < GEMM_MAX_SPW * GEMM_MAX_M / 16) __builtin_amdgcn_sched_barrier(0);
            f4 s = v[0];
#pragma unroll
            for (int p = 1; p < GEMM_WAVES; ++p) s += v[p];
            if constexpr (EPI == GEMM_ROPE && !AHEAD) {
                rope_row(a, 16 * wv + r, ra);
                rope_tile(a, tile, lane, ra);
            }
            if (EPI != GEMM_PLAIN || a.splits == 1) {
                finish_tile<EPI>(a, tile, wv, lane, s, ra);
            } else {
                // write-through (sc1), 1 KiB of its own a wave (by a builtin: a
                // store in inline asm is not counted by the compiler, whose
                // next wait for W would then also wait for the tile just
                // requested)
                const __amdgpu_buffer_rsrc_t rs =
                    coherent_rsrc(wave_uniform(part_tile<MB>(a, blockIdx.y, tile) + wv * WAVE * 4));
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, s), rs, lane * 16, 0,
                                                       16);
            }
        }
        if constexpr (AHEAD) rope_tile(a, tile + G, lane, ra);
    };
    // (tiles in pairs, a last odd one after the loop: with an exit inside the
    // pair, the compiler merges it with the loop's own and then waits for
    // every load in flight at the top of each pair)
    using std::integral_constant;
    const int mine = a.walk + ((int)blockIdx.x < a.walk_more ? 1 : 0);
    int tile = blockIdx.x;
    for (int p = 0; p < mine / SETS; ++p, tile += SETS * G) {
        do_tile(integral_constant<int, 0>(), std::true_type(), tile);
        do_tile(integral_constant<int, 1>(), std::true_type(), tile + G);
    }
    if (mine % SETS) do_tile(integral_constant<int, 0>(), std::false_type(), tile);
    if (EPI != GEMM_PLAIN || a.splits == 1) return;

    // ---- split K: every partial of the group's tiles is stored through to
    // memory, then it arrives at each tile (a wave a tile), and the last group
    // of a tile to arrive sums its partials in split order ----
    handoff_release();
    __syncthreads();
    for (int q = wv; q < mine; q += GEMM_WAVES) {
        const int t = blockIdx.x + q * G;
        int prev = 0;
        if (lane == 0)
            prev = __hip_atomic_fetch_add(a.counters + t, 1u, __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_AGENT);
        prev = __builtin_amdgcn_readfirstlane(prev);
        if (prev != a.splits - 1) continue;
        f4 sum[MB];
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) sum[mb] = (f4){0.f, 0.f, 0.f, 0.f};
        if (a.splits <= 4)
            add_partials<4, MB>(a, t, lane, sum);
        else
            add_partials<8, MB>(a, t, lane, sum);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) finish_tile<EPI>(a, t, mb, lane, sum[mb], ra);
        // back to zero for the next launch
        if (lane == 0)
            __hip_atomic_store(a.counters + t, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

template <int MB, int EPI, bool PW, bool NRM = false>
void launch_spw(const GemmParams& p, int spw, dim3 grid, hipStream_t stream) {
    const dim3 block(GEMM_WAVES * WAVE);
    // (K up to 512: a group stages no more of X than it has.  us, four steps ->
    // two: 1000 x 96 at M 64 4.93 -> 3.77, 16384 x 256 at M 64 8.46 -> 7.01, 4096 x
    // 512 at M 64 5.56 -> 4.46.  The other epilogues, whose K is a hidden size,
    // have no such form.)
    constexpr int FEW = EPI == GEMM_PLAIN && !NRM ? 2 : 4;
    if (FEW == 2 && spw <= 2)
        hipLaunchKernelGGL((decode_gemm_kernel<FEW, MB, EPI, PW, NRM, false>), grid, block, 0, stream, p);
    else if (spw <= 4)
        hipLaunchKernelGGL((decode_gemm_kernel<4, MB, EPI, PW, NRM, false>), grid, block, 0, stream, p);
    else if (spw <= 6)
        hipLaunchKernelGGL((decode_gemm_kernel<6, MB, EPI, PW, NRM, false>), grid, block, 0, stream, p);
    else
        hipLaunchKernelGGL((decode_gemm_kernel<8, MB, EPI, PW, NRM, false>), grid, block, 0, stream, p);
}

template <int MB, int EPI>
void launch_mb(const GemmParams& p, int spw, bool far, dim3 grid, hipStream_t stream) {
    if (p.w_packed)
        launch_spw<MB, EPI, true>(p, spw, grid, stream);
    else if (!far)
        launch_spw<MB, EPI, false>(p, spw, grid, stream);
    else
        hipLaunchKernelGGL((decode_gemm_kernel<GEMM_MAX_SPW, MB, EPI, false, false, true>), grid,
                           dim3(GEMM_WAVES * WAVE), 0, stream, p);
}

// The launch of one epilogue's kernels: `spw` steps a wave at most.
template <int EPI>
hipError_t launch_epilogue(const GemmParams& p, int spw, dim3 grid, hipStream_t stream) {
    // a lane's byte offset from its tile's first row must stay below 2^31
    const int64_t rows = EPI == GEMM_GLU ? (int64_t)p.N / 2 + 8 : EPI == GEMM_ROPE ? p.rope.d : 16;
    const bool far = !p.w_packed && rows * p.ldw * 2 + (int64_t)p.K * 2 >= (1LL << 31);
    if (p.norm)
        launch_spw<1, EPI, true, true>(p, spw, grid, stream);
    else if (p.M <= 16)
        launch_mb<1, EPI>(p, spw, far, grid, stream);
    else if (p.M <= 32)
        launch_mb<2, EPI>(p, spw, far, grid, stream);
    else if (p.M <= 48)
        launch_mb<3, EPI>(p, spw, far, grid, stream);
    else
        launch_mb<4, EPI>(p, spw, far, grid, stream);
    return hipGetLastError();
}

}  // namespace

}  // namespace ls
