// The decode GEMM's host side (ls_gemm_kernel.h has the kernel): launch
// shapes, the split of K, weight packing.
//
// The reference runs these projections as torch (cuBLAS) GEMMs inside its
// model layers (model/fused.py, model/latentserve_qwen.py), the activation
// as silu_and_mul (kernels/fused_elementwise.py:222-233) and the decode
// token's rope_qk and cache write in its attention layer
// (model/attention/gqa.py:251-253, cache/paged_cache.py write).
#include "ls_common.h"
#include "ls_gemm.h"
#include "ls_gemm_tile.h"

namespace ls {

namespace {

// One group a CU over the splits of K together.
int gemm_groups(int splits, int tiles) {
    const int g = 256 / splits;
    return g < 1 ? 1 : g > tiles ? tiles : g;
}

int gemm_splits(int N, int K) {
    const int steps = K / 32, tiles = (N + 15) / 16;
    const int lo = (steps + GEMM_WAVES * GEMM_MAX_SPW - 1) / (GEMM_WAVES * GEMM_MAX_SPW);
    if (lo == 1) return 1;
    // A group's work is its tiles (at most `most` a group) and its X, over its
    // share of K; more splits even it out until their partials cost more than
    // they save.  X weighs two tiles.  (M 48, us at 5 / 6 / 7 / 8 / 10 splits:
    // 1536 x 8960 14.2 / 13.1 / 12.8 / 13.3 / 15.0; at 2 / 3 / 4 / 5: 1024 x
    // 2816 8.2 / 7.6 / 7.9 / 8.8, 3584 x 3584 12.7 / 12.2 / 11.5 / 13.3; at 3 /
    // 4 / 5: 2048 x 5632 12.7 / 11.2 / 12.4.)
    int best = lo;
    int64_t cost = INT64_MAX;
    for (int s = lo; s <= lo + 2; ++s) {
        const int groups = gemm_groups(s, tiles);
        const int most = (tiles + groups - 1) / groups;
        const int64_t c = (int64_t)(most + 2) * ((steps + s - 1) / s);
        if (c < cost) {
            cost = c;
            best = s;
        }
    }
    return best;
}

// Packed weights (gemm_packed_bytes): tile T's step s is 64 lanes x 16 B at
// ((T * steps + s) * 64 + lane) * 8 halves.
constexpr int GEMM_PACK_TILES = 4;    // tiles padded to a multiple of this

// grid (padded tiles, steps), 64 threads: lane (r, g) copies row r's
// channels 8g .. 8g + 7 of the step (zeros for rows past the weight).
template <int EPI>
__global__ __launch_bounds__(64) void pack_gemm_kernel(const half_t* w, int64_t ldw, int N, int K,
                                                       int d, half_t* out) {
    const int T = blockIdx.x, s = blockIdx.y, lane = threadIdx.x, r = lane & 15, g = lane >> 4;
    const int steps = K / 32;
    bool real;
    const int row = w_row_of<EPI>(N, d, T, r, real);
    u4 v = {0u, 0u, 0u, 0u};
    if (real) v = *(const u4*)(w + (int64_t)row * ldw + 32 * s + 8 * g);
    *(u4*)(out + (((int64_t)T * steps + s) * WAVE + lane) * 8) = v;
}

}  // namespace

size_t gemm_packed_bytes(int N, int K, int epi, int head_dim) {
    (void)epi;
    (void)head_dim;
    const int tiles = (N + 15) / 16;
    const int padded = (tiles + GEMM_PACK_TILES - 1) / GEMM_PACK_TILES * GEMM_PACK_TILES;
    return (size_t)padded * (K / 32) * WAVE * 16;
}

hipError_t launch_pack_gemm_weight(const void* w, int64_t ldw, int N, int K, int epi, int head_dim,
                                   void* packed, hipStream_t stream) {
    const int tiles = (N + 15) / 16;
    const int padded = (tiles + GEMM_PACK_TILES - 1) / GEMM_PACK_TILES * GEMM_PACK_TILES;
    const dim3 grid(padded, K / 32);
    if (epi == GEMM_GLU)
        hipLaunchKernelGGL(pack_gemm_kernel<GEMM_GLU>, grid, dim3(WAVE), 0, stream,
                           (const half_t*)w, ldw, N, K, head_dim, (half_t*)packed);
    else if (epi == GEMM_ROPE)
        hipLaunchKernelGGL(pack_gemm_kernel<GEMM_ROPE>, grid, dim3(WAVE), 0, stream,
                           (const half_t*)w, ldw, N, K, head_dim, (half_t*)packed);
    else
        hipLaunchKernelGGL(pack_gemm_kernel<GEMM_PLAIN>, grid, dim3(WAVE), 0, stream,
                           (const half_t*)w, ldw, N, K, head_dim, (half_t*)packed);
    return hipGetLastError();
}

int decode_gemm_splits(int M, int N, int K) {
    (void)M;
    return gemm_splits(N, K);
}

int decode_gemm_units(int M, int N, int K) {
    (void)M;
    (void)K;
    return (N + 15) / 16;
}

size_t decode_gemm_workspace_bytes(int M, int N, int K) {
    const int splits = gemm_splits(N, K);
    if (splits == 1) return 0;
    // whole tiles: 1 KiB a (split, tile, column block)
    return GEMM_PART_OFFSET + (size_t)splits * ((N + 15) / 16) * ((M + 15) / 16) * WAVE * sizeof(f4);
}

hipError_t launch_decode_gemm(const GemmParams& params, hipStream_t stream) {
    if (params.M == 0 || params.N == 0) return hipSuccess;
    GemmParams p = params;
    const int steps = p.K / 32, tiles = (p.N + 15) / 16;
    if (p.splits != gemm_splits(p.N, p.K)) return hipErrorInvalidValue;
    const int pairs = (steps + 1) / 2, chunks = p.splits * GEMM_WAVES;
    p.chunk_pairs = pairs / chunks;
    p.chunk_more = pairs % chunks;
    // steps a wave takes at most
    const int spw = 2 * (p.chunk_pairs + (p.chunk_more ? 1 : 0));
    if (spw > GEMM_MAX_SPW || p.M > GEMM_MAX_M) return hipErrorInvalidValue;
    // the norm prologue: a packed weight, one column block, a group covering
    // the whole row
    if (p.norm && (!p.w_packed || p.M > 16 || p.splits != 1)) return hipErrorInvalidValue;
    const dim3 grid(gemm_groups(p.splits, tiles), p.splits);
    p.walk = tiles / grid.x;
    p.walk_more = tiles % grid.x;
    if (p.epi == GEMM_GLU) {
        if (p.splits != 1 || p.N % 2 != 0) return hipErrorInvalidValue;
        return launch_gemm_glu(p, spw, grid, stream);
    }
    if (p.epi == GEMM_ROPE) {
        if (p.splits != 1 || p.N % 16 != 0 || p.rope.d % 16 != 0) return hipErrorInvalidValue;
        RopeWriteParams& w = p.rope;
        const auto at = [](const void* x) { return (uintptr_t)x; };
        w.ahead = w.st >= 0 && w.st % 2 == 0 && (int64_t)w.tab_rows * w.st < (1LL << 30) - w.d &&
                  p.N < (1 << 30) && (at(w.cos) | at(w.sin) | at(p.bias)) % 4 == 0;
        w.vec_out = (at(w.q_out) | at(w.k_pool) | at(w.v_pool)) % 8 == 0 &&
                    (w.sq_b | w.sq_h | w.sq_r | w.sp_b | w.sp_t | w.sp_h) % 4 == 0;
        return launch_gemm_rope(p, spw, grid, stream);
    }
    return launch_gemm_plain(p, spw, grid, stream);
}

}  // namespace ls
