// INT8 KV cache write side on gfx950: the decode-step write (V quantized per
// token into the pool, K copied into the fp16 last-page residual), a prefill
// chunk's write (V and the complete pages' K quantized, the last page's K to
// the residual) and the per-block K quantizer that runs when a page completes.
//
// Reference: kernels/cuda/int8_write.cu:46-80 (int8_decode_write, launched by
// kernels/cuda/int8_write.py:61-82) and cache/int8_paged_cache.py:670-699
// (_finalize_blocks), :741-758 (write(), V part).
//
// Codes are bit-exact with the reference's torch ops: fp32 throughout, every
// multiply / add / divide rounded on its own (no contraction), rintf for
// torch.round (half to even), the same epsilon floor.  One choice is left to
// the caller: torch divides a tensor by a Python number on the GPU as a
// multiply by the fp32 reciprocal formed on the host, and on the CPU as a
// true division (they differ in the last bit of a few percent of scales).
// `recip` = 1 reproduces the GPU form (what the reference stores when it runs
// on a GPU, and what its int8_write.cu computes); 0 the CPU form.
//
// Layout: one wave per (row, head) of 128 channels, two channels a lane; the
// row's max / min is a wave reduction (no LDS).  HBM-bound byte work.
#include "ls_common.h"
#include "ls_int8_write.h"

#pragma clang fp contract(off)

namespace ls {

namespace {

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, shfl_xor(v, o));
    return v;
}
__device__ __forceinline__ float wave_min(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fminf(v, shfl_xor(v, o));
    return v;
}

struct QuantStep {
    float step, zero, lo;
};

// Scale (and zero point) of one row from its max |x| (sym) or min / max (asym).
__device__ __forceinline__ QuantStep fit(float amax, float lo, float hi, const QuantArgs& q) {
    QuantStep s;
    s.lo = lo;
    s.zero = 0.f;
    if (!q.asym) {
        const float m = fmaxf(amax, q.eps);                       // clamp_min(eps)
        s.step = q.recip ? m * q.inv_qmax : m / q.qmax;           // / qmax
    } else {
        const float r = hi - lo;
        const float t = q.recip ? r * q.inv_levels : r / q.levels;  // / levels
        s.step = fmaxf(t, q.eps);                                  // clamp_min(eps)
        s.zero = lo + q.offset * s.step;
    }
    return s;
}

__device__ __forceinline__ int8_t code(float x, const QuantStep& s, const QuantArgs& q) {
    if (!q.asym) {
        const float r = rintf(x / s.step);
        return (int8_t)(int)fminf(fmaxf(r, -q.qmax), q.qmax);
    }
    const float u = fminf(fmaxf(rintf((x - s.lo) / s.step), 0.f), q.levels);
    return (int8_t)(int)(u - q.offset);
}

// One wave per (b, h): grid (ceil(B * H / 4)), 256 threads.  A few kilobytes:
// bound by the launch and by its chain of memory round trips, so everything it
// reads is requested at once (the residual row, then K, after V's
// quantization were two trips more: 4.80 -> 4.71 us between two decode
// launches of a graph, most of them the launch).
__global__ __launch_bounds__(256) void decode_write_kernel(DecodeWriteParams a) {
    const int lane = threadIdx.x & 63;
    // (B * H rows of 256 bytes in memory: 32 bits hold it, and a 64-bit
    // division is a hundred instructions)
    const unsigned row = blockIdx.x * 4 + (threadIdx.x >> 6);
    const unsigned H = a.H;
    const int b = (int)(row / H), h = (int)(row % H);
    if (b >= a.B) return;
    const int d = 2 * lane;
    const h2 vv = *(const h2*)((const half_t*)a.v + (int64_t)b * a.sv_b + (int64_t)h * a.sv_h + d);
    const h2 kk = *(const h2*)((const half_t*)a.k + (int64_t)b * a.sk_b + (int64_t)h * a.sk_h + d);
    const int64_t slot = a.slots[b];
    const int64_t ri = a.res_idx[b];
    issue_here();
    // K into the fp16 residual: its page is quantized when it completes.
    if (ri >= 0 && ri < a.num_res) *(h2*)((half_t*)a.k_res + (ri * a.H + h) * HEAD_DIM + d) = kk;
    const float x0 = (float)vv.x, x1 = (float)vv.y;
    if (slot >= 0 && slot < a.num_slots) {
        float amax = 0.f, lo = 0.f, hi = 0.f;
        if (!a.q.asym) {
            amax = wave_max(fmaxf(fabsf(x0), fabsf(x1)));
        } else {
            hi = wave_max(fmaxf(x0, x1));
            lo = wave_min(fminf(x0, x1));
        }
        const QuantStep s = fit(amax, lo, hi, a.q);
        const int64_t r = slot * a.H + h;            // flat [slots, H] row
        char2 c;
        c.x = code(x0, s, a.q);
        c.y = code(x1, s, a.q);
        *(char2*)((int8_t*)a.flat_v + r * HEAD_DIM + d) = c;
        if (lane == 0) {
            a.flat_v_scale[r] = s.step;
            if (a.q.asym) a.flat_v_zero[r] = s.zero;
        }
    }
}

// One page of one head's K quantized: two channels a lane (x[token][e]),
// step per channel over the 16 tokens; codes to dst (token stride sp_t),
// steps to ks[0..1] (zero points to kz[0..1] when asym).
__device__ __forceinline__ void quantize_page(float (&x)[PAGE][2], const QuantArgs& q, int8_t* dst,
                                              int64_t sp_t, float* ks, float* kz) {
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        float amax = 0.f, lo = x[0][e], hi = x[0][e];
#pragma unroll
        for (int t = 0; t < PAGE; ++t) {
            amax = fmaxf(amax, fabsf(x[t][e]));
            lo = fminf(lo, x[t][e]);
            hi = fmaxf(hi, x[t][e]);
        }
        const QuantStep s = fit(amax, lo, hi, q);
        ks[e] = s.step;
        if (q.asym) kz[e] = s.zero;
#pragma unroll
        for (int t = 0; t < PAGE; ++t) x[t][e] = (float)code(x[t][e], s, q);
    }
#pragma unroll
    for (int t = 0; t < PAGE; ++t) {
        char2 c;
        c.x = (int8_t)(int)x[t][0];
        c.y = (int8_t)(int)x[t][1];
        *(char2*)(dst + (int64_t)t * sp_t) = c;
    }
}

// One wave per (block n, head h): the 16 token rows, two channels a lane;
// step per (block, head, channel) over the 16 tokens.
__global__ __launch_bounds__(256) void finalize_k_kernel(FinalizeParams a) {
    const int lane = threadIdx.x & 63;
    const int64_t item = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (item >= (int64_t)a.N * a.H) return;
    const int64_t n = item / a.H;
    const int h = (int)(item % a.H);
    const int64_t blk = a.ids[n];
    if (blk < 0 || blk >= a.num_blocks) return;
    const int64_t src_n = a.rows ? a.rows[n] : n;
    if (a.rows && (src_n < 0 || src_n >= a.num_rows)) return;
    const int d = 2 * lane;
    const half_t* src = (const half_t*)a.data + src_n * a.sd_n + (int64_t)h * a.sd_h + d;
    float x[PAGE][2];
#pragma unroll
    for (int t = 0; t < PAGE; ++t) {
        const h2 v = *(const h2*)(src + (int64_t)t * a.sd_t);
        x[t][0] = (float)v.x;
        x[t][1] = (float)v.y;
    }
    const int64_t si = blk * a.ss_b + (int64_t)h * a.ss_h + d;
    quantize_page(x, a.q, (int8_t*)a.k_pool + blk * a.sp_b + (int64_t)h * a.sp_h + d, a.sp_t,
                  a.k_scale + si, a.q.asym ? a.k_zero + si : nullptr);
}

// A prefill chunk written in one launch: one wave per (sequence, page the
// chunk touches, head).  The wave quantizes its page's new V rows (16 lanes a
// token, 8 channels a lane, extrema over the 16 lanes), and assembles the
// page's K: rows the chunk brings, and for the chunk's first page the rows
// before it from the fp16 residual.  A page that is not the chunk's last is
// complete: its K is quantized into the pool.  The last page's K goes to the
// residual row whole (zeros past the end).  With a first page that reads the
// residual, its wave also takes the last page, after that read has been
// used, so no wave overwrites rows another still needs.
//
// Bound by latency at one prompt's size (1021 tokens of 2 heads: 128 waves),
// by HBM above: every byte is read and written once.  Before: per layer a
// copy of the chunk for V and for K, a fill, a page-by-page assembly in torch
// (a launch or two each) and the two quantizer launches; measured for 1021
// tokens in two chunks, 2 heads, 28 layers, launches and host work included:
// 5.56 -> 1.25 ms.
__global__ __launch_bounds__(256) void prefill_write_kernel(PrefillWriteParams a) {
    const int lane = threadIdx.x & 63;
    // (page, head) unit of the sequence blockIdx.y
    const int unit = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int h = unit % a.H, b = blockIdx.y;
    int p = unit / a.H;
    const int64_t* slots = a.slots + (int64_t)b * a.N;
    const int off = (int)(slots[0] & (PAGE - 1));            // the chunk's offset in its first page
    const int last = (off + a.N - 1) / PAGE;                 // the chunk's last page
    if (p > last || (p == last && p > 0 && off > 0)) return;
    const int64_t row = a.rows[b];
    const bool row_ok = row >= 0 && row < a.num_res;
    const int c = lane & 15, g = lane >> 4, d = 2 * lane;
    const half_t* kb = (const half_t*)a.k + (int64_t)b * a.sk_b + (int64_t)h * a.sk_h;
    const half_t* vb = (const half_t*)a.v + (int64_t)b * a.sv_b + (int64_t)h * a.sv_h;
    half_t* res = (half_t*)a.k_res + ((row_ok ? row * PAGE : 0) * a.H + h) * HEAD_DIM;
    const int64_t tok = (int64_t)a.H * HEAD_DIM;             // a token's elements in every pool
    while (true) {
        const int t0 = p * PAGE - off;                       // chunk token in the page's row 0
        const int64_t slot = slots[t0 < 0 ? 0 : t0];
        const int64_t blk = slot / PAGE;
        const bool blk_ok = slot >= 0 && blk < a.num_blocks;
        // V: lanes (g, c) hold rows 4j + g, channels 8c .. 8c + 7
        u4 vv[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int t = t0 + 4 * j + g, tc = t < 0 ? 0 : t < a.N ? t : a.N - 1;
            vv[j] = *(const u4*)(vb + (int64_t)tc * a.sv_t + 8 * c);
        }
        // K: row i, channels 2 lane, 2 lane + 1
        float x[PAGE][2];
#pragma unroll
        for (int i = 0; i < PAGE; ++i) {
            const int t = t0 + i;
            h2 v = {(half_t)0.f, (half_t)0.f};
            if (t >= 0 && t < a.N)
                v = *(const h2*)(kb + (int64_t)t * a.sk_t + d);
            else if (t < 0 && row_ok)
                v = *(const h2*)(res + i * tok + d);
            x[i][0] = (float)v.x;
            x[i][1] = (float)v.y;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t w[4] = {vv[j].x, vv[j].y, vv[j].z, vv[j].w};
            float y[8];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const h2 t = __builtin_bit_cast(h2, w[e]);
                y[2 * e] = (float)t.x;
                y[2 * e + 1] = (float)t.y;
            }
            float amax = 0.f, lo = 0.f, hi = 0.f;
            if (!a.qv.asym) {
#pragma unroll
                for (int e = 0; e < 8; ++e) amax = fmaxf(amax, fabsf(y[e]));
#pragma unroll
                for (int o = 8; o > 0; o >>= 1) amax = fmaxf(amax, shfl_xor(amax, o));
            } else {
                lo = hi = y[0];
#pragma unroll
                for (int e = 1; e < 8; ++e) {
                    lo = fminf(lo, y[e]);
                    hi = fmaxf(hi, y[e]);
                }
#pragma unroll
                for (int o = 8; o > 0; o >>= 1) {
                    lo = fminf(lo, shfl_xor(lo, o));
                    hi = fmaxf(hi, shfl_xor(hi, o));
                }
            }
            const QuantStep s = fit(amax, lo, hi, a.qv);
            const int i = 4 * j + g, t = t0 + i;
            if (blk_ok && t >= 0 && t < a.N) {
                u2 o = {0u, 0u};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    o.x |= (uint32_t)(uint8_t)code(y[e], s, a.qv) << (8 * e);
                    o.y |= (uint32_t)(uint8_t)code(y[4 + e], s, a.qv) << (8 * e);
                }
                const int64_t r = (blk * PAGE + i) * a.H + h;
                *(u2*)((int8_t*)a.v_pool + r * HEAD_DIM + 8 * c) = o;
                if (c == 0) {
                    a.v_scale[r] = s.step;
                    if (a.qv.asym) a.v_zero[r] = s.zero;
                }
            }
        }
        if (p < last) {
            if (blk_ok) {
                const int64_t si = (blk * a.H + h) * HEAD_DIM + d;
                quantize_page(x, a.qk, (int8_t*)a.k_pool + (blk * PAGE * a.H + h) * HEAD_DIM + d, tok,
                              a.k_scale + si, a.qk.asym ? a.k_zero + si : nullptr);
            }
            if (p > 0 || off == 0) return;
            p = last;                                        // the first page's wave: the last too
            continue;
        }
        if (row_ok) {
#pragma unroll
            for (int i = 0; i < PAGE; ++i)
                if (t0 + i >= 0)
                    *(h2*)(res + i * tok + d) = (h2){(half_t)x[i][0], (half_t)x[i][1]};
        }
        return;
    }
}

}  // namespace

hipError_t launch_decode_write(const DecodeWriteParams& p, hipStream_t stream) {
    const int64_t rows = (int64_t)p.B * p.H;
    if (rows == 0) return hipSuccess;
    hipLaunchKernelGGL(decode_write_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, stream,
                       p);
    return hipGetLastError();
}

hipError_t launch_prefill_write(const PrefillWriteParams& p, hipStream_t stream) {
    if (p.B == 0 || p.N == 0) return hipSuccess;
    // pages a chunk can touch: one more than its own where it starts in a page
    const int64_t units = (((int64_t)p.N + 2 * PAGE - 2) / PAGE) * p.H;
    hipLaunchKernelGGL(prefill_write_kernel, dim3((unsigned)((units + 3) / 4), p.B), dim3(256), 0,
                       stream, p);
    return hipGetLastError();
}

hipError_t launch_finalize_k(const FinalizeParams& p, hipStream_t stream) {
    const int64_t items = (int64_t)p.N * p.H;
    if (items == 0) return hipSuccess;
    hipLaunchKernelGGL(finalize_k_kernel, dim3((unsigned)((items + 3) / 4)), dim3(256), 0, stream,
                       p);
    return hipGetLastError();
}

hipError_t int8_write_resources(int what, KernelResources* r) {
    if (what == 0) return func_resources(decode_write_kernel, 256, r);
    if (what == 1) return func_resources(finalize_k_kernel, 256, r);
    if (what == 2) return func_resources(prefill_write_kernel, 256, r);
    return hipErrorInvalidValue;
}

}  // namespace ls
