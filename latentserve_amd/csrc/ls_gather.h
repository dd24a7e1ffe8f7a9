// Byte movement between a paged K/V cache and dense rows: the block-table
// gather of one pool or both into [B, L, H, D], and the write of new K/V rows
// to their slots.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ls {

struct GatherParams {
    const void* pool[2];           // [num_blocks, 16, H, D], `elem`-byte elements (K, V)
    int64_t sp_b, sp_t, sp_h;      // element strides
    int num_blocks;
    const int32_t* block_tables;
    int64_t sbt_b;
    int max_pages;
    const int32_t* seq_lens;
    void* out[2];                  // [B, L, H, D]
    int64_t so_b, so_t, so_h;      // element strides
    int elem, row_bytes;           // bytes per element, per (token, head) row (multiple of 16)
    int B, L, H;
    int pools;                     // 1 or 2
};

struct PagedWriteParams {
    const void* src[2];            // K, V [B, H, N, D]
    int64_t ss_b[2], ss_h[2], ss_t[2];
    const int64_t* slots;          // [B, N] flat token slots
    void* pool[2];                 // [num_blocks, 16, H, D]
    int64_t sp_b, sp_t, sp_h;
    int64_t num_blocks;
    int elem, row_bytes;
    int B, H, N;
};

hipError_t launch_gather(const GatherParams& p, hipStream_t stream);
hipError_t launch_paged_write(const PagedWriteParams& p, hipStream_t stream);

}  // namespace ls
