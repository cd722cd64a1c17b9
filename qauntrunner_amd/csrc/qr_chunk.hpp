// qr_chunk.hpp -- launch interface of the MFMA causal multi-query (chunk) kernels.
#pragma once

#include "qr_kernels.hpp"

namespace qr {

struct ChunkArgs {
    const void* pool;
    const int* page_table;  // device, entries of this (sequence, layer)
    PageGeom geom;          // planes = 2
    int kv_dtype;           // F16 or BF16 (any for the fp32 tiles)
    int heads;
    int pos0;               // position of query 0
    // Device-side position of query 0: when set the kernels read it, clamped to [0, pos0];
    // pos0 is then the largest position query 0 may take, which the plan is made for.
    const int* pos0_dev;
    int nq;
    const void* q;          // device [nq][heads][head_dim] in q_dtype
    int q_dtype;
    float* out;             // device [nq][heads][head_dim]
    float scale;
    // bytes that the split partials may take; the plans that came after the decode entries (fp32
    // tiles, groups that are not a power of two) use fewer splits when it is less than they want
    size_t room = ~size_t(0);
};

struct ChunkPlan {
    int nt;                 // 16-row N tiles per wave
    int pg;                 // fp32 tiles: waves that share a row group, one part of a tile's positions each
    int queries_per_block;
    int qblocks;
    int splits;
    int split_tokens;       // 16-bit tiles (the fp32 tiles spread each query block's own keys)
    size_t workspace_bytes;
};

// 16-bit cache, head_dim 64 or 128, power-of-two group heads/kv_heads <= 64.
bool chunk_mfma_eligible(int kv_dtype, int head_dim, int heads, int kv_heads);
// The same with any other group of up to 64, host positions only.
bool chunk_mfma_split_eligible(int kv_dtype, int head_dim, int heads, int kv_heads, int pos0, int nq);
ChunkPlan plan_chunk(const ChunkArgs& a);
// after_split: when not null, recorded on `stream` right after the main kernel.
hipError_t launch_chunk(const ChunkArgs& a, const ChunkPlan& plan, void* workspace, hipStream_t stream,
                        hipEvent_t after_split = nullptr);

// fp32 MFMA tiles (qr_chunk_f32.hip): fp32 caches and the 16-bit caches with token-major pages,
// head_dim 64/96/128/256.  Host positions only.  Below kChunkF32MinRows (query, head) rows per
// kv head most of a 16-row tile would be padding: one decode entry per query instead.
constexpr int kChunkF32MinRows = 8;
bool chunk_f32_eligible(int kv_dtype, int head_dim, int heads, int kv_heads, int pos0, int nq);
ChunkPlan plan_chunk_f32(const ChunkArgs& a);
hipError_t launch_chunk_f32(const ChunkArgs& a, const ChunkPlan& plan, void* workspace, hipStream_t stream,
                            hipEvent_t after_split = nullptr);

}  // namespace qr
