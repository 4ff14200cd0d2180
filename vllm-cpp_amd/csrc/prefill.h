// prefill.h -- internal launch interface of the chunked prefill kernel.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "vcpp_attention.h"

namespace vcpp {

struct PrefillParams {
    // KV pages (see vcpp_kv_pages)
    const void* k;
    const void* v;
    const uint16_t* k_scale;
    const uint16_t* v_scale;
    int64_t num_blocks;
    int64_t block_stride;
    int64_t scale_block_stride;
    int32_t block_size;
    int32_t num_kv_heads;
    int32_t head_dim;
    int32_t kv_dtype;
    // queries (fp16 [rows][num_heads][head_dim]) and fp32 outputs
    const uint16_t* q;
    float* out;
    int32_t num_heads;
    int32_t group;        // num_heads / num_kv_heads
    int32_t head_groups;  // workgroups per kv head (4 query heads each)
    // chunks
    const int32_t* block_tables;  // [num_chunks][max_blocks]
    const int32_t* q_start;       // [num_chunks + 1] device
    const int32_t* prefix_lens;   // [num_chunks] device
    int32_t max_blocks;
    int32_t num_chunks;
    int32_t max_chunk_len;
    float scale_log2;  // log2(e) / sqrt(head_dim)
    // split-K over the keys (1: none): part k of a tile's key blocks leaves
    // unnormalised outputs and (max, sum) in ws_o / ws_ml at row
    // k * rows_cap + row, for launch_prefill's merge
    int32_t splits;
    int32_t live;      // 1: in 1 .. splits parts, by the chunks' real lengths (live_splits)
    int32_t rows_cap;  // >= the rows of all chunks (num_chunks * max_chunk_len)
    float* ws_o;       // [splits][rows_cap][num_heads][head_dim]
    float2* ws_ml;     // [splits][rows_cap][num_heads] (max in log2 units, sum)
    uint64_t bs_magic; // ceil(2^40 / block_size): pos / block_size = (pos * bs_magic) >> 40
    int32_t xcd_cus;   // CUs per XCD (0: unknown; no pairing of heavy and light tiles)
    int32_t tile_rows; // query rows per workgroup tile (set by launch_prefill for the merge)
#ifdef VCPP_GATHER_DUMP
    int32_t* gather_dump;    // checker builds: [rows][gather_stride][2] (block, slot)
    int64_t gather_stride;
#endif
};

// Cost of a split call in s key parts, of `items` workgroups a part whose
// longest keys are `keys` and whose keys sum to `work`, in units of one 32-key
// block of two resident workgroups per CU (about 1.3 us): a round of a part's
// blocks, 0.72 of that where the last round leaves one workgroup per CU, or
// (uneven prefixes) the blocks spread evenly and half the longest part's after
// them; 5 for a round's start and end, and the partials' traffic.  The fullest
// count is not the best where it spills a few workgroups into a round of their
// own: 48 tiles in 11 parts are 528 workgroups, 56.0 us for three 40-token
// chunks on 7000-token prefixes (32/8 heads of 128), 41.9 in 10 parts; but 384
// tiles (three 500-token chunks on 8192, 64/8 heads of 80) take 365 us whole
// and 325 in two parts.  Every count of drawn calls was timed: over 3746 calls
// of up to 3 chunks the count of least cost takes 1.0015 of the best one's time
// in the geometric mean (the fullest one 1.038), over 5286 of 4 to 64 chunks
// 1.003 (1.026; by rounds of the longest keys alone 1.0065).
// (full: items * s / (2 * cus), whole rounds.)
__host__ __device__ inline float prefill_split_cost(int s, int items, int full, float keys, float work,
                                                    float out_values, int cus) {
    const int slots = 2 * cus, rest = items * s - full * slots;
    const float part = keys / (32.f * s);
    const float rounds = part * (full + (rest == 0 ? 0.f : rest <= cus ? 0.72f : 1.f));
    const float even = work / (32.f * slots) + 0.5f * part;
    return (rounds < even ? rounds : even) + 5.f * (full + (rest > 0)) + (s > 1 ? s * out_values * (8.f / 6.5e6f) : 0.f);
}

hipError_t launch_prefill(const PrefillParams& p, hipStream_t stream);
// Workspace bytes of a split prefill (0 when splits <= 1).
// Most key parts a split prefill cuts a query tile into.
constexpr int kMaxPrefillSplits = 16;
size_t prefill_split_bytes(int splits, int rows_cap, int num_heads, int head_dim);
int prefill_head_groups(int group);
// Whether fp16 pages of this shape run prefill_wide_kernel (128-row tiles)
// rather than prefill_dma_kernel, and the query rows per workgroup tile of
// the kernel that serves them.
bool prefill_uses_wide(int kv_dtype, int head_dim, int block_size);
int prefill_tile_rows(int kv_dtype, int head_dim, int block_size);
size_t prefill_ring_bytes(int kv_dtype, int head_dim);
// Dynamic LDS bytes of the prefill kernel for a table of max_blocks entries
// (the larger of the two kernels' needs where both serve the dtype).
size_t prefill_lds_bytes(int kv_dtype, int head_dim, int max_blocks);

}  // namespace vcpp
