// Definitions of the suffix-attention kernels (miikv_suffix.hip): launch
// constants, argument blocks, the split-record layout and small device helpers.
#pragma once
#include "miikv_common.hpp"

namespace miikv {

// suffix_kernel's two forms: 8 waves (256 query rows) per workgroup, one workgroup per CU,
// and 4 waves (128 rows) with half the LDS, two workgroups per CU.
constexpr uint32_t kSufWaves = 8;
constexpr uint32_t kSufWavesSmall = 4;
constexpr uint32_t kSufStep = 32;              // keys per step
constexpr float kLog2eS = 1.4426950408889634f;
constexpr float kSlackS = 6.0f;        // lazy-rescale threshold (log2 units): p <= 64
// Resident waves of suffix_kernel on the chip: 256 CUs, two waves per SIMD (at <= 256
// VGPRs), in LDS tile buffers of 128 KiB per CU at D = 256.
constexpr uint32_t kSufResidentWaves = 256 * 8;
constexpr uint32_t kSufMaxSplits = 64;
constexpr uint32_t kSufMinKeys = 256;  // keys per split, at least: 8-wave form
constexpr uint32_t kSufMinKeysSmall = 160;  // 4-wave form
// Suffixes of at most this many decode row sets (tokens / tokens per evenly packed row set)
// run as a batch of decodes (miikv_decode.hip): caches of more than 16384 positions,
// and of at most that many.
constexpr uint32_t kSuffixDecodeMaxRows = 6;
constexpr uint32_t kSuffixDecodeMaxRowsShort = 12;
constexpr uint32_t kSuffixDecodeMaxT = 64;
uint32_t suffix_pack(const miikv_view* view, uint32_t q_heads, uint32_t token_count, bool device_count,
                     uint32_t max_cols = 16, bool ragged = false);
bool decode_columns_fit(uint32_t G, uint32_t D);  // decode_kernel serves G columns at head_dim D
// Workspace with which a suffix of at most `bound` keys runs as decodes; and the most that any
// context up to `bound` can use.
uint64_t suffix_by_decode_bytes(const miikv_view* view, uint32_t q_heads, uint32_t token_count, uint32_t bound);
uint64_t suffix_by_decode_bytes_up_to(const miikv_view* view, uint32_t q_heads, uint32_t token_count, uint32_t bound);
miikv_status suffix_by_decode(const miikv_view* view, const void* q, uint32_t q_dtype, uint32_t q_heads, float scale,
                              uint32_t token_count, uint32_t base_position, uint32_t seq,
                              const miikv_prefill_state* prefill_state, uint32_t bound, float* out, const float* gate,
                              float* gated_out, void* workspace, uint64_t workspace_bytes, void* stream);

// fp16 halves of one expanded step: K fragments [D/16][64 lanes][8], then
// V fragments [D/32][2 key halves][64 lanes][8].
__host__ __device__ constexpr uint32_t tile_halves(uint32_t D) { return 2 * D * kSufStep; }

struct ExpandArgs {
    Geo g;
    uint32_t seq;
    uint32_t key_count;  // host: P + T; with a device state: the capacity bound
    const miikv_prefill_state* ps;
    uint32_t steps;      // steps per kv head in the tile area
    _Float16* tiles;
    // Fused append (k_new set): the suffix's fp16 rows [token_count][kv_heads][D],
    // quantised and stored at positions base_position + t (or the prefill state's).
    const uint16_t* k_new;
    const uint16_t* v_new;
    uint32_t token_count;
    uint32_t base_position;
    // Incremental tiles: grid x covers steps step0 + (gridDim.x - 1 - blockIdx.x); with
    // `current` set the steps wholly below the base position (the prefill state's, on
    // the device) are already expanded in the tile area and are skipped.
    uint32_t step0;
    uint32_t current;
};

// Order of (kv head, split, row block) along an XCD's workgroups: the row blocks of one
// (kv head, split) next to each other; the splits of one row block next to each other; or,
// without splits, each kv head's row blocks with the most keys first (kSufLongFirst), in
// the 4-wave form the second half shortest first (kSufPaired).  With whole heads on each XCD
// (a multiple of 8 kv heads) the two workgroups that a CU then runs together have about the
// same keys in all; with other counts some XCDs hold more long row blocks than others.
enum SuffixOrder : uint32_t { kSufTilesTogether = 0, kSufRowsTogether = 1, kSufLongFirst = 2, kSufPaired = 3 };

struct SuffixArgs {
    Geo g;
    const void* q;
    uint32_t q_f32;
    uint32_t q_heads;
    uint32_t group;
    float scale_log2;
    uint32_t token_count;  // host upper bound
    uint32_t base_position;
    const miikv_prefill_state* ps;
    uint32_t split_keys;   // keys per split (multiple of kSufStep)
    uint32_t splits;
    uint32_t row_blocks;   // workgroups per (kv head, split) group
    uint32_t steps;        // steps per kv head in the tile area
    const _Float16* tiles;
    void* part;            // partial records when splits > 1
    float* out;
    const float* gate;
    float* gated_out;
    uint32_t order;        // suffix_kernel order of the work items (SuffixOrder)
};

// Partial records of split-K, laid out so that a wave's 32 rows write one
// contiguous block: O / l in fp16 [split][kv head][row][D] (row = t*G + g, rows
// counted up to the host token bound), then (m, l) fp32 pairs [split][kv head][row].
// The split's output is stored normalised (a convex combination of V rows, so
// fp16 holds it to the same relative precision as the fp16 V tiles it came from),
// which halves the record traffic of the split kernel and the combine.
struct SuffixCombineArgs {
    uint32_t kv_heads;
    uint32_t q_heads;
    uint32_t group;
    uint32_t token_count;  // host bound
    uint32_t base_position;
    const miikv_prefill_state* ps;
    uint32_t split_keys;
    uint32_t splits;
    const void* part;
    float* out;
    const float* gate;
    float* gated_out;
};

__host__ __device__ inline size_t part_o_halves(uint32_t splits, uint32_t kv_heads, uint32_t rows, uint32_t D) {
    return static_cast<size_t>(splits) * kv_heads * rows * D;
}
// Bytes of one row's record in one split: D fp16 values and an (m, l) pair.
__host__ __device__ constexpr uint32_t part_row_bytes(uint32_t D) { return 2 * D + 8; }

__device__ __forceinline__ float sfx_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

__device__ __forceinline__ float16v mfma_32x32x16(half8 a, half8 b, float16v c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
// Workgroup barrier after this wave's LDS reads have returned; copies stay in flight.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

}  // namespace miikv
