// Split-K partial records and their combine, shared by decode and suffix attention.
#pragma once

#include "miikv_common.hpp"

namespace miikv {
namespace {

#ifndef MIIKV_WPW
#define MIIKV_WPW 4
#endif
constexpr uint32_t kWavesPerWg = MIIKV_WPW;

struct SplitArgs {
    Geo g;
    const void* q;
    uint32_t q_heads;
    uint32_t group;  // columns per (row set, kv head), <= 16: pack tokens x query heads per kv head
    // Tokens per row set (1: decode).  A short suffix packs `pack` consecutive tokens of
    // one sequence into a row set: column c is token t = pack*b + c / (group / pack), query
    // head h * (group / pack) + c % (group / pack), with t's context (host lengths, the last
    // token's is max_context); the last row set's tokens past it are not stored.
    uint32_t pack;
    float scale_log2;
    // Context length of row-set b: (len_ptr ? len_ptr[b * len_stride] : 0) + len_add
    // + b * len_bstep (decode: per-sequence lengths; suffix: base + t + 1).
    const uint32_t* len_ptr;
    uint32_t len_stride;
    uint32_t len_add;
    uint32_t len_bstep;
    const uint32_t* count_ptr;  // if set, row-sets b >= *count_ptr are skipped
    uint32_t max_context;
    uint32_t cpw;         // chunks per wave
    uint32_t max_splits;  // splits per (sequence, kv head)
    uint32_t batch;       // sequences (row-sets)
    // batch > 1, streamed plan: workgroups of the split kernel over which the batch's
    // steps are cut evenly (StreamTotal); 0: every (sequence, kv head) is cut by itself
    // into splits of cpw steps per wave
    uint32_t stream_wgs;
    // [batch][kv_heads][max_splits + 1][record]: the splits, then with the fused append
    // the new token's record at slot nsplit.  Streamed plan: segment records (StreamSeq)
    // in the first batch * kv_heads * max_splits slots, then one slot per (sequence, kv
    // head) for the new token.
    float* part;
    float* out;
    const float* gate;
    float* gated_out;
    uint8_t* gated_q8_1;  // nullable: Q8_1 blocks [batch][q_heads][D/32] of gated_out
    const uint16_t* k_new;  // fused append: fp16 rows [batch][kv_heads][D] stored at position L-1
    const uint16_t* v_new;
    // fused append of fp32 rows instead (k_new / v_new then null), with the reference's
    // K prologue when k_norm_weight is set (RMSNorm * weight, RoPE on dims 0..63)
    const float* k_new32;
    const float* v_new32;
    const float* k_norm_weight;
    float rope_step;        // theta^(-2/64), from the host
    float epsilon;
    uint32_t q_f32;         // q dtype (scoring the appended token)
    uint32_t rowset_order;  // row sets of one sequence: XCD-ordered (kv head, split, row set) items
};


__device__ __forceinline__ float exp2_safe(float x) { return exp2f(x); }  // exp2(-inf) == 0

// Floats in one split's partial record: O [G*D], m [G], l [G], padded to 4.
__host__ __device__ __forceinline__ uint32_t record_floats(uint32_t G, uint32_t D) {
    return G * D + ((2 * G + 3) / 4) * 4;
}

__device__ __forceinline__ uint32_t split_length(const SplitArgs& a, uint32_t b) {
    uint32_t L = (a.len_ptr ? a.len_ptr[static_cast<size_t>(b) * a.len_stride] : 0u) + a.len_add + b * a.len_bstep;
    return L > a.max_context ? a.max_context : L;
}

// Streamed plan of a ragged batch.  The lengths are only known on the device, so every
// wave derives the plan from them, by itself and without a barrier (a lane per sequence,
// 64 sequences at a time).  In the order (sequence, kv head), every pair that holds keys
// takes kSegmentCost units plus one per 32-key step on one axis, which is cut into
// stream_wgs runs of `quota` units; workgroup w takes run w, which may cross from one pair
// into the next: every workgroup of the one resident round has the same work whatever the
// lengths are.  Each (workgroup, pair) with steps in common is a segment with a record of
// its own, number w + pair: both only grow along the axis and no two segments share both,
// so the numbers are distinct, and one pair's are consecutive.
// Bound: the cache stream (HBM), then a segment's fixed latency (lengths, query, first
// step, record), which kSegmentCost prices in steps.  Measured, fused append + attend, us,
// against splits of one size per sequence that fit one round: 48 sequences of 64..4096
// tokens, 32q/8kv/D128 (220 MB) 89.6 -> 48.3 (4.6 TB/s); 48 of 2080, 75.2 -> 47.3; 96 of
// 500..1000, 24q/4kv/D256 66.0 -> 48.4; config 3 (1.18 GB) 192.0 -> 190.9.  kSegmentCost
// 0 / 3 / 6 / 10 / 16 on the first: 58.9 / 50.8 / 48.3 / 49.1 / 49.7.
#ifndef MIIKV_SEGMENT_COST
#define MIIKV_SEGMENT_COST 6
#endif
constexpr uint32_t kSegmentCost = MIIKV_SEGMENT_COST;
struct StreamTotal {
    unsigned long long units;  // of one kv head, all sequences
    unsigned long long quota;  // units per workgroup
};

// Keys of sequence b that the splits cover (the fused append's new token has a record of
// its own), in 32-key steps.
__device__ __forceinline__ uint32_t stream_steps(const SplitArgs& a, uint32_t b, uint32_t appended) {
    const uint32_t L = split_length(a, b);
    return (L - min(L, appended) + kChunk - 1) / kChunk;
}
__device__ __forceinline__ uint32_t stream_units(uint32_t steps) { return steps + (steps != 0 ? kSegmentCost : 0u); }

__device__ __forceinline__ StreamTotal stream_total(const SplitArgs& a, uint32_t appended) {
    const uint32_t lane = threadIdx.x & 63;
    unsigned long long sum = 0;
    for (uint32_t b = lane; b < a.batch; b += 64) sum += stream_units(stream_steps(a, b, appended));
#pragma unroll
    for (uint32_t off = 1; off < 64; off <<= 1) sum += __shfl_xor(sum, off, 64);
    StreamTotal t;
    t.units = sum;
    // At least one step for each wave of a workgroup.  (Asking for a segment's cost on top
    // left half the round idle in small batches: us of splits per sequence / so / now, 3
    // sequences of 2048..4096 tokens, 32q/8kv/D128 16.6 / 17.6 / 15.9; 8 of 100..200,
    // 24q/4kv/D256 17.2 / 21.2 / 16.9.)
    const unsigned long long q = (sum * a.g.kv_heads + a.stream_wgs - 1) / a.stream_wgs;
    t.quota = q < kWavesPerWg ? kWavesPerWg : q;
    return t;
}

// This lane's sequence b0 + lane: its steps, and the units of one kv head before it given
// those before b0.
struct StreamSeq {
    uint32_t steps;
    unsigned long long before;
};
__device__ __forceinline__ StreamSeq stream_chunk(const SplitArgs& a, uint32_t b0, unsigned long long base,
                                                  uint32_t appended) {
    const uint32_t lane = threadIdx.x & 63;
    StreamSeq s;
    s.steps = b0 + lane < a.batch ? stream_steps(a, b0 + lane, appended) : 0u;
    unsigned long long incl = stream_units(s.steps);
#pragma unroll
    for (uint32_t off = 1; off < 64; off <<= 1) {
        const unsigned long long up = __shfl_up(incl, off, 64);
        if (lane >= off) incl += up;
    }
    s.before = base + incl - stream_units(s.steps);
    return s;
}

// Records of (sequence b, kv head h): `first` and `count` (the new token's record not
// counted).  b and h may differ between the lanes of a wave; every lane takes part.
__device__ __forceinline__ void stream_records(const SplitArgs& a, uint32_t b, uint32_t h, uint32_t appended,
                                               uint32_t& first, uint32_t& count) {
    const StreamTotal t = stream_total(a, appended);
    unsigned long long base = 0, before = 0;
    uint32_t steps = 0;
    for (uint32_t b0 = 0; b0 < a.batch; b0 += 64) {
        const StreamSeq s = stream_chunk(a, b0, base, appended);
        const unsigned long long bf = __shfl(s.before, b & 63, 64);
        const uint32_t st = __shfl(s.steps, b & 63, 64);
        if (b - b0 < 64) {
            before = bf;
            steps = st;
        }
        base = __shfl(s.before, 63, 64) + stream_units(__shfl(s.steps, 63, 64));
    }
    first = count = 0;
    if (steps == 0) return;
    // the pair's steps follow its kSegmentCost units
    const unsigned long long start = before * a.g.kv_heads + static_cast<unsigned long long>(h) * stream_units(steps) + kSegmentCost;
    const uint32_t w0 = static_cast<uint32_t>(start / t.quota);
    const uint32_t w1 = static_cast<uint32_t>((start + steps - 1) / t.quota);
    first = w0 + b * a.g.kv_heads + h;
    count = w1 - w0 + 1;
}

// Context of token tp of row set b of a packed suffix (past the suffix: above max_context).
__device__ __forceinline__ uint32_t packed_context(const SplitArgs& a, uint32_t b, uint32_t tp) {
    return a.len_add + b * a.len_bstep - (a.pack - 1 - tp);
}

// Split count of sequence b at `cpw` steps per wave (0 when L == 0).
__device__ __forceinline__ uint32_t split_count(uint32_t L, uint32_t cpw) {
    const uint32_t tps = kWavesPerWg * cpw * kChunk;
    return (L + tps - 1) / tps;
}

// Cross-split combine.  Workgroup (sequence * kv_heads + head, block of 32
// consecutive output elements, all in one query-head row) holds one record slot per
// thread group: thread (q = tid & 7, rg = tid >> 3) reads elements 4q..4q+3 of records
// rg, rg + 32, rg + 64 (issued before the context length arrives, so one memory round
// trip covers a single sequence's 64 splits and the fused append's record) and of any
// further ones after it, folding them with its own running max.  The 32 record groups
// are then merged in a fixed butterfly (lanes 8, 16, 32 apart) and across the four
// waves in LDS, so the result is deterministic.
// Fused append (APPEND): the splits covered the L-1 cached keys and decode_kernel
// wrote the new token's record (m = score, l = 1, O = its dequantised V row) at
// slot nsplit, merged here as one more record.  The merge follows the reference
// combine (gfx906/kernels/qwen3_primitives.hip:2295-2385).
__device__ __forceinline__ void merge_state(float& m, float& l, float4& acc, float m2, float l2, float4 a2) {
    if (m2 == -INFINITY) return;
    if (m == -INFINITY) {
        m = m2; l = l2; acc = a2;
        return;
    }
    const float mn = fmaxf(m, m2);
    const float f1 = exp2_safe(m - mn), f2 = exp2_safe(m2 - mn);
    m = mn;
    l = l * f1 + l2 * f2;
    acc.x = acc.x * f1 + a2.x * f2;
    acc.y = acc.y * f1 + a2.y * f2;
    acc.z = acc.z * f1 + a2.z * f2;
    acc.w = acc.w * f1 + a2.w * f2;
}

// Records of one (sequence b, kv head h), and how many may be read before the count is
// known.  STREAM: the segments' records, then the new token's; otherwise all of the pair's
// slots.  (Two instances: choosing at run time cost one sequence's decode 0.1 us.)
template <bool STREAM>
struct CombineRecords {
    const float* part;      // the first record
    const float* appended;  // STREAM: the new token's record
    uint32_t nseg;          // STREAM: segments
    uint32_t slots;
    __device__ __forceinline__ const float* at(uint32_t j, uint32_t rec) const {
        if constexpr (STREAM) return j < nseg ? part + static_cast<size_t>(j) * rec : appended;
        else return part + static_cast<size_t>(j) * rec;
    }
};
template <bool STREAM>
__device__ __forceinline__ CombineRecords<STREAM> combine_records(const SplitArgs& a, uint32_t b, uint32_t h, uint32_t bh,
                                                                  uint32_t rec, bool append) {
    CombineRecords<STREAM> r;
    if constexpr (STREAM) {
        uint32_t first;
        stream_records(a, b, h, append ? 1u : 0u, first, r.nseg);
        r.part = a.part + static_cast<size_t>(first) * rec;
        r.appended = a.part + (static_cast<size_t>(a.batch) * a.g.kv_heads * a.max_splits + bh) * rec;
        r.slots = r.nseg + (append && split_length(a, b) > 0 ? 1u : 0u);
    } else {
        r.slots = a.max_splits + 1;
        r.part = a.part + (static_cast<size_t>(bh) * r.slots) * rec;
    }
    return r;
}
// Records of sequence b (the plan of fixed splits waits for its length here).
template <bool STREAM>
__device__ __forceinline__ uint32_t combine_count(const SplitArgs& a, uint32_t b, const CombineRecords<STREAM>& r, bool append) {
    if constexpr (STREAM) return r.slots;
    const uint32_t L = split_length(a, b);
    return split_count(L, a.cpw) + (append && L > 0 ? 1u : 0u);
}

// Gate values of elements i..i+3.  Called after the record loads are issued: a load
// in a branch is waited for at the branch's end, which would otherwise hold back the
// loads issued after it (here everything it waits for is needed next).
__device__ __forceinline__ void combine_gate(const SplitArgs& a, size_t i, float (&gv)[4]) {
    gv[0] = gv[1] = gv[2] = gv[3] = 0.0f;
    if (a.gate != nullptr) {
        const float4 g4 = *reinterpret_cast<const float4*>(a.gate + i);
        gv[0] = g4.x; gv[1] = g4.y; gv[2] = g4.z; gv[3] = g4.w;
    }
}

// Output of 4 merged elements e..e+3 (thread q of the 8 holding a 32-value block that
// starts at element blk0 of the launch's rows): out = acc / L, 0 when L == 0
// (qwen3_primitives.hip:2349); gated = out * sigmoid(gate); the Q8_1 block.  All 8
// threads of a block call it (the block's reductions); `live` = false computes but
// stores nothing.
__device__ __forceinline__ void combine_emit(const SplitArgs& a, size_t out_row0, uint32_t e, uint32_t q, size_t blk0,
                                             float l, float4 acc, const float (&gv)[4], bool live) {
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    const float vals[4] = {acc.x * inv, acc.y * inv, acc.z * inv, acc.w * inv};
    float gated[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (a.out && live) *reinterpret_cast<float4*>(a.out + out_row0 + e) = make_float4(vals[0], vals[1], vals[2], vals[3]);
    if (a.gate) {
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) gated[k] = vals[k] * (1.0f / (1.0f + expf(-gv[k])));
        if (a.gated_out && live)
            *reinterpret_cast<float4*>(a.gated_out + out_row0 + e) = make_float4(gated[0], gated[1], gated[2], gated[3]);
    }
    if (a.gate && a.gated_q8_1) {
        // Q8_1 block of these 32 gated values (qwen3_primitives.hip:2354-2384):
        // d = amax/127, q = clamp(roundf(x/d), -127, 127), s = sum(q)*d.
        float amax = fmaxf(fmaxf(fabsf(gated[0]), fabsf(gated[1])), fmaxf(fabsf(gated[2]), fabsf(gated[3])));
        amax = group_reduce<8>(amax, MaxOp{});
        const float d = amax / 127.0f;
        const float qinv = d != 0.0f ? 1.0f / d : 0.0f;
        int qs[4];
        int sum = 0;
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            qs[k] = max(-127, min(127, static_cast<int>(roundf(gated[k] * qinv))));
            sum += qs[k];
        }
        sum = group_reduce<8>(sum, AddOp{});
        if (!live) return;
        const size_t blk = (out_row0 + blk0) / 32;
        uint8_t* bp = a.gated_q8_1 + blk * 36;
        *reinterpret_cast<uint32_t*>(bp + 4 + 4 * q) =
            (static_cast<uint32_t>(qs[0]) & 0xffu) | ((static_cast<uint32_t>(qs[1]) & 0xffu) << 8) |
            ((static_cast<uint32_t>(qs[2]) & 0xffu) << 16) | ((static_cast<uint32_t>(qs[3]) & 0xffu) << 24);
        if (q == 0) {
            *reinterpret_cast<uint16_t*>(bp) = f32_to_f16_bits(d);
            *reinterpret_cast<uint16_t*>(bp + 2) = f32_to_f16_bits(static_cast<float>(sum) * d);
        }
    }
}


template <uint32_t D, bool APPEND, bool STREAM>
__global__ void __launch_bounds__(256) combine_kernel(SplitArgs a) {
    const uint32_t bh = blockIdx.x;
    const uint32_t b = bh / a.g.kv_heads;
    const uint32_t h = bh % a.g.kv_heads;
    const uint32_t G = a.group;
    const uint32_t GD = G * D;
    const uint32_t tid = threadIdx.x;
    const uint32_t q = tid & 7, rg = tid >> 3;
    const uint32_t e = blockIdx.y * 32 + 4 * q;  // < GD: the grid covers GD / 32 blocks
    const uint32_t hn = (blockIdx.y * 32) / D;
    // output row of column hn (packed tokens: token pack*b + hn / Gt, head h*Gt + hn % Gt),
    // indexed below with the column's offset e - hn * D folded back in
    const uint32_t Gt = G / a.pack, tp = hn / Gt;
    if (a.pack > 1 && packed_context(a, b, tp) > a.max_context) return;  // past the suffix (workgroup-uniform)
    const size_t out_row0 = ((static_cast<size_t>(b) * a.pack + tp) * a.q_heads + static_cast<size_t>(h) * Gt +
                             (hn - tp * Gt)) * D - static_cast<size_t>(hn) * D;
    const uint32_t rec = record_floats(G, D);
    const CombineRecords<STREAM> R = combine_records<STREAM>(a, b, h, bh, rec, APPEND);
    const uint32_t slots = R.slots;

    constexpr uint32_t kSpec = 3;
    float ms[kSpec], ls[kSpec];
    float4 vv[kSpec];
#pragma unroll
    for (uint32_t j = 0; j < kSpec; ++j) {
        const uint32_t sp = rg + 32 * j;
        ms[j] = -INFINITY;
        ls[j] = 0.0f;
        vv[j] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (sp < slots) {
            const float* r = R.at(sp, rec);
            ms[j] = r[GD + hn];
            ls[j] = r[GD + G + hn];
            vv[j] = *reinterpret_cast<const float4*>(r + e);
        }
    }
    float gv[4];
    combine_gate(a, out_row0 + e, gv);
    if (a.count_ptr != nullptr && b >= *a.count_ptr) return;
    const uint32_t nrec = combine_count(a, b, R, APPEND);

    float m = -INFINITY, l = 0.0f;
    float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
    for (uint32_t j = 0; j < kSpec; ++j)
        if (rg + 32 * j < nrec) merge_state(m, l, acc, ms[j], ls[j], vv[j]);
    for (uint32_t sp = rg + 32 * kSpec; sp < nrec; sp += 32) {
        const float* r = R.at(sp, rec);
        merge_state(m, l, acc, r[GD + hn], r[GD + G + hn], *reinterpret_cast<const float4*>(r + e));
    }
    // Butterfly over the 8 record groups of this wave (lanes 8, 16, 32 apart).
#pragma unroll
    for (uint32_t off = 8; off < 64; off <<= 1) {
        const float m2 = __shfl_xor(m, off), l2 = __shfl_xor(l, off);
        float4 a2;
        a2.x = __shfl_xor(acc.x, off);
        a2.y = __shfl_xor(acc.y, off);
        a2.z = __shfl_xor(acc.z, off);
        a2.w = __shfl_xor(acc.w, off);
        merge_state(m, l, acc, m2, l2, a2);
    }
    __shared__ float4 s_acc[4][8];
    __shared__ float s_m[4][8], s_l[4][8];
    const uint32_t wave = tid >> 6;
    if ((tid & 63) < 8) {
        s_acc[wave][q] = acc;
        s_m[wave][q] = m;
        s_l[wave][q] = l;
    }
    __syncthreads();
    if (tid >= 8) return;
#pragma unroll
    for (uint32_t w = 1; w < 4; ++w) merge_state(m, l, acc, s_m[w][q], s_l[w][q], s_acc[w][q]);
    combine_emit(a, out_row0, e, q, blockIdx.y * 32, l, acc, gv, true);
}


// Cross-split combine for launches with few records per row set or many row sets:
// one thread per 4 consecutive outputs of one (row set, kv head) folds all of that row
// set's records itself, kNarrowRecords loads in flight at a time, so the grid is one
// thread per 4 outputs instead of a 256-thread workgroup per 32; 8 consecutive threads
// hold one 32-value block (Q8_1 epilogue).
constexpr uint32_t kNarrowRecords = 8;
template <uint32_t D, bool APPEND, bool STREAM>
__global__ void __launch_bounds__(256) combine_narrow_kernel(SplitArgs a) {
    const uint32_t G = a.group;
    const uint32_t GD = G * D;
    const uint64_t idx = static_cast<uint64_t>(blockIdx.x) * 256 + threadIdx.x;
    const uint64_t per = GD / 4;
    const uint32_t bh = static_cast<uint32_t>(idx / per);
    const bool row_live = bh < a.batch * a.g.kv_heads;
    const uint32_t bhc = row_live ? bh : 0;
    const uint32_t b = bhc / a.g.kv_heads;
    const uint32_t h = bhc % a.g.kv_heads;
    const uint32_t e = static_cast<uint32_t>(idx % per) * 4;
    const uint32_t q = (e / 4) & 7;
    const uint32_t hn = e / D;
    const uint32_t Gt = G / a.pack, tp = hn / Gt;
    const bool past = a.pack > 1 && packed_context(a, b, tp) > a.max_context;  // past the suffix: not stored
    const bool live = row_live && !past;
    const size_t out_row0 = ((static_cast<size_t>(b) * a.pack + (past ? 0u : tp)) * a.q_heads +
                             static_cast<size_t>(h) * Gt + (hn - tp * Gt)) * D - static_cast<size_t>(hn) * D;
    const uint32_t rec = record_floats(G, D);
    const CombineRecords<STREAM> R = combine_records<STREAM>(a, b, h, bhc, rec, APPEND);
    // The first batch of record slots is read before the context length arrives (slots
    // past the row set's count hold stale bytes and are dropped below; a streamed plan
    // has its count already), then the gate.
    const uint32_t slots = R.slots;
    float ms[kNarrowRecords], ls[kNarrowRecords];
    float4 vv[kNarrowRecords];
#pragma unroll
    for (uint32_t j = 0; j < kNarrowRecords; ++j) {
        if (j < slots) {
            const float* r = R.at(j, rec);
            ms[j] = r[GD + hn];
            ls[j] = r[GD + G + hn];
            vv[j] = *reinterpret_cast<const float4*>(r + e);
        }
    }
    float gv[4];
    combine_gate(a, out_row0 + e, gv);
    // a whole 32-value block shares b (GD is a multiple of 32), so the 8 threads of a
    // block take the same exit
    if (a.count_ptr != nullptr && b >= *a.count_ptr) return;
    const uint32_t nrec = combine_count(a, b, R, APPEND);
    float m = -INFINITY, l = 0.0f;
    float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
    for (uint32_t j = 0; j < kNarrowRecords; ++j)
        if (j < nrec) merge_state(m, l, acc, ms[j], ls[j], vv[j]);
    for (uint32_t sp0 = kNarrowRecords; sp0 < nrec; sp0 += kNarrowRecords) {  // further batches
#pragma unroll
        for (uint32_t j = 0; j < kNarrowRecords; ++j) {
            ms[j] = -INFINITY;
            if (sp0 + j < nrec) {
                const float* r = R.at(sp0 + j, rec);
                ms[j] = r[GD + hn];
                ls[j] = r[GD + G + hn];
                vv[j] = *reinterpret_cast<const float4*>(r + e);
            }
        }
#pragma unroll
        for (uint32_t j = 0; j < kNarrowRecords; ++j)
            if (sp0 + j < nrec) merge_state(m, l, acc, ms[j], ls[j], vv[j]);
    }
    combine_emit(a, out_row0, e, q, e - 4 * q, l, acc, gv, live);
}

}  // namespace
}  // namespace miikv
