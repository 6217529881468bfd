// attn_walk.h — which chunks of a sequence the decode attention walks and over how many slots it splits them: a function of the
// position on the device, known to the attention (layer_kernels.hip) and to the product that reads its slots (gemv_kernels.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define OXB_ATTN_PART_PAD 4  // floats after the hd outputs of a slot: maximum, sum, 2 unused (16-byte rows)

// Slots in use for a walk of n_walk chunks.  A second slot saves a chunk's time and costs a merge, and the two are about
// equal (one fp16 sequence at 200, 128-position chunks: 7.6 us with one slot, 8.2 with two; six: 8.6 and 9.7): two
// chunks stay with one workgroup, also where eight waves make them 256 positions each (INT8 at 350: one sequence
// 9.5 and 9.7, four 10.2 and 10.5; FP8, eight at 500: 10.6 and 11.3).
__device__ __forceinline__ uint32_t oxb_attn_slots_used(uint32_t n_walk, uint32_t n_splits) {
    return n_walk <= 2 ? 1u : n_walk < n_splits ? n_walk : n_splits;
}

// The keys that position `pos` sees are [0, sink_n) and [lo, pos].  The chunks of `ch` positions that hold one of them, in
// ascending order: `skip_at` chunks, then a gap of `gap`, then up to the new position's; n_walk in all.
struct OxbAttnWalk {
    uint32_t lo, sink_n, skip_at, gap, n_walk;
};
__device__ __forceinline__ OxbAttnWalk oxb_attn_walk(uint32_t pos, uint32_t window, uint32_t sinks, uint32_t ch) {
    OxbAttnWalk w;
    const uint32_t seq_len = pos + 1, budget = window > sinks ? window - sinks : 0u;
    w.lo = window ? (seq_len > budget ? seq_len - budget : 0u) : 0u;
    w.sink_n = window ? (sinks < seq_len ? sinks : seq_len) : 0u;
    const uint32_t lo_chunk = (w.lo < pos ? w.lo : pos) / ch, sink_chunks = (w.sink_n + ch - 1) / ch;
    w.skip_at = sink_chunks < lo_chunk ? sink_chunks : lo_chunk;
    w.gap = lo_chunk - w.skip_at;
    w.n_walk = (seq_len + ch - 1) / ch - w.gap;
    return w;
}

// What the reader of one sequence's slots needs: the attention leaves 2 .. `most` slots as they are (`most` 0: none) and
// merges others itself.  part: [q head][n_splits][hd + OXB_ATTN_PART_PAD], hd = 1 << hd_shift.
struct OxbAttnSlots {
    const float* part;
    const uint32_t* pos;
    uint32_t hd_shift, n_splits, chunk, window, sinks, most;
};
