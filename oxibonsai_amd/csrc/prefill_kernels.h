// prefill_kernels.h — launch interface of the prefill attention (see prefill_kernels.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stdint.h>

#include "kv_quant_device.h"
#include "operand_device.h"

struct OxbPrefillAttnParams {
    const float* qkv;                 // [M][qkv_stride]: the raw projections, q heads first (QK-norm and RoPE happen in the kernel)
    uint32_t qkv_stride;
    const float* q_norm;              // [hd]
    const float *cos_t, *sin_t;       // [max_seq][hd/2]
    float eps;
    const float* k_norm;              // null: the new rows are in the cache; else (oxb_attn_prefill_can_store) the launch stores them
    const void *k_cache, *v_cache;    // cache rows of hd values each (fp16 or one-byte codes), placed by `kv`
    const float *k_scale, *v_scale;   // quantised cache: one scale per row
    uint32_t kv_mode;                 // OXB_KV_* (kv_quant_device.h)
    OxbKvLayout kv;
    uint32_t seq, layer;              // whose rows the queries attend to
    uint32_t window, sinks;           // sliding window with attention sinks; window 0 = off
    float* out;                       // [M][nq * hd]
    OxbOperandOut op;                 // optional: the outputs as the packed activations of the O projection's GEMM instead
    uint32_t M, pos_start;            // query t sits at position pos_start + t and sees keys 0 .. pos_start + t
    uint32_t nq, nkv, hd, max_seq;
    float scale;                      // 1 / sqrt(hd)
    float* part;                      // oxb_attn_prefill_part_bytes(...) of scratch where that is not 0: sums of the runs of keys
    uint32_t blocks_per_split;        // key blocks of a run (filled by the launcher)
};

// How the launcher cuts the work: q heads per workgroup, query tiles per wave, workgroups, runs of keys.
struct OxbPrefillAttnPlan { uint32_t hpw, qt, wgs, n_splits, blocks_per_split; };
#define OXB_PF_ATTN_MAX_SPLITS 32u

// Whether the launch can work out and store the new positions' K and V itself.
bool oxb_attn_prefill_can_store(uint32_t hd, uint32_t pos_start, uint32_t M);
size_t oxb_attn_prefill_part_bytes(const OxbPrefillAttnParams& p, uint32_t n_cus);
hipError_t oxb_launch_attn_prefill(OxbPrefillAttnParams p, uint32_t n_cus, hipStream_t st);
