// layer_kernels.hip — the Qwen3 layer glue between the quantised GEMVs, for gfx950.
//
// Reference sequence (one decode token, crates/oxibonsai-kernels/src/gpu_backend/
// cuda_full_layer/encode_ternary.rs:142-290, CPU twin crates/oxibonsai-model/src/block/types/forward.rs:92-408):
//   RMSNorm -> QKV GEMV -> per-head QK-RMSNorm + half-split RoPE -> FP16 KV store ->
//   attention over seq_len -> O GEMV + residual -> RMSNorm -> gate||up GEMV -> SiLU(g)*u -> down GEMV + residual.
// RMSNorm, the residual adds and SwiGLU live in the GEMV kernel's prologue and epilogues (gemv_kernels.hip); here
// are the attention kernels, the merge of their slots, the KV row quantiser and the greedy selection.
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stdint.h>

#include <type_traits>

#include "device_utils.h"
#include "kv_quant_device.h"
#include "kv_row_device.h"
#include "layer_kernels.h"
#include "gemv_pack_device.h"

// ---------------------------------------------------------------------------
// The new K and V rows of a prefill: K per-head RMSNorm + half-split RoPE, V as it is, to the cache rows of positions
// pos_base + t (fp16 round-to-nearest-even, or quantised: kv_quant_device.h).
// (fused_qk_norm_rope + fused_kv_store, gpu_backend/cuda_attn_kernels.rs:160-251;
//  CPU: block/types/forward.rs:179-213, rope pairs (d, d + hd/2) simd_float_ops.rs:240-253; the attention kernel norms and
//  rotates Q itself.)
// hd / 4 lanes hold a head's row, four values each, so that a wave takes 256 / hd heads of a token side by side; everything it
// needs is requested at once.  What bounds it is that one round trip to memory (few tokens) and the way there and back
// (2048 tokens x 8 heads: 25 MB).  Two heads a wave one after the other, a value per lane and request, took 5.0 us for 23 tokens,
// 6.9 for 301 with INT8 rows and 9.0 to 10 for 2048; this form 2.8, 5.0 and 5.7 (kernel traces).
// ---------------------------------------------------------------------------
template <int HD, int KVM>
__global__ __launch_bounds__(256) void kv_norm_rope_store_kernel(OxbKvStoreParams p) {
    constexpr int L = HD / 4, HPW = 64 / L;  // lanes of a head, heads of a wave
    const uint32_t lane = threadIdx.x & 63u, j = lane % L;
    const uint32_t n_hg = (p.nkv + HPW - 1) / HPW, id = blockIdx.x * 4 + (threadIdx.x >> 6);  // (token, group of heads)
    const uint32_t t = id / n_hg, head = (id % n_hg) * HPW + lane / L;
    if (t >= p.M || head >= p.nkv) return;  // (whole groups of lanes)
    const uint32_t pos = p.pos_base + t;
    const KvRowIn in = kv_row_load<HD>(p.qkv + (size_t)t * p.qkv_stride, p.nq, p.nkv, head, j, p.cos_t, p.sin_t, pos);
    const float4 w = *reinterpret_cast<const float4*>(p.k_norm + 4 * j);
    kv_row_store<HD, KVM>(kv_row_make<HD, KVM>(in, w, p.eps, j), p.k_cache, p.v_cache, p.k_scale, p.v_scale, kv_row(p.kv, p.seq, p.layer, head, pos), j);
}

// Rows of f32 values -> quantised cache rows (codes + scale), one wave per row; the arithmetic of the attention
// kernels' own stores, exposed for callers that fill a cache themselves and for tests.
template <int KVM>
__global__ __launch_bounds__(64) void kv_quantize_rows_kernel(const float* __restrict__ x, uint32_t n, uint8_t* __restrict__ codes,
                                                               float* __restrict__ scales) {
    const float* row = x + (size_t)blockIdx.x * n;
    float mx = 0.f;
    for (uint32_t d = threadIdx.x; d < n; d += 64) mx = fmaxf(mx, fabsf(row[d]));
    mx = wave_max_f32(mx);
    const float scale = kv_row_scale<KVM>(mx);
    for (uint32_t d = threadIdx.x; d < n; d += 64) codes[(size_t)blockIdx.x * n + d] = (uint8_t)kv_encode<KVM>(row[d], scale);
    if (threadIdx.x == 0) scales[blockIdx.x] = scale;
}

// Quantised rows back to f32 as attention reads them, code * scale (dequantize_row, kv_cache_quant.rs:69-71, 545-556):
// the codes are widened four at a time by the routine the attention kernels use (kv_dec4), which is what this is for.
template <int KVM>
__global__ __launch_bounds__(256) void kv_dequantize_rows_kernel(const uint32_t* __restrict__ codes4, const float* __restrict__ scales,
                                                                 uint32_t n, uint64_t total4, float* __restrict__ out) {
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;  // one dword of four codes; n % 4 == 0
    if (i >= total4) return;
    uint32_t lo, hi;
    kv_dec4<KVM>(codes4[i], lo, hi);
    const kvh2_t a = __builtin_bit_cast(kvh2_t, lo), b = __builtin_bit_cast(kvh2_t, hi);
    const float sc = scales[(i * 4) / n];
    out[i * 4 + 0] = (float)a[0] * sc;
    out[i * 4 + 1] = (float)a[1] * sc;
    out[i * 4 + 2] = (float)b[0] * sc;
    out[i * 4 + 3] = (float)b[1] * sc;
}

hipError_t oxb_launch_kv_dequantize_rows(int kv_mode, const uint8_t* d_codes, const float* d_scales, uint32_t n_rows, uint32_t n,
                                         float* d_out, hipStream_t st) {
    if (n_rows == 0 || n == 0 || (n & 3u)) return hipErrorInvalidValue;
    const uint64_t total4 = (uint64_t)n_rows * n / 4;
    const dim3 grid((uint32_t)((total4 + 255) / 256));
    if (kv_mode == OXB_KV_I8)
        hipLaunchKernelGGL(kv_dequantize_rows_kernel<OXB_KV_I8>, grid, dim3(256), 0, st, (const uint32_t*)d_codes, d_scales, n, total4, d_out);
    else if (kv_mode == OXB_KV_FP8_E4M3)
        hipLaunchKernelGGL(kv_dequantize_rows_kernel<OXB_KV_FP8_E4M3>, grid, dim3(256), 0, st, (const uint32_t*)d_codes, d_scales, n, total4, d_out);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t oxb_launch_kv_quantize_rows(int kv_mode, const float* d_x, uint32_t n_rows, uint32_t n, uint8_t* d_codes, float* d_scales,
                                       hipStream_t st) {
    if (n_rows == 0 || n == 0) return hipErrorInvalidValue;
    if (kv_mode == OXB_KV_I8) hipLaunchKernelGGL(kv_quantize_rows_kernel<OXB_KV_I8>, dim3(n_rows), dim3(64), 0, st, d_x, n, d_codes, d_scales);
    else if (kv_mode == OXB_KV_FP8_E4M3)
        hipLaunchKernelGGL(kv_quantize_rows_kernel<OXB_KV_FP8_E4M3>, dim3(n_rows), dim3(64), 0, st, d_x, n, d_codes, d_scales);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Decode attention, split over the KV sequence (flash-decode), on the matrix cores: softmax(q K^T / sqrt(hd)) V
// with GQA (kv_head = q_head / (nq / nkv)) over positions 0..pos[b]
// (batched_attn_scores_v2 / batched_softmax / batched_attn_weighted_sum, cuda_attn_kernels.rs:264-438;
//  CPU: block/functions.rs:78-127 -> layers/attention_fused.rs:329-400), fused with what precedes it in the layer:
// per-head QK-RMSNorm, RoPE and the FP16 store of the new position's K and V (fused_qk_norm_rope + fused_kv_store,
// cuda_attn_kernels.rs:160-251).  Grid (n_splits, nkv, batch), NW = 4 or 8 waves.  It writes, per q head and
// slot, the un-normalised partial output, the running maximum and the running sum; the last workgroup of a
// (sequence, kv head) to finish merges the slots (attn_last_arrival, attn_merge_heads).
// A workgroup serves all q heads of one kv head (<= 16, the columns of the MFMA tiles) for one slot of the KV
// sequence: slot s walks chunks s, s + n_splits, ... of 32 NW positions, wave w takes keys [32w, 32w + 32) of each.
//   S^T[key][head] = sum_d K[key][d] Q[head][d]     A = K rows straight from the cache, B = Q * scale as fp16 hi + lo
//   O^T[d][head]  += sum_key V[key][d] P[head][key]  A = V gathered from the wave's LDS copy of the block,
//                                                    B = the lane's own probabilities as fp16 hi + lo
// so scores and weighted sums keep fp32-level accuracy.  Every wave runs its own online softmax; the results
// meet in LDS.  The workgroup whose slot holds the new position computes K (norm + RoPE) and V of that position, stores
// them to the cache and leaves a copy in LDS, as stored, which takes the row's place in the chunk that holds it: nothing waits
// for the stores.
// ---------------------------------------------------------------------------
typedef _Float16 v8h_t __attribute__((ext_vector_type(8)));

// Options of the kernel (template KVM, fields window / sinks):
//  * quantised cache rows (kv_quant_device.h): one byte per value plus an f32 scale per row.  The codes enter the
//    matrix cores as exact fp16 numbers; the K row scale multiplies the score, the V row scale the probability
//    (relative to a running largest scale `u`, so that the fp16 hi + lo pair of the product stays in range; the
//    accumulator is kept in units of u and rescaled like the running maximum of the softmax).  A lane takes a
//    contiguous quarter of a K row (hd / 4 bytes), so the Q operand follows that order.
//    Eight waves widen the codes of one CU's walk twice as fast as four, but cost 1 us more to start, to meet and to
//    merge; fp16 rows, which need no widening, are limited by the requests in flight either way: four waves, except for
//    long walks of quantised rows (model.hip: attn_wide).  8B shape, us per launch with 4 / 8 waves: one FP8 sequence at
//    32 000 28.2 / 22.4, at 8 000 13.5 / 14.0; 32 of INT8 at 2048 35.8 / 33.0, at 500 13.0 / 13.3; one of fp16 at 700
//    8.7 / 10.8, at 20 000 21.0 / 22.5.
//  * sliding window with attention sinks (is_in_window, crates/oxibonsai-model/src/layers/sliding_window.rs:173-189):
//    the first `sinks` keys stay visible, the others while pos - key < window - sinks; chunks without a visible key
//    are not walked.  window == 0: every key up to pos is visible.
// The outputs as fp32 (p.out), as those and superblocks of the O projection's packed GEMV (p.pack_out), or as its GEMM's operand (p.op).
enum { OXB_ATTN_OUT_F32 = 0, OXB_ATTN_OUT_PACK = 1, OXB_ATTN_OUT_XH = 2 };
#define OXB_ATTN_MERGE_LDS_BYTES(heads, threads) ((heads) * 65 * 4 + 12 + (threads) * 16)  // LDS attn_merge_heads needs
template <uint32_t NT, int OUT>
__device__ __forceinline__ void attn_merge_heads(const OxbAttnParams& p, uint32_t b, uint32_t h_first, uint32_t nh, uint32_t used, float* sm);
__device__ __forceinline__ void attn_pack_outputs(const OxbAttnParams& p, uint32_t b, uint32_t h_first, const float* kf);

// The workgroups of one (sequence, kv head) count themselves off once their slot results are written; the last one
// to arrive merges the slots of the group's heads into the attention output, so that no second launch is needed.
// The counter returns to 0 for the next launch.  The slot results travel between workgroups (other CUs, other XCDs)
// through agent-coherent stores and loads: every store of this workgroup has been acknowledged by memory before its
// count is added, and the merge's loads bypass the caches that another workgroup's stores do not reach.
__device__ __forceinline__ bool attn_last_arrival(const OxbAttnParams& p, uint32_t b, uint32_t kvh, uint32_t expected, uint32_t* flag) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t* ctr = p.done + (size_t)b * p.nkv + kvh;
        const uint32_t prev = atomicAdd(ctr, 1u);
        const uint32_t last = prev + 1u == expected ? 1u : 0u;
        if (last) atomicExch(ctr, 0u);
        *flag = last;
    }
    __syncthreads();
    return *flag != 0u;
}

// NW: waves; OPT: a window and / or a paged cache may be in use (else neither costs anything); OUT: what the outputs leave as.
// (With tests of the fields instead 23 scalar registers are spilled: one fp16 sequence at 700 8.7 us against 8.4.)
template <int HD, int KVM, uint32_t NW, bool OPT, int OUT>
__global__ __launch_bounds__(64 * NW) void attn_decode_fused_kernel(OxbAttnParams p) {
    constexpr uint32_t NT = 64 * NW, CH = 32 * NW;  // threads, KV positions of a chunk
    constexpr bool QC = KVM != OXB_KV_F16;
    constexpr int KS = HD / 32, NS = HD / 16, VSTR = HD + 8;
    constexpr int VPR = QC ? HD / 16 : HD / 8;  // 16-byte pieces per V row
    constexpr int VL = 32 * VPR / 64;           // pieces of the wave's 32-row V block per lane
    // V block per wave; after the loop the merge buffers.  Q * scale of the group's heads has an area of its own, so
    // that a wave whose Q operands are in registers starts staging V without waiting for the others.
    __shared__ __attribute__((aligned(16))) _Float16 vs_all[NW][32 * VSTR];
    __shared__ __attribute__((aligned(16))) _Float16 qs[2][16 * HD];  // fp16 hi and lo parts, as the B operands take them
    __shared__ uint32_t last_flag;
    typedef typename std::conditional<QC, uint8_t, _Float16>::type cache_t;
    __shared__ __attribute__((aligned(16))) cache_t kv_new[2][HD];  // the new position's K and V rows as stored
    __shared__ float kv_new_scale[2];
    static_assert(sizeof(vs_all) >= OXB_ATTN_MERGE_LDS_BYTES(16, NT), "the merge's slot weights and partial sums must fit in the V slices");
    const uint32_t tid = threadIdx.x, lane = tid & 63u, qi = lane & 15u, g = lane >> 4;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t slot = blockIdx.x, kvh = blockIdx.y, b = blockIdx.z;
    const uint32_t G = p.nq / p.nkv, h0 = kvh * G, half = HD / 2;
    const uint32_t pos = p.pos[b], seq_len = pos + 1;
    // visible keys: [0, sink_n) and [lo, seq_len); the chunks that hold one
    const OxbAttnWalk walk = oxb_attn_walk(pos, OPT ? p.window : 0u, p.sinks, CH);
    const uint32_t lo = walk.lo, sink_n = walk.sink_n, skip_at = walk.skip_at, gap = walk.gap, n_walk = walk.n_walk;
    auto chunk_of = [&](uint32_t i) -> uint32_t { return OPT && i >= skip_at ? i + gap : i; };
    const uint32_t used = oxb_attn_slots_used(n_walk, p.n_splits);
    if (slot >= used) return;  // never read by the merge
    const bool owner = (n_walk - 1) % used == slot;  // this workgroup stores the new position
    float* part = p.part + (((size_t)b * p.nq + h0) * p.n_splits + slot) * (HD + OXB_ATTN_PART_PAD);
    const size_t part_head = (size_t)p.n_splits * (HD + OXB_ATTN_PART_PAD);
    // slot results go out through agent-coherent stores: a workgroup of this same launch merges them
    const __amdgpu_buffer_rsrc_t r_out = make_rsrc(part, (uint32_t)(G * part_head * 4u));
    auto put = [&](size_t idx, float v) { buf_store_b32_coherent(r_out, (uint32_t)idx * 4u, v); };
    const float* qkv = p.qkv + (size_t)b * p.qkv_stride;
    const float* cs = p.cos_t + (size_t)pos * half;
    const float* sn = p.sin_t + (size_t)pos * half;
    cache_t* Kc = reinterpret_cast<cache_t*>(p.k_cache);
    cache_t* Vc = reinterpret_cast<cache_t*>(p.v_cache);
    float* Ksc = p.k_scale;  // one scale per row
    float* Vsc = p.v_scale;
    // Rows of this (sequence, layer, kv head).  A wave's block of 32 keys is two tiles of 16, each contiguous (pages hold 16 positions or more):
    // where a tile lies is the same for every lane, so its rows are read through a buffer descriptor that begins there, at offsets that never
    // change, and that ends with the sequence: rows past the last key read as zeros and take no bandwidth (their scores are masked).  Per-lane
    // addresses and a test of every key's visibility were a third of a chunk's 400 to 500 vector instructions; without them, us per launch (8B
    // shape): FP8 in pages of 16 at 32 000 23.1 -> 21.4, INT8 there 21.6 -> 20.5, 32 of INT8 at 2048 33.0 -> 32.3, eight at 4000 21.9 -> 21.0; fp16,
    // one at 2048 9.2 -> 8.9, six 16.9 -> 16.4, one of 16 heads at 700 7.6 -> 7.3.  In a paged cache the two page numbers come from the sequence's
    // table, one broadcast load each, one chunk before the rows are requested, so that no row load waits for a lookup.  (Keeping the table in
    // LDS instead was measured slower: the 8 KB cost a workgroup per CU.)
    const bool paged = OPT && p.kv.page_table != nullptr;
    const uint32_t pshift = p.kv.page_shift, pmask = (1u << pshift) - 1u;
    const size_t row0 = paged ? ((size_t)(p.layer * p.nkv + kvh) * p.kv.n_pages) << pshift : kv_row(p.kv, b, p.layer, kvh, 0);
    const uint32_t* tbl = paged ? p.kv.page_table + (size_t)b * p.kv.table_stride : nullptr;
    auto pages_of = [&](uint32_t chunk, uint32_t& pa, uint32_t& pb) {
        pa = pb = 0;
        if (!paged) return;
        const uint32_t key0 = chunk * CH + 32 * wave, i0 = min(key0, seq_len - 1) >> pshift, i1 = min(key0 + 16, seq_len - 1) >> pshift;
        pa = (uint32_t)__builtin_amdgcn_readfirstlane((int)tbl[i0]);
        pb = (uint32_t)__builtin_amdgcn_readfirstlane((int)tbl[i1]);
    };
    struct Tile { size_t row; uint32_t n; };  // first row, and how many of the 16 are there
    auto tile_of = [&](uint32_t key, uint32_t page) -> Tile {
        // (Opaque: of key < seq_len ? min(seq_len - key, 16) : 0 the compiler drops the test, for it takes the difference in the minimum
        // for one that never wraps; other ways to write it become vector instructions, and the descriptors loops: six sequences
        // 16.7 -> 18.4 us.)
        uint32_t left = seq_len - key;
        asm("" : "+s"(left));
        const uint32_t n = key < seq_len ? min(left, 16u) : 0u;
        return {paged ? row0 + ((size_t)page << pshift) + (key & pmask) : row0 + key, n};
    };

    // K rows of the two 16-key tiles (A operands) and this lane's pieces of the 32-key V block of a chunk.
    v8h_t k0r[QC ? 1 : KS], k1r[QC ? 1 : KS];
    kvi2_t k0q[QC ? KS : 1], k1q[QC ? KS : 1];
    float4 ksc0, ksc1, vsc0, vsc1;  // row scales of the lane's keys 4g .. 4g+3 and 16+4g .. 16+4g+3
    v4i vr[VL];
    constexpr uint32_t RB = HD * sizeof(cache_t);  // bytes of a row
    const uint32_t k_at = qi * RB + g * (QC ? HD / 4 : 16), v_at = (lane / VPR) * RB + (lane % VPR) * 16;
    auto scales = [&](const float* s, const Tile& t) -> float4 {
        const v4i v = buf_load_b128(make_rsrc(s + t.row, t.n * 4u), 16u * g);
        return make_float4(__int_as_float(v.x), __int_as_float(v.y), __int_as_float(v.z), __int_as_float(v.w));
    };
    auto load_k = [&](uint32_t chunk, uint32_t pa, uint32_t pb) {
        const uint32_t key0 = chunk * CH + 32 * wave;
        const Tile t0 = tile_of(key0, pa), t1 = tile_of(key0 + 16, pb);
        const __amdgpu_buffer_rsrc_t r0 = make_rsrc(Kc + t0.row * HD, t0.n * RB), r1 = make_rsrc(Kc + t1.row * HD, t1.n * RB);
        if constexpr (QC && KS % 2 == 0) {
#pragma unroll
            for (int s = 0; s < KS; s += 2) {
                const v4i a = buf_load_b128(r0, k_at + 8 * s), c = buf_load_b128(r1, k_at + 8 * s);
                k0q[s] = (kvi2_t){a.x, a.y}, k0q[QC ? s + 1 : 0] = (kvi2_t){a.z, a.w};
                k1q[s] = (kvi2_t){c.x, c.y}, k1q[QC ? s + 1 : 0] = (kvi2_t){c.z, c.w};
            }
        } else {
#pragma unroll
            for (int s = 0; s < KS; s++) {
                if constexpr (QC) {
                    const v2u a = __builtin_amdgcn_raw_buffer_load_b64(r0, (int)(k_at + 8 * s), 0, 0), c = __builtin_amdgcn_raw_buffer_load_b64(r1, (int)(k_at + 8 * s), 0, 0);
                    k0q[s] = (kvi2_t){(int)a.x, (int)a.y}, k1q[s] = (kvi2_t){(int)c.x, (int)c.y};
                } else {
                    k0r[s] = __builtin_bit_cast(v8h_t, buf_load_b128(r0, k_at + 64 * s));
                    k1r[s] = __builtin_bit_cast(v8h_t, buf_load_b128(r1, k_at + 64 * s));
                }
            }
        }
        if constexpr (QC) ksc0 = scales(Ksc, t0), ksc1 = scales(Ksc, t1);
    };
    auto load_v = [&](uint32_t chunk, uint32_t pa, uint32_t pb) {
        const uint32_t key0 = chunk * CH + 32 * wave;
        const Tile t0 = tile_of(key0, pa), t1 = tile_of(key0 + 16, pb);
        const __amdgpu_buffer_rsrc_t r0 = make_rsrc(Vc + t0.row * HD, t0.n * RB), r1 = make_rsrc(Vc + t1.row * HD, t1.n * RB);
        // piece i: rows i * 64 / VPR + lane / VPR of the block
        if constexpr (VL == 1) {  // (rows of 32 bytes: one piece a lane, its tile by lane)
            const v4i a = buf_load_b128(r0, lane < 32 ? v_at : OXB_OOB), c = buf_load_b128(r1, lane < 32 ? OXB_OOB : v_at - 16 * RB);
            vr[0] = (v4i){a.x | c.x, a.y | c.y, a.z | c.z, a.w | c.w};
        } else {
#pragma unroll
            for (int i = 0; i < VL; i++) vr[i] = buf_load_b128(i < VL / 2 ? r0 : r1, v_at + (i % (VL / 2 ? VL / 2 : 1)) * (64 / VPR) * RB);
        }
        if constexpr (QC) vsc0 = scales(Vsc, t0), vsc1 = scales(Vsc, t1);
    };

    // The rows of the first chunk are requested before anything else, so that their way from HBM overlaps the Q prologue.
    // The new position's row is not in the cache then (rows past the end read as zeros): in the chunk that holds it, it is
    // patched in from LDS, with the very values the cache receives, so no workgroup waits for its own stores.
    const uint32_t pos_walk = n_walk - 1;
    uint32_t na = 0, nb = 0;  // pages of the chunk whose rows are requested next
    auto request_first = [&]() {
        uint32_t pa, pb;
        const uint32_t first = chunk_of(slot);
        pages_of(first, pa, pb);
        load_k(first, pa, pb);
        load_v(first, pa, pb);
        if (slot + used < n_walk) pages_of(chunk_of(slot + used), na, nb);
    };
    // Inputs of the prologue, requested before the cache rows: loads return in issue order, so whatever the prologue
    // waits for must not queue behind the rows from HBM.  Lane d holds elements d and d + hd/2 of a head (the RoPE pair).
    constexpr int KI = (HD / 2 + 63) / 64;
    struct HeadIn { float lo[KI], hi[KI]; };
    auto load_head = [&](const float* in, HeadIn& r) {
#pragma unroll
        for (int it = 0; it < KI; it++) {
            const uint32_t d = lane + 64 * it;
            r.lo[it] = d < half ? in[d] : 0.f;
            r.hi[it] = d < half ? in[d + half] : 0.f;
        }
    };
    // sum of squares in the order of a strided walk over the head (all low halves, then all high halves)
    auto head_inv_rms = [&](const HeadIn& r) {
        float ss = 0.f;
#pragma unroll
        for (int it = 0; it < KI; it++) ss = fmaf(r.lo[it], r.lo[it], ss);
#pragma unroll
        for (int it = 0; it < KI; it++) ss = fmaf(r.hi[it], r.hi[it], ss);
        ss = wave_sum_f32(ss);
        return 1.0f / sqrtf(ss / (float)HD + p.eps);
    };
    // The owner's last two waves take the new K and V rows: up to NW - 2 heads have waves of their own.
    constexpr uint32_t KW = NW - 2, VW = NW - 1;
    HeadIn q_in, cs_sn, qn, kv_in, kn;  // cs_sn: lo = cos, hi = sin; kv_in: the new K row (wave KW) or V row (wave VW) of the owner
    {
#pragma unroll
        for (int it = 0; it < KI; it++) {
            const uint32_t d = lane + 64 * it;
            cs_sn.lo[it] = d < half ? cs[d] : 0.f;
            cs_sn.hi[it] = d < half ? sn[d] : 0.f;
        }
        load_head(p.q_norm, qn);
        if (wave < G) load_head(qkv + (size_t)(h0 + wave) * HD, q_in);
        if (owner && wave == KW) {
            load_head(qkv + (size_t)(p.nq + kvh) * HD, kv_in);
            load_head(p.k_norm, kn);
        } else if (owner && wave == VW) {
            load_head(qkv + (size_t)(p.nq + p.nkv + kvh) * HD, kv_in);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    request_first();
    __builtin_amdgcn_sched_barrier(0);
    // --- Q of the group's heads: RMSNorm over the head, RoPE on the pairs (d, d + hd/2), times 1/sqrt(hd) ---
    for (uint32_t h = wave; h < G; h += NW) {
        if (h != wave) load_head(qkv + (size_t)(h0 + h) * HD, q_in);
        const float inv = head_inv_rms(q_in);
#pragma unroll
        for (int it = 0; it < KI; it++) {
            const uint32_t d = lane + 64 * it;
            if (d < half) {
                const float lo_ = qn.lo[it] * q_in.lo[it] * inv, hi_ = qn.hi[it] * q_in.hi[it] * inv;
                // split into fp16 hi + lo here, once per value (not once per lane that reads it)
                const float qa = (lo_ * cs_sn.lo[it] - hi_ * cs_sn.hi[it]) * p.scale, qb = (lo_ * cs_sn.hi[it] + hi_ * cs_sn.lo[it]) * p.scale;
                const _Float16 ha = (_Float16)qa, hb = (_Float16)qb;
                qs[0][h * HD + d] = ha;
                qs[1][h * HD + d] = (_Float16)(qa - (float)ha);
                qs[0][h * HD + d + half] = hb;
                qs[1][h * HD + d + half] = (_Float16)(qb - (float)hb);
            }
        }
    }
    // --- K and V of the new position, by the workgroup whose slot walks its chunk ---
    const size_t new_row = kv_row(p.kv, b, p.layer, kvh, pos);
    if (owner) {
        if (wave == KW) {
            const float inv = head_inv_rms(kv_in);
            float klo[KI], khi[KI], mx = 0.f;
#pragma unroll
            for (int it = 0; it < KI; it++) {
                const uint32_t d = lane + 64 * it;
                klo[it] = khi[it] = 0.f;
                if (d < half) {
                    const float lo_ = kn.lo[it] * kv_in.lo[it] * inv, hi_ = kn.hi[it] * kv_in.hi[it] * inv;
                    klo[it] = lo_ * cs_sn.lo[it] - hi_ * cs_sn.hi[it];
                    khi[it] = lo_ * cs_sn.hi[it] + hi_ * cs_sn.lo[it];
                    mx = fmaxf(mx, fmaxf(fabsf(klo[it]), fabsf(khi[it])));
                }
            }
            float scale = 1.f;
            if constexpr (QC) {
                mx = wave_max_f32(mx);
                scale = kv_row_scale<KVM>(mx);
                if (lane == 0) Ksc[new_row] = kv_new_scale[0] = scale;
            }
#pragma unroll
            for (int it = 0; it < KI; it++) {
                const uint32_t d = lane + 64 * it;
                if (d < half) {
                    if constexpr (QC) {
                        Kc[new_row * HD + d] = kv_new[0][d] = (uint8_t)kv_encode<KVM>(klo[it], scale);
                        Kc[new_row * HD + d + half] = kv_new[0][d + half] = (uint8_t)kv_encode<KVM>(khi[it], scale);
                    } else {
                        Kc[new_row * HD + d] = kv_new[0][d] = (_Float16)klo[it];
                        Kc[new_row * HD + d + half] = kv_new[0][d + half] = (_Float16)khi[it];
                    }
                }
            }
        } else if (wave == VW) {
            float mx = 0.f;
#pragma unroll
            for (int it = 0; it < KI; it++) mx = fmaxf(mx, fmaxf(fabsf(kv_in.lo[it]), fabsf(kv_in.hi[it])));
            float scale = 1.f;
            if constexpr (QC) {
                mx = wave_max_f32(mx);
                scale = kv_row_scale<KVM>(mx);
                if (lane == 0) Vsc[new_row] = kv_new_scale[1] = scale;
            }
#pragma unroll
            for (int it = 0; it < KI; it++) {
                const uint32_t d = lane + 64 * it;
                if (d < half) {
                    if constexpr (QC) {
                        Vc[new_row * HD + d] = kv_new[1][d] = (uint8_t)kv_encode<KVM>(kv_in.lo[it], scale);
                        Vc[new_row * HD + d + half] = kv_new[1][d + half] = (uint8_t)kv_encode<KVM>(kv_in.hi[it], scale);
                    } else {
                        Vc[new_row * HD + d] = kv_new[1][d] = (_Float16)kv_in.lo[it];
                        Vc[new_row * HD + d + half] = kv_new[1][d + half] = (_Float16)kv_in.hi[it];
                    }
                }
            }
        }
    }
    lds_barrier();  // publishes qs and the LDS copy of the new rows; the requested cache rows stay in flight across it

    // B operands: lane (head = qi, g) holds the eight Q values that meet its K values in step s, as hi + lo: one
    // 16-byte LDS read each.  Columns past the group's heads repeat head 0; nothing of them is ever stored.
    v8h_t qh[KS], ql[KS];
    const uint32_t hq = qi < G ? qi : 0u;
#pragma unroll
    for (int s = 0; s < KS; s++) {
        const uint32_t d = QC ? (HD / 4) * g + 8 * s : 32 * s + 8 * g;
        qh[s] = *reinterpret_cast<const v8h_t*>(&qs[0][hq * HD + d]);
        ql[s] = *reinterpret_cast<const v8h_t*>(&qs[1][hq * HD + d]);
    }
    v4f O[NS];
#pragma unroll
    for (int i = 0; i < NS; i++) O[i] = (v4f){0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f, u_run = QC ? 0.f : 1.f;  // u_run: the unit of O (largest V row scale so far)
    _Float16* vs = vs_all[wave];

    for (uint32_t i = slot; i < n_walk;) {
        const uint32_t key0 = chunk_of(i) * CH + 32 * wave;
        const bool patch = i == pos_walk;  // (the last chunk of the owner's walk)
        i += used;
        const bool more = i < n_walk;
        const uint32_t nxt = chunk_of(i);
        if (patch) {  // (uniform)
#pragma unroll
            for (int j = 0; j < VL; j++) {
                const uint32_t id = j * 64 + lane;
                if (key0 + id / VPR == pos) vr[j] = *reinterpret_cast<const v4i*>(&kv_new[1][(id % VPR) * (QC ? 16 : 8)]);
            }
        }
        // stage the V block in the wave's LDS slice (the previous block's gathers were issued before: LDS runs in
        // order) and request the next chunk's
#pragma unroll
        for (int j = 0; j < VL; j++) {
            const uint32_t id = j * 64 + lane;
            if constexpr (QC) {
                uint32_t d[8];
                const v4i piece = vr[j];
                kv_dec4<KVM>((uint32_t)piece.x, d[0], d[1]);
                kv_dec4<KVM>((uint32_t)piece.y, d[2], d[3]);
                kv_dec4<KVM>((uint32_t)piece.z, d[4], d[5]);
                kv_dec4<KVM>((uint32_t)piece.w, d[6], d[7]);
                _Float16* dst = vs + (id / VPR) * VSTR + (id % VPR) * 16;
                *reinterpret_cast<v4i*>(dst) = (v4i){(int)d[0], (int)d[1], (int)d[2], (int)d[3]};
                *reinterpret_cast<v4i*>(dst + 8) = (v4i){(int)d[4], (int)d[5], (int)d[6], (int)d[7]};
            } else {
                *reinterpret_cast<v4i*>(vs + (id / VPR) * VSTR + (id % VPR) * 8) = vr[j];
            }
        }
        float4 vc0 = vsc0, vc1 = vsc1;
        auto patch_scale = [&](float4& a, uint32_t first_key, float v) {  // the scale of position `pos`, if it is one of the four
            if (first_key == pos) a.x = v;
            if (first_key + 1 == pos) a.y = v;
            if (first_key + 2 == pos) a.z = v;
            if (first_key + 3 == pos) a.w = v;
        };
        if (QC && patch) {
            patch_scale(vc0, key0 + 4 * g, kv_new_scale[1]);
            patch_scale(vc1, key0 + 16 + 4 * g, kv_new_scale[1]);
        }
        if (more) load_v(nxt, na, nb);
        v4f s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
        if (patch) {  // (uniform)
#pragma unroll
            for (int s = 0; s < KS; s++) {
                if constexpr (QC) {
                    const kvi2_t cn = *reinterpret_cast<const kvi2_t*>(&kv_new[0][(HD / 4) * g + 8 * s]);
                    if (key0 + qi == pos) k0q[s] = cn;
                    if (key0 + 16 + qi == pos) k1q[s] = cn;
                } else {
                    if (key0 + qi == pos) k0r[s] = *reinterpret_cast<const v8h_t*>(&kv_new[0][32 * s + 8 * g]);
                    if (key0 + 16 + qi == pos) k1r[s] = *reinterpret_cast<const v8h_t*>(&kv_new[0][32 * s + 8 * g]);
                }
            }
        }
#pragma unroll
        for (int s = 0; s < KS; s++) {
            v8h_t a0, a1;
            if constexpr (QC) {
                a0 = kv_dec8<KVM>(k0q[s]);
                a1 = kv_dec8<KVM>(k1q[s]);
            } else {
                a0 = k0r[s];
                a1 = k1r[s];
            }
            s0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(a0, qh[s], s0, 0, 0, 0);
            s0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(a0, ql[s], s0, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(a1, qh[s], s1, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(a1, ql[s], s1, 0, 0, 0);
        }
        float4 kc0 = ksc0, kc1 = ksc1;
        if (QC && patch) {
            patch_scale(kc0, key0 + 4 * g, kv_new_scale[0]);
            patch_scale(kc1, key0 + 16 + 4 * g, kv_new_scale[0]);
        }
        if (more) {
            load_k(nxt, na, nb);
            if (i + used < n_walk) pages_of(chunk_of(i + used), na, nb);  // used by the next iteration's requests
        }
        // this wave's part of the chunk holds no visible key (past the end, or outside the window)
        if (!(key0 < sink_n || max(key0, lo) < min(key0 + 32, seq_len))) continue;
        // this lane: head qi, keys key0 + 4g + v and key0 + 16 + 4g + v
        const bool whole = (key0 >= lo && key0 + 32 <= seq_len) || (OPT && key0 + 32 <= sink_n);  // every key of the block is visible
        float sv[8];
        if constexpr (QC) {
            const float ka[8] = {kc0.x, kc0.y, kc0.z, kc0.w, kc1.x, kc1.y, kc1.z, kc1.w};
#pragma unroll
            for (int v = 0; v < 4; v++) sv[v] = s0[v] * ka[v], sv[4 + v] = s1[v] * ka[4 + v];
        } else {
#pragma unroll
            for (int v = 0; v < 4; v++) sv[v] = s0[v], sv[4 + v] = s1[v];
        }
        if (!whole) {  // (uniform) an invisible key's score and V row scale count for nothing
            float va[8] = {vc0.x, vc0.y, vc0.z, vc0.w, vc1.x, vc1.y, vc1.z, vc1.w};
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const uint32_t key = key0 + (e >> 2) * 16 + 4 * g + (e & 3);
                const bool vis = key < sink_n || (key >= lo && key < seq_len);
                sv[e] = vis ? sv[e] : -INFINITY;
                va[e] = vis ? va[e] : 0.f;
            }
            if (QC) vc0 = make_float4(va[0], va[1], va[2], va[3]), vc1 = make_float4(va[4], va[5], va[6], va[7]);
        }
        float mx = sv[0];
#pragma unroll
        for (int e = 1; e < 8; e++) mx = fmaxf(mx, sv[e]);
        mx = max_rows4(mx);
        const float m_new = fmaxf(m_run, mx);      // finite: the block holds a visible key
        float alpha = __expf(m_run - m_new);         // 0 for the wave's first block
        float vw[8] = {1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f};  // V row scales of the lane's keys in units of u_run
        if constexpr (QC) {
            const float va[8] = {vc0.x, vc0.y, vc0.z, vc0.w, vc1.x, vc1.y, vc1.z, vc1.w};
            float vmx = 0.f;
#pragma unroll
            for (int e = 0; e < 8; e++) vmx = fmaxf(vmx, va[e]);
            vmx = max_rows4(vmx);
            const float u_new = fmaxf(u_run, vmx);  // > 0: a visible row's scale is at least f32::EPSILON
            const float inv_u = 1.0f / u_new;
#pragma unroll
            for (int e = 0; e < 8; e++) vw[e] = va[e] * inv_u;
            l_run = l_run * alpha;                  // the sum is rescaled by the softmax factor only
            alpha *= u_run * inv_u;                 // the accumulator also changes its unit
            u_run = u_new;
        } else {
            l_run = l_run * alpha;
        }
        float sum = 0.f;
        v8h_t ph, pl;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const float pe = __expf(sv[e] - m_new);
            sum += pe;
            const float pv = QC ? pe * vw[e] : pe;
            const _Float16 hi = (_Float16)pv;
            ph[e] = hi;
            pl[e] = (_Float16)(pv - (float)hi);
        }
        sum = sum_rows4(sum);
        l_run += sum;
        m_run = m_new;
        // O^T += V^T P^T; A operand gathered from the staged block
#pragma unroll
        for (int sl = 0; sl < NS; sl++) {
            // a[e] = V[4 g + e][16 sl + qi], a[4 + e] = V[16 + 4 g + e][16 sl + qi]: two transposing LDS reads.  The 16 lanes
            // of a block hand in the addresses of a 4 x 16 tile (lane i: row i / 4, columns 4 (i % 4) .. + 3) and lane j
            // receives column j.
            const _Float16* tile = vs + (4 * g + (qi >> 2)) * VSTR + 16 * sl + 4 * (qi & 3u);
            const v4h_t t0 = lds_read_tr16(tile), t1 = lds_read_tr16(tile + 16 * VSTR);
            const v8h_t a = {t0[0], t0[1], t0[2], t0[3], t1[0], t1[1], t1[2], t1[3]};
#pragma unroll
            for (int v = 0; v < 4; v++) O[sl][v] *= alpha;
            O[sl] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, ph, O[sl], 0, 0, 0);
            O[sl] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, pl, O[sl], 0, 0, 0);
        }
    }
    // --- merge the waves: lane (head = qi, g) holds O[head][16 sl + 4 g + v], m_run, l_run ---
    __syncthreads();  // the V slices are dead: reuse them
    static_assert(sizeof(vs_all) >= (NW * 16 * HD + 2 * NW * 16) * sizeof(float), "merge buffers must fit in the V slices");
    float* mo = reinterpret_cast<float*>(&vs_all[0][0]);  // [wave][head 16][HD], then [wave][head 16] m, [wave][head 16] l
    float* mm = mo + NW * 16 * HD;
    float* ml = mm + NW * 16;
    if (qi < G) {
#pragma unroll
        for (int sl = 0; sl < NS; sl++)
            *reinterpret_cast<float4*>(&mo[(wave * 16 + qi) * HD + 16 * sl + 4 * g]) =
                make_float4(O[sl][0] * u_run, O[sl][1] * u_run, O[sl][2] * u_run, O[sl][3] * u_run);
    }
    if (g == 0) {
        mm[wave * 16 + qi] = m_run;
        ml[wave * 16 + qi] = l_run;
    }
    __syncthreads();
    constexpr bool pack = OUT == OXB_ATTN_OUT_PACK;  // (G * HD is 512)
    float* keep = reinterpret_cast<float*>(&qs[0][0]);  // a single slot's outputs, for the quantiser
    static_assert(sizeof(qs) >= 512 * sizeof(float), "room for them");
    for (uint32_t i = tid; i < G * HD; i += NT) {
        const uint32_t h = i / HD, d = i % HD;
        float M = mm[h];
#pragma unroll
        for (uint32_t w = 1; w < NW; w++) M = fmaxf(M, mm[w * 16 + h]);
        float o = 0.f, l = 0.f;
#pragma unroll
        for (uint32_t w = 0; w < NW; w++) {
            const float wgt = mm[w * 16 + h] == -INFINITY ? 0.f : __expf(mm[w * 16 + h] - M);  // a wave that saw no key
            o = fmaf(mo[(w * 16 + h) * HD + d], wgt, o);
            l = fmaf(ml[w * 16 + h], wgt, l);
        }
        if (used == 1) {  // the only slot: what the merge would compute (weight 1, times 1 / sum)
            o *= l > 0.f ? 1.0f / l : 0.f;
            if constexpr (OUT == OXB_ATTN_OUT_XH) p.op.xh[oxb_operand_index(p.op.fmt, (h0 + h) * HD + d, b, p.op.M_pad)] = (_Float16)ldexpf(o, p.op.shift);
            else p.out[((size_t)b * p.nq + h0 + h) * HD + d] = o;
            if (pack) keep[i] = o;
            continue;
        }
        put(h * part_head + d, o);
        if (d == 0) {
            put(h * part_head + HD, M);
            put(h * part_head + HD + 1, l);
        }
    }
    if (used == 1) {
        if (pack) {
            __syncthreads();
            attn_pack_outputs(p, b, h0, keep);
        }
        return;
    }
    if (OUT == OXB_ATTN_OUT_F32 && used <= p.leave) return;  // (few slots: the O projection adds them up)
    if (attn_last_arrival(p, b, kvh, used, &last_flag))  // (the barrier inside also retires mo / mm / ml)
        attn_merge_heads<NT, OUT>(p, b, h0, G, used, reinterpret_cast<float*>(&vs_all[0][0]));
}

// One wave quantises the 512 outputs of a kv head's q heads (LDS) for the O projection: superblock h_first * hd / 512 of
// vector b.
__device__ __forceinline__ void attn_pack_outputs(const OxbAttnParams& p, uint32_t b, uint32_t h_first, const float* kf) {
    const uint32_t tid = threadIdx.x, e0 = h_first * p.hd;
    if (tid >= 64) return;
    float xe[2][4];
    if (p.pack_fmt == OXB_FMT_Q1) {
#pragma unroll
        for (int pass = 0; pass < 2; pass++)
#pragma unroll
            for (int bb = 0; bb < 4; bb++) xe[pass][bb] = kf[gemv_pack_elem<OXB_FMT_Q1>(tid, pass, bb)];
        gemv_pack_write<OXB_FMT_Q1>(xe, 0.f, tid, e0 / 512u, b, p.pack_n_sb, p.pack_nvg, p.pack_out);
    } else {
#pragma unroll
        for (int pass = 0; pass < 2; pass++)
#pragma unroll
            for (int bb = 0; bb < 4; bb++) xe[pass][bb] = kf[gemv_pack_elem<OXB_FMT_TQ2>(tid, pass, bb)];
        gemv_pack_write<OXB_FMT_TQ2>(xe, 0.f, tid, e0 / 512u, b, p.pack_n_sb, p.pack_nvg, p.pack_out);
    }
}

// Merge the slot results of heads h_first .. h_first + nh - 1 of sequence b into the attention output
// [batch][nq * hd] (fp32), the input of the O projection, by the NT threads of a workgroup: per head one wave works
// out the softmax weights of the slots (one slot per lane); the weighted slot outputs of a group of four dimensions
// are added by NPAR threads, thread j taking slots j, j + NPAR, ... in ascending order, and the NPAR sums meet in LDS
// in thread order.  Every thread requests its first 16 slot outputs before the weights are worked out; NPAR is the
// smallest of 1, 2, 4 that covers the slots in use with those requests (one round trip to memory for the whole merge),
// as far as the threads allow for the heads' nh * hd / 4 groups.
// sm: nh * 65 floats of LDS ([head][64] slot weights | [head] 1 / sum), then NT float4 for the partial sums.
// The slot results were written by other workgroups of this same launch: agent-coherent loads.
template <uint32_t NT, int OUT>
__device__ __forceinline__ void attn_merge_heads(const OxbAttnParams& p, uint32_t b, uint32_t h_first, uint32_t nh, uint32_t used, float* sm) {
    const uint32_t tid = threadIdx.x, lane = tid & 63u, hd = p.hd, qd = p.nq * hd;
    const uint32_t stride = hd + OXB_ATTN_PART_PAD;
    float* wts = sm;
    float* inv_l = wts + nh * 64;
    float4* sums = reinterpret_cast<float4*>(sm + ((nh * 65 + 3) & ~3u));
    // The merged outputs once more, for the quantiser at the end: 128 groups of four, in the entries of `sums` that the
    // partial sums never use (those are written by threads tg and up, and with 128 groups tg >= 128).
    float4* keep = sums;
    constexpr bool pack = OUT == OXB_ATTN_OUT_PACK;  // (nh * hd is 512)
    const uint32_t e0 = h_first * hd;
    const float* part = p.part + (size_t)b * p.nq * p.n_splits * stride;
    const __amdgpu_buffer_rsrc_t r_part = make_rsrc(part, p.nq * p.n_splits * stride * 4u);
    auto ld4 = [&](const float* q) -> float4 {
        const v4f v = buf_load_f128_coherent(r_part, (uint32_t)(q - part) * 4u);
        return make_float4(v.x, v.y, v.z, v.w);
    };
    auto ld1 = [&](const float* q) -> float { return buf_load_f32_coherent(r_part, (uint32_t)(q - part) * 4u); };
    const uint32_t groups = nh * hd / 4;
    // as few threads per group as keep all slots within the first 16 requests (more would only add the LDS step)
    const uint32_t npar_max = groups <= NT / 4 ? 4u : groups <= NT / 2 ? 2u : 1u;
    const uint32_t npar = used <= 16u || npar_max == 1u ? 1u : (used <= 32u || npar_max == 2u ? 2u : 4u);
    const uint32_t tg = NT / npar, sh = tid / tg, egl = tid % tg;  // this thread: group egl (+ tg, ...), slots sh + npar u
    constexpr int PRE = 16;
    float4 pre[PRE];
    // the maxima and sums of the wave's first head are requested ahead of the slot outputs: loads return in issue
    // order, and the weights are worked out while the outputs are still on their way
    float mv0 = -INFINITY, lv0 = 0.f;
    if ((tid >> 6) < nh) {
        const float* ph = part + ((size_t)(h_first + (tid >> 6)) * p.n_splits + lane) * stride + hd;
        if (lane < used) mv0 = ld1(ph), lv0 = ld1(ph + 1);
    }
    {
        const uint32_t e = e0 + egl * 4;
        const float* ph = part + (size_t)(e / hd) * p.n_splits * stride + e % hd;
#pragma unroll
        for (int u = 0; u < PRE; u++) {
            const uint32_t sl = sh + npar * u;
            pre[u] = (egl < groups && sl < used) ? ld4(ph + (size_t)sl * stride) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    }
    for (uint32_t hh = tid >> 6; hh < nh; hh += NT / 64) {
        const float* ph = part + ((size_t)(h_first + hh) * p.n_splits + lane) * stride + hd;
        const bool first_head = hh == (tid >> 6);
        const float mv = first_head ? mv0 : (lane < used ? ld1(ph) : -INFINITY), lv = first_head ? lv0 : (lane < used ? ld1(ph + 1) : 0.f);
        float M = mv;
        M = wave_max_f32(M);
        const float w = lane < used ? __expf(mv - M) : 0.f;
        float L = w * lv;
        L = wave_sum_f32(L);
        wts[hh * 64 + lane] = w;
        if (lane == 0) inv_l[hh] = L > 0.f ? 1.0f / L : 0.f;
    }
    __syncthreads();
    for (uint32_t eg0 = 0; eg0 < groups; eg0 += tg) {  // uniform trip count: the barrier below is reached by every thread
        const uint32_t eg = eg0 + egl, e = e0 + eg * 4;
        const bool live = eg < groups;
        const uint32_t h = live ? e / hd : h_first, d = e % hd, hh = h - h_first;
        const float* ph = part + (size_t)h * p.n_splits * stride + d;
        float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
        // PRE requests in flight at a time; slots past `used` count as zeros with weight 0
        auto fold = [&](const float4 (&v)[PRE], uint32_t u0) {
#pragma unroll
            for (int u = 0; u < PRE; u++) {
                const uint32_t sl = sh + npar * (u0 + u);
                const float w = sl < used ? wts[hh * 64 + sl] : 0.f;
                acc.x = fmaf(v[u].x, w, acc.x), acc.y = fmaf(v[u].y, w, acc.y), acc.z = fmaf(v[u].z, w, acc.z), acc.w = fmaf(v[u].w, w, acc.w);
            }
        };
        uint32_t u0 = 0;
        if (eg0 == 0) {  // the group whose first slots are already here
            fold(pre, 0);
            u0 = PRE;
        }
        for (; live && sh + npar * u0 < used; u0 += PRE) {
            float4 v[PRE];
#pragma unroll
            for (int u = 0; u < PRE; u++) {
                const uint32_t sl = sh + npar * (u0 + u);
                v[u] = sl < used ? ld4(ph + (size_t)sl * stride) : make_float4(0.f, 0.f, 0.f, 0.f);
            }
            fold(v, u0);
        }
        if (npar > 1) {  // (then all groups fit one pass)
            if (sh) sums[tid] = acc;
            __syncthreads();
            if (!sh)
                for (uint32_t j = 1; j < npar; j++) {
                    const float4 o = sums[j * tg + egl];
                    acc.x += o.x, acc.y += o.y, acc.z += o.z, acc.w += o.w;
                }
        }
        if (live && !sh) {
            const float il = inv_l[hh];
            acc.x *= il, acc.y *= il, acc.z *= il, acc.w *= il;
            if constexpr (OUT == OXB_ATTN_OUT_XH) operand_store4(p.op, e, b, acc.x, acc.y, acc.z, acc.w);
            else *reinterpret_cast<float4*>(p.out + (size_t)b * qd + e) = acc;
            if (pack) keep[eg] = acc;
        }
    }
    if (pack) {  // (uniform)
        __syncthreads();
        attn_pack_outputs(p, b, h_first, reinterpret_cast<const float*>(keep));
    }
}

// ---------------------------------------------------------------------------
// Greedy selection: index of the first maximum (strict '>', as argmax_f32, cuda_kernels.rs:407-436).
// Two stages: grid (parts, vectors) workgroups each reduce a contiguous span to (value, index), then one
// wave per vector merges the parts; ties go to the lower index at every step.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void argmax_merge(float& best, uint32_t& idx, float ob, uint32_t oi) {
    if (oi != 0xFFFFFFFFu && (idx == 0xFFFFFFFFu || ob > best || (ob == best && oi < idx))) { best = ob; idx = oi; }
}

__global__ __launch_bounds__(256) void argmax_partial_kernel(const float* __restrict__ logits, uint32_t n, uint32_t span,
                                                              float* __restrict__ pv, uint32_t* __restrict__ pi) {
    __shared__ float sv[4];
    __shared__ uint32_t si[4];
    const float* v = logits + (size_t)blockIdx.y * n;
    const uint32_t i0 = blockIdx.x * span, i1 = min(i0 + span, n);
    float best = -INFINITY;
    uint32_t idx = 0xFFFFFFFFu;
    for (uint32_t i = i0 + threadIdx.x; i < i1; i += 256) {
        const float x = v[i];
        if (idx == 0xFFFFFFFFu || x > best) { best = x; idx = i; }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) argmax_merge(best, idx, __shfl_xor(best, o, 64), __shfl_xor(idx, o, 64));
    if ((threadIdx.x & 63u) == 0) { sv[threadIdx.x >> 6] = best; si[threadIdx.x >> 6] = idx; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 4; w++) argmax_merge(best, idx, sv[w], si[w]);
        pv[blockIdx.y * gridDim.x + blockIdx.x] = best;
        pi[blockIdx.y * gridDim.x + blockIdx.x] = idx;
    }
}

__global__ __launch_bounds__(64) void argmax_final_kernel(const float* __restrict__ pv, const uint32_t* __restrict__ pi,
                                                           uint32_t parts, uint32_t* __restrict__ out, uint32_t* __restrict__ host_copy) {
    float best = -INFINITY;
    uint32_t idx = 0xFFFFFFFFu;
    for (uint32_t i = threadIdx.x; i < parts; i += 64) argmax_merge(best, idx, pv[blockIdx.x * parts + i], pi[blockIdx.x * parts + i]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) argmax_merge(best, idx, __shfl_xor(best, o, 64), __shfl_xor(idx, o, 64));
    if (threadIdx.x == 0) {
        out[blockIdx.x] = idx == 0xFFFFFFFFu ? 0u : idx;
        if (host_copy) {  // pinned host memory: the caller reads it after synchronising, without a copy of its own
            host_copy[blockIdx.x] = idx == 0xFFFFFFFFu ? 0u : idx;
            __threadfence_system();
        }
    }
}

// Pinned host staging -> device: the hidden rows and positions of a decode call, in one launch ahead of the step's
// graph (two small asynchronous copies cost more than the step's first kernel).
__global__ __launch_bounds__(256) void stage_in_kernel(const float4* __restrict__ h_hidden, uint32_t n4, const uint32_t* __restrict__ h_pos,
                                                        uint32_t n_pos, float4* __restrict__ hidden, uint32_t* __restrict__ pos) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < n4) hidden[i] = h_hidden[i];
    if (i < n_pos) pos[i] = h_pos[i];
}

hipError_t oxb_launch_stage_in(const float* h_hidden, uint32_t n_floats, const uint32_t* h_pos, uint32_t n_pos, float* d_hidden,
                               uint32_t* d_pos, hipStream_t st) {
    if ((n_floats & 3u) || n_floats == 0) return hipErrorInvalidValue;
    const uint32_t n4 = n_floats / 4, n = n4 > n_pos ? n4 : n_pos;
    hipLaunchKernelGGL(stage_in_kernel, dim3((n + 255) / 256), dim3(256), 0, st, reinterpret_cast<const float4*>(h_hidden), n4, h_pos, n_pos,
                       reinterpret_cast<float4*>(d_hidden), d_pos);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
hipError_t oxb_launch_kv_norm_rope_store(const OxbKvStoreParams& p, hipStream_t st) {
    if (p.kv_mode > OXB_KV_FP8_E4M3 || (p.kv_mode != OXB_KV_F16 && (!p.k_scale || !p.v_scale)) || (p.qkv_stride & 3u)) return hipErrorInvalidValue;
#define OXB_KV_STORE(HD_)                                                                                                                       \
    case HD_: {                                                                                                                                 \
        constexpr uint32_t hpw = 256 / HD_;                                                                                                     \
        const dim3 grid((uint32_t)(((uint64_t)p.M * ((p.nkv + hpw - 1) / hpw) + 3) / 4)), block(256);                                           \
        if (p.kv_mode == OXB_KV_I8) hipLaunchKernelGGL((kv_norm_rope_store_kernel<HD_, OXB_KV_I8>), grid, block, 0, st, p);                     \
        else if (p.kv_mode == OXB_KV_FP8_E4M3) hipLaunchKernelGGL((kv_norm_rope_store_kernel<HD_, OXB_KV_FP8_E4M3>), grid, block, 0, st, p);    \
        else hipLaunchKernelGGL((kv_norm_rope_store_kernel<HD_, OXB_KV_F16>), grid, block, 0, st, p);                                           \
        break;                                                                                                                                  \
    }
    switch (p.hd) {
        OXB_KV_STORE(32)
        OXB_KV_STORE(64)
        OXB_KV_STORE(128)
        OXB_KV_STORE(256)
        default: return hipErrorInvalidValue;
    }
#undef OXB_KV_STORE
    return hipGetLastError();
}

hipError_t oxb_launch_attn_decode(const OxbAttnParams& p, uint32_t batch, hipStream_t st) {
    if (p.n_splits == 0 || p.n_splits > OXB_ATTN_MAX_SPLITS || p.nq % p.nkv || p.nq / p.nkv > 16 ||
        !p.qkv || !p.q_norm || !p.k_norm || !p.cos_t || !p.sin_t || p.kv_mode > OXB_KV_FP8_E4M3 || !p.out || (p.n_splits > 1 && (!p.done || !p.part)) ||
        (p.kv_mode != OXB_KV_F16 && (!p.k_scale || !p.v_scale)) || (p.wide && (p.kv_mode == OXB_KV_F16 || p.hd > 128)) ||
        (p.kv.page_table ? (p.kv.page_shift < 4 || p.kv.page_shift > 7) : (p.kv.row_stride % 128 != 0 || p.kv.row_stride < p.max_seq)))
        return hipErrorInvalidValue;
    const dim3 grid(p.n_splits, p.nkv, batch), block(p.wide ? 512 : 256);
    const bool opt = p.window != 0 || p.kv.page_table != nullptr, pack = p.pack_out != nullptr && p.nq / p.nkv * p.hd == 512u;
    switch (p.hd) {
#define OXB_ATTN_LAUNCH_AS(HD_, KVM_, NW_, OUT_)                                                                     \
    if (opt) hipLaunchKernelGGL((attn_decode_fused_kernel<HD_, KVM_, NW_, true, OUT_>), grid, block, 0, st, p);      \
    else hipLaunchKernelGGL((attn_decode_fused_kernel<HD_, KVM_, NW_, false, OUT_>), grid, block, 0, st, p);
#define OXB_ATTN_LAUNCH(HD_, KVM_, NW_)                                                                              \
    if (p.op.xh) { OXB_ATTN_LAUNCH_AS(HD_, KVM_, NW_, OXB_ATTN_OUT_XH) }                                             \
    else if (pack) { OXB_ATTN_LAUNCH_AS(HD_, KVM_, NW_, OXB_ATTN_OUT_PACK) }                                         \
    else { OXB_ATTN_LAUNCH_AS(HD_, KVM_, NW_, OXB_ATTN_OUT_F32) }
#define OXB_ATTN_CASE(HD_)                                                                            \
    case HD_:                                                                                         \
        if (p.kv_mode == OXB_KV_F16) {                                                                \
            OXB_ATTN_LAUNCH(HD_, OXB_KV_F16, 4)                                                       \
        } else if constexpr (HD_ <= 128) { /* (eight waves of head dimension 256 exceed the LDS) */   \
            if (p.kv_mode == OXB_KV_I8) {                                                             \
                if (p.wide) { OXB_ATTN_LAUNCH(HD_, OXB_KV_I8, 8) } else { OXB_ATTN_LAUNCH(HD_, OXB_KV_I8, 4) }             \
            } else {                                                                                  \
                if (p.wide) { OXB_ATTN_LAUNCH(HD_, OXB_KV_FP8_E4M3, 8) } else { OXB_ATTN_LAUNCH(HD_, OXB_KV_FP8_E4M3, 4) } \
            }                                                                                         \
        } else if (p.kv_mode == OXB_KV_I8) {                                                          \
            OXB_ATTN_LAUNCH(HD_, OXB_KV_I8, 4)                                                        \
        } else {                                                                                      \
            OXB_ATTN_LAUNCH(HD_, OXB_KV_FP8_E4M3, 4)                                                  \
        }                                                                                             \
        break;
        OXB_ATTN_CASE(32)
        OXB_ATTN_CASE(64)
        OXB_ATTN_CASE(128)
        OXB_ATTN_CASE(256)
#undef OXB_ATTN_LAUNCH
#undef OXB_ATTN_LAUNCH_AS
#undef OXB_ATTN_CASE
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// RMSNorm of `nvec` vectors of n values (simd_float_ops.rs:204-215): out = w * x / sqrt(mean(x^2) + eps), w == nullptr
// copies x.  One workgroup per vector.  The fused paths carry their norms inside the GEMV / GEMM kernels; this one
// finishes a forward that ends at the normed hidden state (no LM head on the device).
__global__ __launch_bounds__(256) void rmsnorm_kernel(const float* __restrict__ x, const float* __restrict__ w, uint32_t n,
                                                      float eps, float* __restrict__ out) {
    __shared__ float part[4];
    const float* xv = x + (size_t)blockIdx.x * n;
    float* ov = out + (size_t)blockIdx.x * n;
    const uint32_t tid = threadIdx.x;
    if (!w) {
        for (uint32_t i = tid; i < n; i += 256) ov[i] = xv[i];
        return;
    }
    float ss = 0.f;
    for (uint32_t i = tid; i < n; i += 256) ss += xv[i] * xv[i];
    ss = wave_sum_f32(ss);
    if ((tid & 63u) == 0) part[tid >> 6] = ss;
    __syncthreads();
    const float inv_rms = 1.0f / sqrtf((part[0] + part[1] + part[2] + part[3]) / (float)n + eps);
    for (uint32_t i = tid; i < n; i += 256) ov[i] = w[i] * xv[i] * inv_rms;
}

hipError_t oxb_launch_rmsnorm(const float* d_x, const float* d_w, uint32_t n, uint32_t nvec, float eps, float* d_out, hipStream_t st) {
    if (n == 0 || nvec == 0 || !d_x || !d_out) return hipErrorInvalidValue;
    hipLaunchKernelGGL(rmsnorm_kernel, dim3(nvec), dim3(256), 0, st, d_x, d_w, n, eps, d_out);
    return hipGetLastError();
}

uint32_t oxb_argmax_parts(uint32_t n) {
    const uint32_t p = (n + 2047u) / 2048u;
    return p < 1 ? 1 : (p > OXB_ARGMAX_MAX_PARTS ? OXB_ARGMAX_MAX_PARTS : p);
}

hipError_t oxb_launch_argmax(const float* d_logits, uint32_t n, uint32_t batch, uint32_t* d_out, void* d_ws, hipStream_t st,
                             uint32_t* host_copy_or_null) {
    if (n == 0 || batch == 0 || !d_ws) return hipErrorInvalidValue;
    const uint32_t parts = oxb_argmax_parts(n), span = (n + parts - 1) / parts;
    float* pv = reinterpret_cast<float*>(d_ws);
    uint32_t* pi = reinterpret_cast<uint32_t*>(d_ws) + (size_t)batch * parts;
    hipLaunchKernelGGL(argmax_partial_kernel, dim3(parts, batch), dim3(256), 0, st, d_logits, n, span, pv, pi);
    hipLaunchKernelGGL(argmax_final_kernel, dim3(batch), dim3(64), 0, st, pv, pi, parts, d_out, host_copy_or_null);
    return hipGetLastError();
}
