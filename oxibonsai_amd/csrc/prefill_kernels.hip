// prefill_kernels.hip — causal attention of the prefill pipeline over the KV cache (fp16 or quantised rows) on the matrix cores
// (the row-wise RMSNorm of the pipeline lives in the GEMM's activation packer, SwiGLU in the gate || up GEMM's
// epilogue, gemm_kernels.hip).
//
// The reference's prefill (gpu_backend/cuda_prefill/encode_q1.rs:123-300, encode_ternary.rs:114-314) batches
// the projections but walks the tokens one by one through its decode attention kernels
// (cuda_prefill/mod.rs:36-39); here all M query tokens of a sequence attend in one launch.
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stdint.h>

#include <type_traits>

#include "device_utils.h"
#include "kv_quant_device.h"
#include "kv_row_device.h"
#include "prefill_kernels.h"

typedef _Float16 v8h __attribute__((ext_vector_type(8)));

// ---------------------------------------------------------------------------
// Causal attention of M query tokens (positions pos_start .. pos_start + M - 1) over keys 0 .. own position
// of one sequence, GQA, online softmax (semantics: block/functions.rs:78-127 -> layers/attention_fused.rs:329-400
// applied per token).  One wave = QT tiles of 16 queries of one q head.
//
// Both products run on v_mfma_f32_16x16x32_f16 in transposed form, so the score tile comes out with the
// query in the lane (column) and needs no transposition before the second product:
//   S^T[key][q]  = sum_d K[key][d] Q[q][d]      A = K rows (16 bytes per lane),
//                                               B = Q * scale * log2 e, split into fp16 hi + lo (two MFMAs: the
//                                               scores keep fp32-level accuracy)
//   O^T[d][q]   += sum_key V[key][d] P[q][key]  B = the lane's own 8 probabilities of 32 keys,
//                                               A = V gathered for exactly those 8 keys (two transposing LDS reads)
// Lane (q = lane % 16, g = lane / 16) holds keys {4g..4g+3} and {16+4g..16+4g+3} of every 32 keys, and sums their
// probabilities in fp32 as they are before the rounding to fp16 that the second product needs.  They are relative to the
// row's running maximum itself, so that the largest is exactly 1: against float64, 16 000 keys, the output is 5e-7 off where one
// key lies 12 above the rest, 4e-5 with scores of spread 3.  (Summing the rounded values on the matrix cores, relative to a
// power of two that follows the maximum at a distance, gives 2e-5 and 1.7e-4.)
//
// The four waves of a workgroup walk the same keys and values: they take `hpw` q heads of ONE kv head (4, 2 or 1,
// whatever divides the group) times 4 / hpw consecutive runs of QT query tiles.  Each block of KB keys (K and V) is
// fetched once per workgroup into LDS, double-buffered: fp16 rows go there directly (global_load_lds), quantised rows
// wait in registers and are widened on their way.  Rows are stored without padding, their 16-byte pieces permuted by an
// XOR with the row number, which keeps both kinds of read free of bank conflicts.
//
// What bounds it: the SIMDs' issue slots, where there are workgroups for the chip, and the latency of a block's chain of reads,
// products, maximum and products where there are not.  Two forms:
//  - QT = 1: one query tile per wave, 93 registers (head_dim 64) to 138 (128, one-byte rows), so three or four waves of a SIMD
//    fill each other's waits.
//  - QT = 2 (head_dim 128): two tiles share every K and V operand, which halves the LDS reads and the widening of one-byte rows
//    per product, and 64-key blocks halve the maxima.  That takes the registers of two waves per SIMD and the LDS of a CU: the
//    eight waves are two walkers, four waves each, that take the blocks in turn and add their sums in LDS at the end.
// In both the scores start from -m (the products' C operand), so a block without a new maximum for any query of a tile costs no
// rescaling, and the visibility tests run only in blocks that some query of the wave sees in part.
// us per layer, 32 q heads and 8 kv heads of 128, merge included, one form for all (two tiles, four waves) -> these two:
// fp16 rows, 100 tokens 12.6 -> 9.6, 300 18.7 -> 15.8, 1000 43.8 -> 34.0, 2048 88 -> 73, 32 behind 6000 31.9 -> 26.8; INT8 rows,
// 300 behind 6000 93 -> 81, 2048 behind 6000 459 -> 426.  Heads of 64: 1400 behind 4000 161 -> 112.
//
// Options as in the decode attention: quantised cache rows (template KVM; the codes are widened to exact fp16
// numbers on their way into LDS, V already multiplied by its row scale there, the K row scale multiplies the
// score) and a sliding window with attention sinks (key visible to the query at qpos iff key < sinks or
// qpos - key < window - sinks; blocks no query of the workgroup can see are skipped).
//
// Few queries behind a long cache leave most of the chip idle when a workgroup walks all keys: then blockIdx.y splits the
// walk into runs of p.blocks_per_split blocks, each run leaves its un-normalised sums in p.part, and
// attn_prefill_merge_kernel adds them in order.
// ---------------------------------------------------------------------------
// The upper half of the wave's `a` and the lower half of its `b` change places.
__device__ __forceinline__ void swap_upper_lower(float& a, float& b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]), b = __uint_as_float(r[1]);
}

// p.part: maximum and sum of every (run, query, head), then from a 16-byte boundary on their outputs.
__host__ __device__ constexpr size_t pf_part_head(size_t n_splits, size_t rows) { return (n_splits * rows * 2 + 3) & ~(size_t)3; }

// Keys per block: 64, or 32 where four (head_dim 128) or two (256) workgroups to a CU share its LDS, 4 x KB x 2 HD bytes each.
constexpr int pf_block_keys(int hd, int qt) { return hd == 256 || (hd == 128 && qt == 1) ? 32 : 64; }

// OPT: a window and / or a paged cache may be in use (else neither costs anything).
// NEW: a prompt's first tokens, one block of keys: the cache holds none of them yet.  Every workgroup works its kv head's rows out from
// the projection, keeps them in LDS as the cache will hold them, and one workgroup of each kv head stores them.
template <int HD, int KVM, bool OPT, int QT, bool NEW>
__global__ __launch_bounds__(256 * QT, HD == 256 ? 1 : 2) void attn_prefill_kernel(OxbPrefillAttnParams p, uint32_t hpw) {
    constexpr bool QC = KVM != OXB_KV_F16;
    constexpr int WK = QT;                                           // walkers: groups of four waves that take the keys' blocks in turn
    constexpr int KS = HD / 32, NS = HD / 16, KB = pf_block_keys(HD, QT);
    constexpr int RPW = KB / 4;                                      // rows of a block that a wave fetches
    constexpr int PPR = HD / 8;                                      // 16-byte pieces of an LDS row
    constexpr int RB = PPR >= 16 ? 1 : 16 / PPR, PM = (PPR < 16 ? PPR : 16) - 1;  // rows per 256 bytes; mask of the permutation
    constexpr int NI = QC ? (RPW * HD / 16 + 63) / 64 : RPW * PPR / 64;  // 16-byte pieces per lane and block, of K and of V
    __shared__ __attribute__((aligned(16))) _Float16 ks0_all[WK * KB * HD], ks1_all[WK * KB * HD], vs0_all[WK * KB * HD], vs1_all[WK * KB * HD];
    __shared__ __attribute__((aligned(16))) float kscale0_all[WK * KB], kscale1_all[WK * KB];  // K row scales of the block (quantised cache)
    const uint32_t tid = threadIdx.x, lane = tid & 63u, qi = lane & 15u, g = lane >> 4;
    const uint32_t wave8 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6)), wave = wave8 & 3u, walker = WK == 1 ? 0u : wave8 >> 2;
    _Float16 *const ks0 = ks0_all + walker * (KB * HD), *const ks1 = ks1_all + walker * (KB * HD);
    _Float16 *const vs0 = vs0_all + walker * (KB * HD), *const vs1 = vs1_all + walker * (KB * HD);
    float *const kscale0 = kscale0_all + walker * KB, *const kscale1 = kscale1_all + walker * KB;
    const uint32_t tpw = 4u / hpw, n_qt = (p.M + 15u) / 16u, per_wg = tpw * QT, n_tg = (n_qt + per_wg - 1) / per_wg, hq = p.nq / hpw;
    // Late query tiles walk more keys than early ones.  With two walkers a CU holds one workgroup, and takes the next one when it
    // is done: the longest walks go first.  Else workgroups are handed out in order, one to a CU, then a second one to each, and
    // so on: the first half of the tiles goes from the latest down, the second half from the earliest up, so that the longest
    // walk shares its CU with the shortest.
    const uint32_t tb = blockIdx.x / hq, tg = WK == 2 || 2 * tb < n_tg ? n_tg - 1 - tb : tb - (n_tg + 1) / 2;
    const uint32_t head = (blockIdx.x % hq) * hpw + wave % hpw;
    const uint32_t kvh = head / (p.nq / p.nkv);                           // the same for the four waves
    const uint32_t t_first = (tg * per_wg + (wave / hpw) * QT) * 16;      // first query of this wave
    const uint32_t kv_len = p.pos_start + min((tg + 1) * per_wg * 16, p.M);  // keys the workgroup's last query sees
    const uint32_t last = kv_len - 1;
    uint32_t t_q[QT], qpos[QT];
#pragma unroll
    for (int t = 0; t < QT; t++) {
        t_q[t] = min(t_first + t * 16 + qi, p.M - 1);                     // rows past M repeat the last one and are not stored
        qpos[t] = p.pos_start + t_q[t];
    }
    const uint32_t q_lo = p.pos_start + min(t_first, p.M - 1), q_hi = p.pos_start + min(t_first + QT * 16 - 1, p.M - 1);
    const bool paged = OPT && p.kv.page_table != nullptr;
    const uint32_t window = OPT ? p.window : 0u;
    const size_t row0 = paged ? 0 : kv_row(p.kv, p.seq, p.layer, kvh, 0);
    // sliding window: a query sees [0, sinks) and (qpos - budget, qpos]; the workgroup's earliest query sits at
    // q_first, so no query of it sees a key in [sinks, q_first + 1 - budget): whole blocks in there are left out of the walk
    const uint32_t budget = window > p.sinks ? window - p.sinks : 0u;
    const uint32_t q_first = p.pos_start + tg * per_wg * 16;
    const uint32_t sink_blocks = window ? (p.sinks + KB - 1) / KB : 0u;
    const uint32_t seen_from = window && q_first + 1 > budget ? (q_first + 1 - budget) / KB : 0u;
    const uint32_t gap = seen_from > sink_blocks ? seen_from - sink_blocks : 0u;  // blocks left out behind the sinks
    auto key_of = [&](uint32_t i) -> uint32_t { return (gap && i >= sink_blocks ? i + gap : i) * KB; };
    const uint32_t n_blk = (last / KB + 1) - min(gap, last / KB + 1);
    const uint32_t i0 = min(blockIdx.y * p.blocks_per_split, n_blk), i1 = blockIdx.y + 1 == gridDim.y ? n_blk : min(i0 + p.blocks_per_split, n_blk);

    // ---- fetching: wave w takes rows w * RPW .. of a block; they lie in one page, so the base is uniform.  Rows past the
    // last key repeat it (their scores are masked, their probabilities 0).
    const uint8_t* const Kc = reinterpret_cast<const uint8_t*>(p.k_cache);
    const uint8_t* const Vc = reinterpret_cast<const uint8_t*>(p.v_cache);
    constexpr uint32_t ROWB = HD * (QC ? 1 : 2), SPR = ROWB / 16;  // bytes and 16-byte pieces of a cache row
    // (worked out again for every block from an opaque copy of the lane: kept, they would cost the registers of a wave)
    auto piece_of = [&](uint32_t l, int i, uint32_t& row, uint32_t& off) {
        const uint32_t id = i * 64 + l;
        row = id / SPR;
        off = QC ? (id % SPR) * 16u : ((id % SPR) ^ (((wave * RPW + row) / RB) & PM)) * 16u;
    };
    const bool f_on = RPW * HD / 16 >= 64 || !QC || lane < RPW * HD / 16;  // (hd 32, quantised: half a wave holds all pieces)
    auto group = [&](uint32_t key0, uint32_t& lim) -> size_t {
        const uint32_t g0 = min(key0 + wave * RPW, last & ~(uint32_t)(RPW - 1));
        lim = min((uint32_t)RPW - 1, last - g0);
        return paged ? kv_row(p.kv, p.seq, p.layer, kvh, g0) : row0 + g0;
    };
    v4i kreg[QC ? NI : 1], vreg[QC ? NI : 1];
    float vsreg[QC ? NI : 1], ksreg = 0.f;
    auto request = [&](uint32_t key0, _Float16* kd, _Float16* vd) {
        uint32_t lim;
        const size_t row = group(key0, lim);
        const uint8_t *kb = Kc + row * ROWB, *vb = Vc + row * ROWB;
        uint32_t l = lane;
        asm volatile("" : "+v"(l));
#pragma unroll
        for (int i = 0; i < NI; i++) {
            uint32_t f_row, f_off;
            piece_of(l, i, f_row, f_off);
            const uint32_t off = min(f_row, lim) * ROWB + f_off;
            if constexpr (QC) {
                if (f_on) {
                    kreg[i] = *reinterpret_cast<const v4i*>(kb + off);
                    vreg[i] = *reinterpret_cast<const v4i*>(vb + off);
                    vsreg[i] = p.v_scale[row + min(f_row, lim)];
                }
            } else {
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(kb + off),
                                                 (__attribute__((address_space(3))) void*)(kd + (wave * RPW * PPR + i * 64) * 8), 16, 0, 0);
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(vb + off),
                                                 (__attribute__((address_space(3))) void*)(vd + (wave * RPW * PPR + i * 64) * 8), 16, 0, 0);
            }
        }
        if constexpr (QC) ksreg = p.k_scale[row + min(lane & (RPW - 1), lim)];
    };
    auto deliver = [&](_Float16* kd, _Float16* vd, float* scd, bool there) {
        if (QC && there) {
            uint32_t l = lane;
            asm volatile("" : "+v"(l));
#pragma unroll
            for (int i = 0; i < NI; i++) {
                if (!f_on) continue;
                uint32_t f_row, f_off;
                piece_of(l, i, f_row, f_off);
                uint32_t kw[8], vw[8];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    kv_dec4<KVM>((uint32_t)kreg[i][e], kw[2 * e], kw[2 * e + 1]);
                    kv_dec4<KVM>((uint32_t)vreg[i][e], vw[2 * e], vw[2 * e + 1]);
                }
                // V leaves for LDS as code * scale in fp16 (the probabilities it meets are fp16 as well)
                const _Float16 sc = (_Float16)vsreg[i];
                const kvh2_t sc2 = {sc, sc};
#pragma unroll
                for (int e = 0; e < 8; e++) vw[e] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(kvh2_t, vw[e]) * sc2);
                const uint32_t row = wave * RPW + f_row, x = (row / RB) & PM, c = f_off / 8u;  // the piece becomes LDS pieces c, c + 1
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    const uint32_t at = (row * PPR + ((c + e) ^ x)) * 8;
                    *reinterpret_cast<v4i*>(kd + at) = (v4i){(int)kw[4 * e], (int)kw[4 * e + 1], (int)kw[4 * e + 2], (int)kw[4 * e + 3]};
                    *reinterpret_cast<v4i*>(vd + at) = (v4i){(int)vw[4 * e], (int)vw[4 * e + 1], (int)vw[4 * e + 2], (int)vw[4 * e + 3]};
                }
            }
            if (lane < RPW) scd[wave * RPW + lane] = ksreg;
        }
        // the barrier that ends a block: every wave has read it, and the next one is complete in LDS
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    };
    const uint32_t steps = i0 < i1 ? (i1 - i0 + WK - 1) / WK : 0u;  // the same for both walkers: they meet at every barrier
    auto mine = [&](uint32_t j) -> uint32_t { return i0 + j * WK + walker; };
    if (!NEW && mine(0) < i1) request(key_of(mine(0)), ks0, vs0);
    if constexpr (NEW) {
        constexpr int L = HD / 4, RPI = 64 / L, IT = RPW / RPI;  // lanes of a row, rows of a wave at a time
        const uint32_t j = lane % L;
        const float4 w = *reinterpret_cast<const float4*>(p.k_norm + 4 * j);
        KvRowIn in[IT];
#pragma unroll
        for (int it = 0; it < IT; it++) {
            const uint32_t t = min(wave * RPW + it * RPI + lane / L, last);  // (rows past the last one repeat it)
            in[it] = kv_row_load<HD>(p.qkv + (size_t)t * p.qkv_stride, p.nq, p.nkv, kvh, j, p.cos_t, p.sin_t, t);
        }
        const bool stores = blockIdx.x < hq && blockIdx.x * hpw % (p.nq / p.nkv) == 0;
#pragma unroll
        for (int it = 0; it < IT; it++) {
            const uint32_t t = wave * RPW + it * RPI + lane / L;
            const KvRowOut r = kv_row_make<HD, KVM>(in[it], w, p.eps, j);
            if (stores && t < p.M) kv_row_store<HD, KVM>(r, const_cast<void*>(p.k_cache), const_cast<void*>(p.v_cache), const_cast<float*>(p.k_scale), const_cast<float*>(p.v_scale), kv_row(p.kv, p.seq, p.layer, kvh, t), j);
            uint2 kw = r.k, vw = r.v;
            if constexpr (QC) {  // as deliver() widens them
                kv_dec4<KVM>(r.k.x, kw.x, kw.y);
                kv_dec4<KVM>(r.v.x, vw.x, vw.y);
                const _Float16 sc = (_Float16)r.vs;
                const kvh2_t sc2 = {sc, sc};
                vw.x = __builtin_bit_cast(uint32_t, __builtin_bit_cast(kvh2_t, vw.x) * sc2);
                vw.y = __builtin_bit_cast(uint32_t, __builtin_bit_cast(kvh2_t, vw.y) * sc2);
                if (j == 0) kscale0[t] = r.ks;
            }
            const uint32_t at = (t * PPR + ((j >> 1) ^ ((t / RB) & PM))) * 8 + (j & 1u) * 4;
            *reinterpret_cast<uint2*>(ks0 + at) = kw;
            *reinterpret_cast<uint2*>(vs0 + at) = vw;
        }
    }

    // Q of this lane's queries: per-head RMSNorm, RoPE on the pairs (d, d + hd/2), times log2(e)/sqrt(hd)
    // (fused_qk_norm_rope, gpu_backend/cuda_attn_kernels.rs:160-226), then split into fp16 hi + lo.  The lane holds
    // elements 32 s + 8 g + e; for hd >= 64 both elements of a pair are its own (steps s and s + KS / 2), for hd = 32
    // the partner sits in lane g ^ 2.
    v8h qh[QT][KS], ql[QT][KS];
#pragma unroll
    for (int t = 0; t < QT; t++) {
        constexpr int half = HD / 2;
        const float* qr = p.qkv + (size_t)t_q[t] * p.qkv_stride + (size_t)head * HD + 8 * g;
        float x[KS][8], ss = 0.f;
#pragma unroll
        for (int s = 0; s < KS; s++) {
            const float4 a = *reinterpret_cast<const float4*>(qr + 32 * s), b = *reinterpret_cast<const float4*>(qr + 32 * s + 4);
            const float f[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
            for (int e = 0; e < 8; e++) {
                x[s][e] = f[e];
                ss = fmaf(f[e], f[e], ss);
            }
        }
        ss = sum_rows4(ss);
        const float inv = 1.0f / sqrtf(ss / (float)HD + p.eps);
#pragma unroll
        for (int s = 0; s < KS; s++)
#pragma unroll
            for (int e = 0; e < 8; e++) x[s][e] = p.q_norm[32 * s + 8 * g + e] * x[s][e] * inv;
        const float* cs = p.cos_t + (size_t)qpos[t] * half;
        const float* sn = p.sin_t + (size_t)qpos[t] * half;
        float r[KS][8];
        if constexpr (KS >= 2) {
#pragma unroll
            for (int s = 0; s < KS / 2; s++)
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const int d = 32 * s + 8 * (int)g + e;  // < half
                    const float lo = x[s][e], hi = x[s + KS / 2][e], c = cs[d], sv = sn[d];
                    r[s][e] = lo * c - hi * sv;
                    r[s + KS / 2][e] = lo * sv + hi * c;
                }
        } else {  // hd = 32: lanes g = 0, 1 hold the first half, g = 2, 3 the second
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float mine = x[0][e], other = __shfl_xor(mine, 32, 64);
                const int d = 8 * (int)(g & 1u) + e;
                const float c = cs[d], sv = sn[d];
                r[0][e] = g < 2 ? mine * c - other * sv : other * sv + mine * c;
            }
        }
        const float mul = p.scale * 1.44269504088896340736f;
#pragma unroll
        for (int s = 0; s < KS; s++)
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float v = r[s][e] * mul;
                const _Float16 hi = (_Float16)v;
                qh[t][s][e] = hi;
                ql[t][s][e] = (_Float16)(v - (float)hi);
            }
    }
    // reading: offset (in halves) of the K operand of step 0 in key tile 0 and of the V tile of dimensions 0..15 in keys
    // 0..15.  Step s and dimension tile sl are an XOR with a constant away (32 s, 16 sl), the other key tiles whole multiples
    // of 16 rows, where the permutation is the same.
    const uint32_t k_at = (qi * PPR + (g ^ ((qi / RB) & PM))) * 8;
    const uint32_t v_row = 4 * g + (qi >> 2), v_at = (v_row * PPR + (((qi >> 1) & 1u) ^ ((v_row / RB) & PM))) * 8 + (qi & 1u) * 4;
    v4f O[QT][NS];
    // The running maximum m of the tile's queries: -m, which the scores start from (fp16 rows: the score products' C operand;
    // quantised ones: the addend of the row scale), and `seen`, 0 once there is one and -infinity before.  This lane's share
    // of the sum of the probabilities.
    v4f neg_m[QT];
    float seen[QT], lsum[QT];
#pragma unroll
    for (int t = 0; t < QT; t++) {
#pragma unroll
        for (int i = 0; i < NS; i++) O[t][i] = (v4f){0.f, 0.f, 0.f, 0.f};
        neg_m[t] = (v4f){0.f, 0.f, 0.f, 0.f};
        lsum[t] = 0.f;
        seen[t] = -INFINITY;
    }
    // The larger of two as the median with an infinity that the compiler does not know (it would make the median a maximum and
    // quiet every operand that comes from a matrix instruction or a lane swap first, an instruction each).
    float inf;
    asm volatile("s_mov_b32 %0, 0x7f800000" : "=s"(inf));
    auto max2 = [&](float a, float b) -> float { return __builtin_amdgcn_fmed3f(a, b, inf); };
    auto max_rows = [&](float v) -> float {
        const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        v = max2(__uint_as_float(a[0]), __uint_as_float(a[1]));
        const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        return max2(__uint_as_float(b[0]), __uint_as_float(b[1]));
    };
    auto block = [&](const _Float16* kb, const _Float16* vb, const float* ksc, uint32_t blk_key0) {
        uint32_t ka = k_at, va = v_at;
        asm volatile("" : "+v"(ka), "+v"(va));  // (the XORs below stay in the loop: their results would cost 12 registers)
        constexpr int NH = KB / 32, NT = KB / 16, NP = NH * NS;  // 32-key steps, key tiles, V operands of a block
        constexpr int VB = QC && QT == 2 && NS >= 4 ? 2 : NP < 4 ? NP : 4;  // V operands read ahead (rows waiting in registers leave room for fewer)
        // (where rows wait in registers there is no room to hold the requests' order: the compiler's own has no spills)
        constexpr bool FENCE = !QC || QT == 1;
        auto fence = [&]() {
            if constexpr (FENCE) __builtin_amdgcn_sched_barrier(0);
        };
        v8h K[2][KS];
        auto read_k = [&](int hb, int s) {
#pragma unroll
            for (int kt = 0; kt < 2; kt++) K[kt][s] = *reinterpret_cast<const v8h*>(kb + (ka ^ (32u * s)) + (2 * hb + kt) * 16 * HD);
        };
        v8h V[2][VB];
        auto read_v = [&](int j) {  // the j-th group of V operands: step i / NS, dimensions 16 (i % NS) ..
#pragma unroll
            for (int u = 0; u < VB; u++) {
                const int i = j * VB + u;
                const _Float16* tile = vb + (va ^ (16u * (i % NS))) + (i / NS) * 32 * HD;
                const v4h_t t0 = lds_read_tr16(tile), t1 = lds_read_tr16(tile + 16 * HD);
                V[j & 1][u] = (v8h){t0[0], t0[1], t0[2], t0[3], t1[0], t1[1], t1[2], t1[3]};
            }
        };
#pragma unroll
        for (int s = 0; s < KS; s++) read_k(0, s);
        fence();  // all K operands have been requested: their latency is paid once
        v4f S[QT][NT];
#pragma unroll
        for (int t = 0; t < QT; t++)
#pragma unroll
            for (int kt = 0; kt < NT; kt++) S[t][kt] = QC ? (v4f){0.f, 0.f, 0.f, 0.f} : neg_m[t];
        // four independent chains of products at a time; a K operand is read again for the next step right after its last use
#pragma unroll
        for (int hb = 0; hb < NH; hb++)
#pragma unroll
            for (int s = 0; s < KS; s++) {
#pragma unroll
                for (int hl = 0; hl < 2; hl++)
#pragma unroll
                    for (int kt = 0; kt < 2; kt++)
#pragma unroll
                        for (int t = 0; t < QT; t++)
                            S[t][2 * hb + kt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(K[kt][s], hl ? ql[t][s] : qh[t][s], S[t][2 * hb + kt], 0, 0, 0);
                if (hb + 1 < NH) {
                    read_k(hb + 1, s);
                    fence();
                }
            }
        read_v(0);  // the first V operands travel while the probabilities are worked out
        fence();
        if constexpr (QC) {
#pragma unroll
            for (int kt = 0; kt < NT; kt++) {
                const float4 a = *reinterpret_cast<const float4*>(ksc + 16 * kt + 4 * g);
#pragma unroll
                for (int t = 0; t < QT; t++) {
                    S[t][kt][0] = fmaf(S[t][kt][0], a.x, neg_m[t][0]), S[t][kt][1] = fmaf(S[t][kt][1], a.y, neg_m[t][0]);
                    S[t][kt][2] = fmaf(S[t][kt][2], a.z, neg_m[t][0]), S[t][kt][3] = fmaf(S[t][kt][3], a.w, neg_m[t][0]);
                }
            }
        }
        // (wave-uniform) every query of the wave sees all of these keys, or the tests run
        const bool all = blk_key0 + KB - 1 <= q_lo && (!window || blk_key0 + KB <= p.sinks || q_hi - blk_key0 < budget);
        if (!all) {
#pragma unroll
            for (int t = 0; t < QT; t++)
#pragma unroll
                for (int kt = 0; kt < NT; kt++)
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        const uint32_t key = blk_key0 + 16 * kt + 4 * g + v;
                        const bool vis = key <= qpos[t] && (!window || key < p.sinks || qpos[t] - key < budget);
                        S[t][kt][v] = vis ? S[t][kt][v] : -INFINITY;
                    }
        }
        v8h P[QT][NH];
#pragma unroll
        for (int t = 0; t < QT; t++) {
            float mk[NT];
#pragma unroll
            for (int kt = 0; kt < NT; kt++) mk[kt] = max2(max2(S[t][kt][0], S[t][kt][1]), max2(S[t][kt][2], S[t][kt][3]));
            float mx = max2(mk[0], mk[1]);
#pragma unroll
            for (int kt = 2; kt < NT; kt += 2) mx = max2(mx, max2(mk[kt], mk[kt + 1]));
            mx = max_rows(mx);
            if (__builtin_amdgcn_ballot_w64(mx > seen[t])) {  // a new maximum for some query of the tile
                // by how much it moves; the first one of a query may lie below 0, and finds nothing to rescale
                const float by = mx > seen[t] ? mx : 0.f, alpha = __builtin_amdgcn_exp2f(fminf(-by, 0.f));
                seen[t] = mx > seen[t] ? 0.f : seen[t];
                neg_m[t][0] -= by;
                if constexpr (!QC) neg_m[t][1] = neg_m[t][2] = neg_m[t][3] = neg_m[t][0];
#pragma unroll
                for (int sl = 0; sl < NS; sl++)
#pragma unroll
                    for (int v = 0; v < 4; v++) O[t][sl][v] *= alpha;
                lsum[t] *= alpha;
#pragma unroll
                for (int kt = 0; kt < NT; kt++)
#pragma unroll
                    for (int v = 0; v < 4; v++) S[t][kt][v] -= by;
            }
            // (a query that has seen nothing yet keeps its empty state: every score -infinity, every probability 0)
#pragma unroll
            for (int hb = 0; hb < NH; hb++) {
                float pe[8];
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    pe[e] = __builtin_amdgcn_exp2f(S[t][2 * hb + (e >> 2)][e & 3]);
                    P[t][hb][e] = (_Float16)pe[e];
                }
                lsum[t] += ((pe[0] + pe[1]) + (pe[2] + pe[3])) + ((pe[4] + pe[5]) + (pe[6] + pe[7]));
            }
        }
#pragma unroll
        for (int j = 0; j < NP / VB; j++) {
            if (j + 1 < NP / VB) read_v(j + 1);
            fence();
#pragma unroll
            for (int u = 0; u < VB; u++)
#pragma unroll
                for (int t = 0; t < QT; t++) {
                    const int i = j * VB + u;
                    O[t][i % NS] = __builtin_amdgcn_mfma_f32_16x16x32_f16(V[j & 1][u], P[t][i / NS], O[t][i % NS], 0, 0, 0);
                }
        }
    };
    if constexpr (NEW) {
        lds_barrier();
        block(ks0, vs0, kscale0, 0);
    } else if (steps) {
        deliver(ks0, vs0, kscale0, mine(0) < i1);
        for (uint32_t j = 0;;) {
            if (mine(j + 1) < i1) request(key_of(mine(j + 1)), ks1, vs1);
            if (mine(j) < i1) block(ks0, vs0, kscale0, key_of(mine(j)));
            if (++j == steps) break;
            deliver(ks1, vs1, kscale1, mine(j) < i1);
            if (mine(j + 1) < i1) request(key_of(mine(j + 1)), ks0, vs0);
            if (mine(j) < i1) block(ks1, vs1, kscale1, key_of(mine(j)));
            if (++j == steps) break;
            deliver(ks0, vs0, kscale0, mine(j) < i1);
        }
    }
    if constexpr (WK == 2) {
        // The second walker's sums go through the stages (nothing is in flight: the last block's requests were waited for), the
        // first one brings both to a common reference.
        __shared__ float2 ex_ml[4][QT][64];
        constexpr int PER = (int)sizeof(ks0_all) / 4096;  // dimension tiles of four waves that a stage holds
        static_assert(4 * PER >= QT * NS, "the sums fit the four stages");
        _Float16* const stages[4] = {ks0_all, ks1_all, vs0_all, vs1_all};
        __syncthreads();
        if (walker) {
#pragma unroll
            for (int t = 0; t < QT; t++) {
                ex_ml[wave][t][lane] = make_float2(seen[t] - neg_m[t][0], lsum[t]);
#pragma unroll
                for (int sl = 0; sl < NS; sl++)
                    reinterpret_cast<v4f*>(stages[(t * NS + sl) / PER])[(wave * PER + (t * NS + sl) % PER) * 64 + lane] = O[t][sl];
            }
        }
        __syncthreads();
        if (walker) return;
#pragma unroll
        for (int t = 0; t < QT; t++) {
            const float2 ml = ex_ml[wave][t][lane];
            const float m0 = seen[t] - neg_m[t][0], m = fmaxf(m0, ml.x);
            const float a0 = m0 == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m0 - m), a1 = ml.x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ml.x - m);
            seen[t] = m == -INFINITY ? m : 0.f;
            neg_m[t][0] = m == -INFINITY ? 0.f : -m;
            lsum[t] = lsum[t] * a0 + ml.y * a1;
#pragma unroll
            for (int sl = 0; sl < NS; sl++) {
                const v4f o = reinterpret_cast<v4f*>(stages[(t * NS + sl) / PER])[(wave * PER + (t * NS + sl) % PER) * 64 + lane];
#pragma unroll
                for (int v = 0; v < 4; v++) O[t][sl][v] = O[t][sl][v] * a0 + o[v] * a1;
            }
        }
    }
#pragma unroll
    for (int t = 0; t < QT; t++) {
        const uint32_t tok = t_first + t * 16 + qi;
        const float l = sum_rows4(lsum[t]);
        if (tok >= p.M) continue;
        if (gridDim.y == 1) {
            const float inv = l > 0.f ? 1.0f / l : 0.f;
            auto four = [&](int sl) -> float4 { return make_float4(O[t][sl][0] * inv, O[t][sl][1] * inv, O[t][sl][2] * inv, O[t][sl][3] * inv); };
            float* o = p.out + ((size_t)tok * p.nq + head) * HD + 4 * g;
#pragma unroll
            for (int sl = 0; sl < NS; sl += 2) {
                float4 a = four(sl), b = four(sl + 1);
                const uint32_t k = head * HD + 16 * sl;
                if (!p.op.xh) {
                    *reinterpret_cast<float4*>(o + 16 * sl) = a;
                    *reinterpret_cast<float4*>(o + 16 * sl + 16) = b;
                } else if (p.op.fmt == OXB_FMT_Q1) {
                    operand_store8(p.op, k + 4 * g, tok, a, b);
                } else {
                    // a piece holds rows 4 (g % 2) .. of one tile of 16 and those 8 further, in lanes g and g + 2: the lower lane
                    // takes the piece of the first tile, the upper one that of the second
                    swap_upper_lower(a.x, b.x), swap_upper_lower(a.y, b.y), swap_upper_lower(a.z, b.z), swap_upper_lower(a.w, b.w);
                    operand_store8(p.op, k + 16 * (g >> 1) + 4 * (g & 1u), tok, a, b);
                }
            }
        } else {
            const size_t at = ((size_t)blockIdx.y * p.M + tok) * p.nq + head;
            if (g == 0) reinterpret_cast<float2*>(p.part)[at] = make_float2(seen[t] - neg_m[t][0], l);
            if (!(l == 0.f)) {  // (an empty run is left out of the merge)
                float* o = p.part + pf_part_head(gridDim.y, (size_t)p.M * p.nq) + at * HD + 4 * g;
#pragma unroll
                for (int sl = 0; sl < NS; sl++)
                    *reinterpret_cast<float4*>(o + 16 * sl) = make_float4(O[t][sl][0], O[t][sl][1], O[t][sl][2], O[t][sl][3]);
            }
        }
    }
}

// out[t][head] = the runs' sums brought to a common exponent, added in order, over the total of their probabilities.
// A workgroup owns four tokens of 256 / hd heads, a thread four dimensions; as the O projection's operand the outputs change
// places in LDS and leave in runs of four tokens.  (Reading in the operand's order instead, two times sixteen bytes 64 bytes
// apart, takes 12 us where this takes 9: 301 tokens, six runs, 30 MB.)
__global__ __launch_bounds__(256) void attn_prefill_merge_kernel(const float* __restrict__ part, uint32_t n_splits, uint32_t M, uint32_t nq,
                                                                  uint32_t hd, float* __restrict__ out, const OxbOperandOut op) {
    __shared__ __attribute__((aligned(16))) float o[1024];
    const uint32_t tid = threadIdx.x, hd4 = hd / 4, c = tid % hd4, r = tid / hd4, hpg = 256 / hd;
    const uint32_t tok = blockIdx.x * 4 + (r & 3u), head = blockIdx.y * hpg + (r >> 2);
    const bool live = tok < M && head < nq;
    const uint32_t rows = M * nq, row = live ? tok * nq + head : 0u;
    const float2* ml = reinterpret_cast<const float2*>(part);
    const float4* po = reinterpret_cast<const float4*>(part + pf_part_head(n_splits, rows));
    // (what eight runs hold is requested together; 32 runs one after the other took 14 us, 16 this way take 8: 32 tokens)
    float m = -INFINITY;
    for (uint32_t s0 = 0; s0 < n_splits; s0 += 8) {
        float2 v[8];
#pragma unroll
        for (uint32_t u = 0; u < 8; u++) v[u] = s0 + u < n_splits ? ml[(size_t)(s0 + u) * rows + row] : make_float2(0.f, 0.f);
#pragma unroll
        for (uint32_t u = 0; u < 8; u++) m = v[u].y == 0.f ? m : fmaxf(m, v[u].x);
    }
    float l = 0.f;
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
    for (uint32_t s0 = 0; s0 < n_splits; s0 += 8) {
        float2 v[8];
        float4 q[8];
#pragma unroll
        for (uint32_t u = 0; u < 8; u++) {
            const bool there = s0 + u < n_splits;
            v[u] = there ? ml[(size_t)(s0 + u) * rows + row] : make_float2(0.f, 0.f);
            q[u] = there ? po[((size_t)(s0 + u) * rows + row) * hd4 + c] : make_float4(0.f, 0.f, 0.f, 0.f);
        }
#pragma unroll
        for (uint32_t u = 0; u < 8; u++) {
            if (v[u].y == 0.f) continue;  // (an empty run has left no outputs)
            const float w = __builtin_amdgcn_exp2f(v[u].x - m);
            l = fmaf(v[u].y, w, l);
            a.x = fmaf(q[u].x, w, a.x), a.y = fmaf(q[u].y, w, a.y), a.z = fmaf(q[u].z, w, a.z), a.w = fmaf(q[u].w, w, a.w);
        }
    }
    const float inv = l > 0.f ? 1.0f / l : 0.f;
    a = make_float4(a.x * inv, a.y * inv, a.z * inv, a.w * inv);
    if (!op.xh) {
        if (live) reinterpret_cast<float4*>(out)[(size_t)row * hd4 + c] = a;
        return;
    }
    reinterpret_cast<float4*>(o)[tid] = a;
    __syncthreads();
    if (tid >= 128) return;
    // piece i >> 2 of the heads' values for token i % 4
    const uint32_t t = blockIdx.x * 4 + (tid & 3u), i = tid >> 2, hl = i / (hd / 8), e = i % (hd / 8), h = blockIdx.y * hpg + hl;
    if (t >= M || h >= nq) return;
    const uint32_t d = 32 * (e >> 2) + (op.fmt == OXB_FMT_Q1 ? 4 * (e & 3u) : 16 * ((e >> 1) & 1u) + 4 * (e & 1u));
    const float* q = o + (hl * 4 + (tid & 3u)) * hd + d;
    operand_store8(op, h * hd + d, t, *reinterpret_cast<const float4*>(q), *reinterpret_cast<const float4*>(q + OXB_OPERAND_STEP(op.fmt)));
}

// Which of the two forms, and into how many runs the keys are split: the cheapest of all, in us.  Measured with 1 to 2048
// queries behind up to 8000 keys, every form alone, and what the rule makes of them is within 4 % of the better form there:
//  - one tile: 7 us (launch, Q, the first keys' way), then per 32 keys of head_dim 128 with k workgroups on the CU 0.84, 0.98,
//    1.29, 1.72 us (fp16 rows; four fit), 0.93, 1.31, 1.69 us (one-byte rows; three fit).  Heads of 64 take 0.55 of it.
//    No CU is done before its longest walk, nor before its share of all walks, counted in whole rounds.
//  - two tiles, two walkers: 14 us, and 0.64 to 0.78 us (one-byte rows 0.75 to 0.93) per 32 keys, the more the more CUs work;
//    one workgroup to a CU.  So it takes long walks by less than a chip full of workgroups, and one-byte rows.
//  - head_dim 256: 2 us per 32 keys, one workgroup to a CU.
//  - a split adds the merge, 4 us and 0.25 per run, and the partial sums' way to memory and back, 0.4 us per MB.
static OxbPrefillAttnPlan plan_attn(const OxbPrefillAttnParams& p, uint32_t n_cus) {
    const uint32_t G = p.nq / p.nkv, hpw = G % 4u == 0 ? 4u : (G % 2u == 0 ? 2u : 1u);
    const bool qc = p.kv_mode != OXB_KV_F16;
    OxbPrefillAttnPlan best = {hpw, 1, 0, 1, 0};
    float best_cost = INFINITY;
    for (uint32_t qt = 1; qt <= (p.hd == 128 ? 2u : 1u); qt++) {
        const uint32_t per_wg = (4u / hpw) * qt, KB = (uint32_t)pf_block_keys((int)p.hd, (int)qt);
        const uint32_t n_tg = ((p.M + 15u) / 16u + per_wg - 1) / per_wg, wgs = n_tg * (p.nq / hpw);
        // keys that the last workgroup walks, and that one walks on average
        uint32_t keys = p.pos_start + p.M;
        float mean = (float)p.pos_start + 0.5f * (float)(p.M + 16 * per_wg);
        if (p.window) {  // sinks, window and the workgroup's own queries
            const uint64_t seen = (uint64_t)p.sinks + p.window + per_wg * 16 + 2 * KB;
            if (seen < keys) keys = (uint32_t)seen;
        }
        mean = fminf(mean, (float)keys);
        const uint32_t n_blk = (keys + KB - 1) / KB + (p.window ? 1 : 0);
        const float part_mb = 1e-6f * (float)p.M * p.nq * p.hd * 4.0f, size = 0.1f + 0.9f * (float)p.hd / 128.0f;
        for (uint32_t s = 1; s <= OXB_PF_ATTN_MAX_SPLITS && s <= n_blk; s++) {
            const uint32_t bps = (n_blk + s - 1) / s, used = (n_blk + bps - 1) / bps;
            if (used != s) continue;
            const float per_cu = (float)wgs * (float)s / (float)n_cus, walk = mean / (float)(s * 32);
            const float longest = (float)((bps + qt - 1) / qt * qt * KB) / 32.0f;
            float cost = s > 1 ? 4.0f + (float)s * (0.25f + 0.4f * part_mb) : 0.f;
            if (qt == 2) {
                const float rounds = ceilf(per_cu), t = qc ? 0.75f + 0.18f * fminf(per_cu, 1.f) : 0.64f + 0.14f * fminf(per_cu, 1.f);
                cost += rounds * 14.0f + t * fmaxf(longest, rounds * walk);
            } else if (p.hd == 256) {
                cost += 10.0f + 2.0f * fmaxf(longest, ceilf(per_cu) * walk);
            } else {
                const float slots = qc && p.hd == 128 ? 3.f : 4.f, n = ceilf(per_cu), full = floorf(n / slots), rest = n - full * slots;
                auto at = [&](float k) -> float { return qc ? 0.55f + 0.38f * k : fmaxf(0.7f + 0.14f * k, 0.43f * k); };
                cost += 7.0f + size * fmaxf(at(1.f) * longest, (full * at(slots) + (rest > 0.f ? at(rest) : 0.f)) * walk);
            }
            if (cost < best_cost) best_cost = cost, best = {hpw, qt, wgs, s, bps};
        }
    }
    return best;
}

// Up to one block of keys with one query tile per wave (which is what plan_attn takes for so few).  23 tokens, 16 q heads and 8 kv
// heads of 128, us per layer in a kernel trace: 2.7 for the rows' own launch and 6.5 for the attention, 7.0 for both in one.
// With more keys every workgroup would work out more rows than its share of the waves can hold in flight.
bool oxb_attn_prefill_can_store(uint32_t hd, uint32_t pos_start, uint32_t M) { return pos_start == 0 && M <= (uint32_t)pf_block_keys((int)hd, 1); }

size_t oxb_attn_prefill_part_bytes(const OxbPrefillAttnParams& p, uint32_t n_cus) {
    const OxbPrefillAttnPlan pl = plan_attn(p, n_cus);
    const size_t rows = (size_t)p.M * p.nq;
    return pl.n_splits > 1 ? (pf_part_head(pl.n_splits, rows) + pl.n_splits * rows * p.hd) * sizeof(float) : 0;
}

hipError_t oxb_launch_attn_prefill(OxbPrefillAttnParams p, uint32_t n_cus, hipStream_t st) {
    if (p.M == 0 || p.nq == 0 || p.nkv == 0 || p.nq % p.nkv || !p.qkv || !p.q_norm || !p.cos_t || !p.sin_t || p.pos_start + p.M > p.max_seq || p.kv_mode > OXB_KV_FP8_E4M3 ||
        (p.kv_mode != OXB_KV_F16 && (!p.k_scale || !p.v_scale)) || (p.kv.page_table && (p.kv.page_shift < 4 || p.kv.page_shift > 7)))
        return hipErrorInvalidValue;
    if (p.k_norm && !oxb_attn_prefill_can_store(p.hd, p.pos_start, p.M)) return hipErrorInvalidValue;
    const OxbPrefillAttnPlan pl = plan_attn(p, n_cus);
    if ((pl.n_splits > 1 && !p.part) || (p.k_norm && (pl.qt != 1 || pl.n_splits != 1))) return hipErrorInvalidValue;
    p.blocks_per_split = pl.blocks_per_split;
    const dim3 grid(pl.wgs, pl.n_splits);
    const bool opt = p.window != 0 || p.kv.page_table != nullptr;
#define OXB_PF_LAUNCH(HD_, KVM_, QT_)                                                                                     \
    if (QT_ == 1 && p.k_norm) {                                                                                                                \
        if (opt) hipLaunchKernelGGL((attn_prefill_kernel<HD_, KVM_, true, 1, true>), grid, dim3(256), 0, st, p, pl.hpw);                   \
        else hipLaunchKernelGGL((attn_prefill_kernel<HD_, KVM_, false, 1, true>), grid, dim3(256), 0, st, p, pl.hpw);                      \
    } else if (opt) hipLaunchKernelGGL((attn_prefill_kernel<HD_, KVM_, true, QT_, false>), grid, dim3(256 * QT_), 0, st, p, pl.hpw);    \
    else hipLaunchKernelGGL((attn_prefill_kernel<HD_, KVM_, false, QT_, false>), grid, dim3(256 * QT_), 0, st, p, pl.hpw);
#define OXB_PF_KVM(HD_, QT_)                                  \
    if (p.kv_mode == OXB_KV_I8) {                             \
        OXB_PF_LAUNCH(HD_, OXB_KV_I8, QT_)                    \
    } else if (p.kv_mode == OXB_KV_FP8_E4M3) {                \
        OXB_PF_LAUNCH(HD_, OXB_KV_FP8_E4M3, QT_)              \
    } else {                                                  \
        OXB_PF_LAUNCH(HD_, OXB_KV_F16, QT_)                   \
    }
    switch (p.hd) {
        case 32: OXB_PF_KVM(32, 1) break;
        case 64: OXB_PF_KVM(64, 1) break;
        case 128:
            if (pl.qt == 2) {
                OXB_PF_KVM(128, 2)
            } else {
                OXB_PF_KVM(128, 1)
            }
            break;
        case 256: OXB_PF_KVM(256, 1) break;
        default: return hipErrorInvalidValue;
    }
#undef OXB_PF_LAUNCH
#undef OXB_PF_KVM
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || pl.n_splits == 1) return e;
    const uint32_t hpg = 256 / p.hd;
    hipLaunchKernelGGL(attn_prefill_merge_kernel, dim3((p.M + 3) / 4, (p.nq + hpg - 1) / hpg), dim3(256), 0, st, p.part, pl.n_splits, p.M, p.nq, p.hd, p.out, p.op);
    return hipGetLastError();
}
