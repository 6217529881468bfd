// gemm_kernels.hip — prefill GEMM for Q1_0_g128 / TQ2_0_g128 weights on gfx950:
//     Y[m][n] = sum_k W[n][k] * X[m][k]      (X: M token rows, W: the resident quantised matrix)
// (reference semantics: crates/oxibonsai-kernels/src/gemm.rs:19-87, gemm_ternary.rs:35-69; the CUDA tier's
// scalar-FMA kernels gemm_q1_g128_v7 / gemm_tq2_g128_v7, gpu_backend/cuda_prefill_kernels.rs:74-140, 457-551).
//
// Arithmetic.  Weights +-d / 0 are exact in fp16 and so is every product with an fp16 activation in the fp32
// accumulator of v_mfma_f32_16x16x32_f16; the only rounding beyond fp32 summation is the activation's
// conversion to fp16 (relative 2^-11 per element), after scaling each token row by a power of two so the
// result does not depend on the row's magnitude.
//
// Data flow.  The weight side never touches LDS: the resident layout (layout.h) already hands lane (r, g) of a
// wave the code bits of row r, k-group g, which is the MFMA A-operand position, so each lane expands its own
// bits to fp16 +-d in registers.  Because the k order inside an MFMA is free as long as A and B agree, the
// expansion pairs weights whose codes lie 16 bits apart in a code dword (one shift + one mask builds two fp16
// values) and the activation packer writes X in exactly that order:
//   xh[(blk * 16 + 4g + s) * M_pad + m]  = 16 bytes = the 8 fp16 that lane (token m, k-group g) feeds to MFMA
//   step s of block blk;  element 2p+h  <->  k = 128 blk + 32 g + 4 s + p + 16 h            (Q1)
//                                             k = 128 blk + 32 g + 16 (s/2) + 4 (s%2) + p + 8 h   (TQ2)
// One workgroup = 4 waves stacked along the weight rows; they share one token tile of X that is staged per
// 128-weight block through double-buffered LDS.  Wave w owns up to RT row tiles (16 rows each) and CT token
// tiles (16 tokens each): RT*CT accumulator tiles, RT decoded A operands reused over CT B operands.
#include <type_traits>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_utils.h"
#include "gemm_kernels.h"
#include "layout.h"
#include "operand_device.h"

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));

#define OXB_GEMM_THREADS 256

// ---------------------------------------------------------------------------
// Activation packer, fused with the row-wise producer of the activations:
//   OXB_PACK_IDENT   a[m][k] = x[m][k]
//   OXB_PACK_RMSNORM a[m][k] = w[k] * x[m][k] / sqrt(mean_k x[m][k]^2 + eps)      (simd_float_ops.rs:204-215)
// Two steps: the row's multiplier - the producer's scalar times the power of two that puts the row's largest |a| into
// [2^14, 2^15) - with the exponent that undoes the power of two; then the fp16 values in MFMA B-operand order.  The
// normalised activations never go to memory in fp32.  (SwiGLU is not a packer operation: the gate || up GEMM applies it in
// its epilogue, simd_float_ops.rs:217-236.)  Both steps take one launch: xh_pack_rows, one workgroup per row, for up to
// OXB_PACK_ROWS_MAX rows, xh_pack_wide beyond.  Rows too long for either to hold in registers take row_stats (one workgroup
// per token row) and xh_pack (one workgroup = 16 token rows x a share of the blocks), which read x twice.
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint32_t pack_h2(float a, float b) {
    const v2h h = {(_Float16)a, (_Float16)b};
    return __builtin_bit_cast(uint32_t, h);
}
__device__ __forceinline__ float sum_sq(const float4& a, float s) { return fmaf(a.x, a.x, fmaf(a.y, a.y, fmaf(a.z, a.z, fmaf(a.w, a.w, s)))); }
__device__ __forceinline__ float silu_mul(float g, float u) { return (g / (1.0f + expf(-g))) * u; }

// What the packer says about one token row: its multiplier, the exponent that undoes the power of two, and (RMSNORM) no less than
// the square of the 2-norm of its activations.
struct RowScale { float mul; int32_t xsh; float norm2; };
// ... from the row's sum of squares, that of its |a| before the producer's scalar, the largest of those and whether it holds
// something non-finite.
template <int OP>
__device__ __forceinline__ RowScale row_scale(float ss, float sa, float mx, int bad, uint32_t k, float eps, float cap) {
    float scalar = 1.0f;
    if (OP == OXB_PACK_RMSNORM) {
        scalar = 1.0f / sqrtf(ss / (float)k + eps);
        mx *= scalar;
        bad |= !(fabsf(scalar) <= 3.402823466e38f) | !(fabsf(mx) <= 3.402823466e38f);
    }
    int E = 0;
    if (mx > 0.0f) (void)frexpf(mx, &E);  // mx = f * 2^E, f in [0.5, 1)
    const int shift = mx > 0.0f ? 15 - E : 0;
    float norm2 = 1.0f;
    if (OP == OXB_PACK_RMSNORM && !bad) {
        // The squares are added up before the scalar: where their sum has left fp32's range at either end (a residual of 1e18 under a
        // norm weight of 20, a row of 1e-24 under a tiny eps) the largest |a| and the norm weights' bound take its place.  The
        // latter needs a sum of squares of x that has lost nothing to the lower end.
        norm2 = sa >= 0x1p-100f && sa <= 3.402823466e38f ? sa * scalar * scalar : (float)k * mx * mx;
        if (ss >= 0x1p-100f) norm2 = fminf(norm2, cap);
        norm2 = fmaxf(fminf(norm2, 3.402823466e38f), (float)k * 0x1p-126f);  // (products below that are lost to the lower end)
    }
    return {bad ? 0.0f : ldexpf(scalar, shift), bad ? INT32_MIN : -shift, norm2};
}

// The threads' partial results (sums of squares of x and of a, largest |a|, non-finite seen) joined; all 256 threads of the
// workgroup call it, thread 0 gets the result.
struct RowRed { float s[4], a[4], m[4]; int b[4]; };
template <int OP>
__device__ __forceinline__ RowScale row_finish(float ss, float sa, float mx, int bad, uint32_t k, float eps, float cap, RowRed& red);

// The same with the pass over the row in front: a float4 per thread and step, in row order.
template <int OP>
__device__ __forceinline__ RowScale row_stats(const float* __restrict__ xr, const float* __restrict__ w, uint32_t k, float eps, float cap, RowRed& red) {
    const uint32_t tid = threadIdx.x;
    float ss = 0.f, sa = 0.f, mx = 0.f;
    int bad = 0;
    for (uint32_t i = tid * 4; i < k; i += 1024) {
        const float4 v = *reinterpret_cast<const float4*>(xr + i);
        float4 a = v;
        if (OP == OXB_PACK_RMSNORM) {
            const float4 g = *reinterpret_cast<const float4*>(w + i);
            ss = fmaf(v.x, v.x, fmaf(v.y, v.y, fmaf(v.z, v.z, fmaf(v.w, v.w, ss))));
            a = make_float4(g.x * v.x, g.y * v.y, g.z * v.z, g.w * v.w);
            sa = sum_sq(a, sa);
        }
        bad |= !(fabsf(a.x) <= 3.402823466e38f) | !(fabsf(a.y) <= 3.402823466e38f) | !(fabsf(a.z) <= 3.402823466e38f) |
               !(fabsf(a.w) <= 3.402823466e38f);
        mx = fmaxf(fmaxf(mx, fmaxf(fabsf(a.x), fabsf(a.y))), fmaxf(fabsf(a.z), fabsf(a.w)));
    }
    return row_finish<OP>(ss, sa, mx, bad, k, eps, cap, red);
}

template <int OP>
__device__ __forceinline__ RowScale row_finish(float ss, float sa, float mx, int bad, uint32_t k, float eps, float cap, RowRed& red) {
    const uint32_t tid = threadIdx.x;
    if (OP == OXB_PACK_RMSNORM) ss = wave_sum_f32(ss), sa = wave_sum_f32(sa);  // DPP and lane swaps: no trips through the LDS pipeline
    mx = wave_max_f32(mx);
    bad = __builtin_amdgcn_ballot_w64(bad != 0) != 0;
    if ((tid & 63u) == 0) red.s[tid >> 6] = ss, red.a[tid >> 6] = sa, red.m[tid >> 6] = mx, red.b[tid >> 6] = bad;
    __syncthreads();
    if (tid) return {0.f, 0, 0.f};
    return row_scale<OP>(red.s[0] + red.s[1] + red.s[2] + red.s[3], red.a[0] + red.a[1] + red.a[2] + red.a[3],
                         fmaxf(fmaxf(red.m[0], red.m[1]), fmaxf(red.m[2], red.m[3])), red.b[0] | red.b[1] | red.b[2] | red.b[3], k, eps, cap);
}

template <int OP>
__global__ __launch_bounds__(256) void row_stats_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                         uint32_t ldx, uint32_t k, float eps, float* __restrict__ rowmul,
                                                         int32_t* __restrict__ xsh, const OxbPackNorm norm) {
    __shared__ RowRed red;
    const uint32_t m = blockIdx.x;
    const RowScale r = row_stats<OP>(x + (size_t)m * ldx, w, k, eps, norm.cap, red);
    if (threadIdx.x) return;
    rowmul[m] = r.mul, xsh[m] = r.xsh;
    if (norm.norm2) norm.norm2[m] = r.norm2;
}

// The eight activations of token row xr that chunk c = 4g + s of block blk holds, scaled by mul, as four fp16 pairs.
template <int FMT, int OP>
__device__ __forceinline__ uint4 pack_item(const float* __restrict__ xr, const float* __restrict__ w, uint32_t k, uint32_t blk,
                                           uint32_t c, float mul) {
    const uint32_t g = c >> 2, s = c & 3u;
    const uint32_t k0 = FMT == OXB_FMT_Q1 ? 32 * g + 4 * s : 32 * g + 16 * (s >> 1) + 4 * (s & 1u);
    const uint32_t k1 = k0 + (FMT == OXB_FMT_Q1 ? 16 : 8);
    const float* xb = xr + blk * 128;
    float4 a = *reinterpret_cast<const float4*>(xb + k0);
    float4 b = *reinterpret_cast<const float4*>(xb + k1);
    if (OP == OXB_PACK_RMSNORM) {
        const float4 wa = *reinterpret_cast<const float4*>(w + blk * 128 + k0), wb = *reinterpret_cast<const float4*>(w + blk * 128 + k1);
        a = make_float4(wa.x * a.x, wa.y * a.y, wa.z * a.z, wa.w * a.w);
        b = make_float4(wb.x * b.x, wb.y * b.y, wb.z * b.z, wb.w * b.w);
    }
    return make_uint4(pack_h2(a.x * mul, b.x * mul), pack_h2(a.y * mul, b.y * mul), pack_h2(a.z * mul, b.z * mul),
                      pack_h2(a.w * mul, b.w * mul));
}

// The two 16-byte pieces of token row xr behind chunk c = 4g + s of block blk (pack_item's loads).
template <int FMT>
__device__ __forceinline__ void item_offsets(uint32_t blk, uint32_t c, uint32_t* o0, uint32_t* o1) {
    const uint32_t g = c >> 2, s = c & 3u;
    const uint32_t k0 = FMT == OXB_FMT_Q1 ? 32 * g + 4 * s : 32 * g + 16 * (s >> 1) + 4 * (s & 1u);
    *o0 = blk * 128 + k0;
    *o1 = *o0 + (FMT == OXB_FMT_Q1 ? 16 : 8);
}

__device__ __forceinline__ float4 add4(const float4& a, const float4& b) { return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w); }

// Both steps in one launch for a few token rows (decode batches): one workgroup per token row, one pass over the row.
// A thread requests all of its items - the pieces it will pack, NI of them for rows of up to 2048 NI values - before
// it uses any, keeps them in registers while the workgroup finds the row's multiplier, and packs them from there;
// rows M .. M_pad - 1 are zero-filled.  With eight to thirty-two workgroups on the whole GPU the launch is as long
// as its chain of memory round trips: this way it is one for the row and one for the store.  (The sum of squares adds
// the row's values in another order than row_stats does: the multiplier may differ from the two-kernel route's in the
// last bit, within what fp16 activations already cost.)
// SUM: x is a product's residual whose partial sums still lie in sum.n planes; they are added here, in slice order, and
// x is written back (a launch of its own for that costs as much as the slices save).
template <int FMT, int OP, int NI, bool SUM>
__global__ __launch_bounds__(256) void xh_pack_rows_kernel(float* x, const float* __restrict__ w, uint32_t ldx,
                                                            uint32_t k, float eps, uint32_t M, uint32_t M_pad, uint32_t nblk_pad,
                                                            int32_t* __restrict__ xsh, const OxbPackNorm norm, uint4* __restrict__ xh, const OxbPackSum sum) {
    __shared__ RowRed red;
    __shared__ float mul_s;
    const uint32_t m = blockIdx.x, tid = threadIdx.x, n_items = nblk_pad * 16;
    if (m >= M) {  // uniform over the workgroup
        for (uint32_t id = tid; id < n_items; id += 256) xh[(size_t)id * M_pad + m] = make_uint4(0, 0, 0, 0);
        return;
    }
    float* xr = x + (size_t)m * ldx;
    float4 a[NI], b[NI], wa[NI], wb[NI];
#pragma unroll
    for (int it = 0; it < NI; it++) {
        const uint32_t id = it * 256 + tid;
        uint32_t o0, o1;
        item_offsets<FMT>(id >> 4, id & 15u, &o0, &o1);
        const bool ok = id < n_items && (id >> 4) * 128 < k;  // blocks past k are padding
        a[it] = ok ? *reinterpret_cast<const float4*>(xr + o0) : make_float4(0.f, 0.f, 0.f, 0.f);
        b[it] = ok ? *reinterpret_cast<const float4*>(xr + o1) : make_float4(0.f, 0.f, 0.f, 0.f);
        if (OP == OXB_PACK_RMSNORM) {
            wa[it] = ok ? *reinterpret_cast<const float4*>(w + o0) : make_float4(0.f, 0.f, 0.f, 0.f);
            wb[it] = ok ? *reinterpret_cast<const float4*>(w + o1) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    }
    if (SUM) {
        const float* pr = sum.part + (size_t)m * ldx;
        float4 ta[NI], tb[NI];
        for (uint32_t s0 = 0; s0 < sum.n; s0 += 4) {  // four planes requested together
            float4 pa[4][NI], pb[4][NI];
#pragma unroll
            for (uint32_t j = 0; j < 4; j++)
#pragma unroll
                for (int it = 0; it < NI; it++) {
                    const uint32_t id = it * 256 + tid;
                    uint32_t o0, o1;
                    item_offsets<FMT>(id >> 4, id & 15u, &o0, &o1);
                    const bool ok = s0 + j < sum.n && id < n_items && (id >> 4) * 128 < k;
                    const float* q = pr + (s0 + j) * sum.plane;
                    pa[j][it] = ok ? *reinterpret_cast<const float4*>(q + o0) : make_float4(0.f, 0.f, 0.f, 0.f);
                    pb[j][it] = ok ? *reinterpret_cast<const float4*>(q + o1) : make_float4(0.f, 0.f, 0.f, 0.f);
                }
#pragma unroll
            for (uint32_t j = 0; j < 4; j++)
#pragma unroll
                for (int it = 0; it < NI; it++) {
                    ta[it] = s0 + j == 0 ? pa[j][it] : add4(ta[it], pa[j][it]);
                    tb[it] = s0 + j == 0 ? pb[j][it] : add4(tb[it], pb[j][it]);
                }
        }
#pragma unroll
        for (int it = 0; it < NI; it++) {
            const uint32_t id = it * 256 + tid;
            uint32_t o0, o1;
            item_offsets<FMT>(id >> 4, id & 15u, &o0, &o1);
            a[it] = add4(ta[it], a[it]);
            b[it] = add4(tb[it], b[it]);
            if (id < n_items && (id >> 4) * 128 < k) {
                *reinterpret_cast<float4*>(xr + o0) = a[it];
                *reinterpret_cast<float4*>(xr + o1) = b[it];
            }
        }
    }
    float ss = 0.f, sa = 0.f, mx = 0.f;
    int bad = 0;
#pragma unroll
    for (int it = 0; it < NI; it++) {
        float4& p = a[it];
        float4& q = b[it];
        if (OP == OXB_PACK_RMSNORM) {
            ss = fmaf(p.x, p.x, fmaf(p.y, p.y, fmaf(p.z, p.z, fmaf(p.w, p.w, ss))));
            ss = fmaf(q.x, q.x, fmaf(q.y, q.y, fmaf(q.z, q.z, fmaf(q.w, q.w, ss))));
            p = make_float4(wa[it].x * p.x, wa[it].y * p.y, wa[it].z * p.z, wa[it].w * p.w);
            q = make_float4(wb[it].x * q.x, wb[it].y * q.y, wb[it].z * q.z, wb[it].w * q.w);
            sa = sum_sq(q, sum_sq(p, sa));
        }
        const float v[8] = {p.x, p.y, p.z, p.w, q.x, q.y, q.z, q.w};
#pragma unroll
        for (int e = 0; e < 8; e++) {
            bad |= !(fabsf(v[e]) <= 3.402823466e38f);
            mx = fmaxf(mx, fabsf(v[e]));
        }
    }
    const RowScale rs = row_finish<OP>(ss, sa, mx, bad, k, eps, norm.cap, red);
    if (tid == 0) {
        mul_s = rs.mul, xsh[m] = rs.xsh;
        if (OP == OXB_PACK_RMSNORM && norm.norm2) norm.norm2[m] = rs.norm2;
    }
    __syncthreads();
    const float mul = mul_s;
#pragma unroll
    for (int it = 0; it < NI; it++) {
        const uint32_t id = it * 256 + tid;
        if (id >= n_items) continue;
        const float4 p = a[it], q = b[it];
        xh[(size_t)id * M_pad + m] = make_uint4(pack_h2(p.x * mul, q.x * mul), pack_h2(p.y * mul, q.y * mul),
                                                pack_h2(p.z * mul, q.z * mul), pack_h2(p.w * mul, q.w * mul));
    }
}

// Both steps in one launch for many token rows: the eight waves of a workgroup own RPW rows (8, 4 or 2), 8 / RPW waves a
// row.  A wave requests its whole share of the row at once (4 NI values per lane) and keeps it in registers, so x is read
// once; the fp16 values then change from row order to chunk order through LDS, SEG pieces per lane at a time, and leave in
// runs of RPW x 16 bytes (RPW rows side by side in a chunk).  row_stats_kernel + xh_pack_kernel read x twice in two
// launches.  What bounds it is the way into and out of a CU (64 bytes a clock each) and, for few rows, the chain of one
// memory round trip, two barriers and the stores.  A layer's four packs, 8B shape, two launches each before: 2048 rows
// 93 -> 56 us, 301 rows 41 -> 26 us.
// (SUM as in xh_pack_rows_kernel.)
template <int FMT, int OP, int RPW, int NI, bool SUM>
__global__ __launch_bounds__(512) void xh_pack_wide_kernel(float* x, const float* __restrict__ w, uint32_t ldx, uint32_t k,
                                                            float eps, uint32_t M, uint32_t M_pad, uint32_t nblk_pad,
                                                            int32_t* __restrict__ xsh, const OxbPackNorm norm, uint4* __restrict__ xh, const OxbPackSum sum) {
    constexpr int WPR = 8 / RPW, SEG = NI <= 16 ? NI : NI == 48 ? 16 : 12;
    static_assert(NI % SEG == 0, "whole segments");
    constexpr uint32_t VALS = SEG * 256 * WPR, STR = VALS + 16;  // values of a row in a segment; LDS row stride (32 bytes of padding spread the rows over the banks)
    constexpr int WG = OP == OXB_PACK_RMSNORM && NI > 16 ? 4 : SEG;  // norm weights requested at a time (registers)
    __shared__ __attribute__((aligned(16))) _Float16 rows[RPW * STR];
    __shared__ float red_s[8], red_a[8], red_m[8];
    __shared__ int red_b[8];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, m0 = blockIdx.x * RPW;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6)), wr = wave / WPR, part = wave % WPR, m = m0 + wr;
    const bool live = m < M;
    float* xr = x + (size_t)(live ? m : 0) * ldx;
    auto at_of = [&](int i) -> uint32_t { return ((i * WPR + part) * 64 + lane) * 4; };
    float4 a[NI];
#pragma unroll
    for (int i = 0; i < NI; i++) a[i] = live && at_of(i) < k ? *reinterpret_cast<const float4*>(xr + at_of(i)) : make_float4(0.f, 0.f, 0.f, 0.f);
    if (SUM && live) {
        const float* pr = sum.part + (size_t)m * ldx;
        float4 t[NI];
        for (uint32_t s = 0; s < sum.n; s++) {
            float4 q[NI];
#pragma unroll
            for (int i = 0; i < NI; i++) q[i] = at_of(i) < k ? *reinterpret_cast<const float4*>(pr + s * sum.plane + at_of(i)) : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int i = 0; i < NI; i++) t[i] = s == 0 ? q[i] : add4(t[i], q[i]);
        }
#pragma unroll
        for (int i = 0; i < NI; i++) {
            a[i] = add4(t[i], a[i]);
            if (at_of(i) < k) *reinterpret_cast<float4*>(xr + at_of(i)) = a[i];
        }
    }
    float ss = 0.f, sa = 0.f, mx = 0.f;
    int bad = 0;
#pragma unroll
    for (int i0 = 0; i0 < NI; i0 += WG) {
        float4 g[OP == OXB_PACK_RMSNORM ? WG : 1];
        if (OP == OXB_PACK_RMSNORM) {
#pragma unroll
            for (int i = 0; i < WG; i++) g[i] = at_of(i0 + i) < k ? *reinterpret_cast<const float4*>(w + at_of(i0 + i)) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
#pragma unroll
        for (int i = 0; i < WG; i++) {
            float4& v = a[i0 + i];
            if (OP == OXB_PACK_RMSNORM) {
                ss = fmaf(v.x, v.x, fmaf(v.y, v.y, fmaf(v.z, v.z, fmaf(v.w, v.w, ss))));
                const float4 q = g[OP == OXB_PACK_RMSNORM ? i : 0];
                v = make_float4(q.x * v.x, q.y * v.y, q.z * v.z, q.w * v.w);
                sa = sum_sq(v, sa);
            }
            bad |= !(fabsf(v.x) <= 3.402823466e38f) | !(fabsf(v.y) <= 3.402823466e38f) | !(fabsf(v.z) <= 3.402823466e38f) |
                   !(fabsf(v.w) <= 3.402823466e38f);
            mx = fmaxf(fmaxf(mx, fmaxf(fabsf(v.x), fabsf(v.y))), fmaxf(fabsf(v.z), fabsf(v.w)));
        }
    }
    if (OP == OXB_PACK_RMSNORM) ss = wave_sum_f32(ss), sa = wave_sum_f32(sa);
    mx = wave_max_f32(mx);
    bad = __builtin_amdgcn_ballot_w64(bad != 0) != 0;
    if constexpr (WPR > 1) {  // the row's waves, added in wave order
        if (lane == 0) red_s[wave] = ss, red_a[wave] = sa, red_m[wave] = mx, red_b[wave] = bad;
        __syncthreads();
        ss = red_s[wr * WPR], sa = red_a[wr * WPR], mx = red_m[wr * WPR], bad = red_b[wr * WPR];
#pragma unroll
        for (int i = 1; i < WPR; i++) ss += red_s[wr * WPR + i], sa += red_a[wr * WPR + i], mx = fmaxf(mx, red_m[wr * WPR + i]), bad |= red_b[wr * WPR + i];
    }
    const RowScale rs = row_scale<OP>(ss, sa, mx, bad, k, eps, norm.cap);
    const float mul = live ? rs.mul : 0.f;
    if (live && part == 0 && lane == 0) {
        xsh[m] = rs.xsh;
        if (OP == OXB_PACK_RMSNORM && norm.norm2) norm.norm2[m] = rs.norm2;
    }
#pragma unroll
    for (int i0 = 0; i0 < NI; i0 += SEG) {
        if (i0) __syncthreads();  // the segment before has been read
#pragma unroll
        for (int i = 0; i < SEG; i++) {
            const float4 v = a[i0 + i];
            *reinterpret_cast<uint2*>(&rows[wr * STR + at_of(i)]) = make_uint2(pack_h2(v.x * mul, v.y * mul), pack_h2(v.z * mul, v.w * mul));
        }
        __syncthreads();
        const uint32_t blk0 = (uint32_t)(i0 / SEG) * (VALS / 128), blks = min(nblk_pad - min(nblk_pad, blk0), VALS / 128);  // blocks of this segment
        for (uint32_t id = tid; id < blks * 16 * RPW; id += 512) {  // (chunk, row), rows first
            const uint32_t row = id % RPW, c = id / RPW;
            uint32_t o0, o1;
            item_offsets<FMT>(c >> 4, c & 15u, &o0, &o1);
            const uint2 p = *reinterpret_cast<const uint2*>(&rows[row * STR + o0]), q = *reinterpret_cast<const uint2*>(&rows[row * STR + o1]);
            // values 0..3 of the first piece side by side with those of the second
            xh[(size_t)(blk0 * 16 + c) * M_pad + m0 + row] =
                make_uint4(__builtin_amdgcn_perm(q.x, p.x, 0x05040100u), __builtin_amdgcn_perm(q.x, p.x, 0x07060302u),
                           __builtin_amdgcn_perm(q.y, p.y, 0x05040100u), __builtin_amdgcn_perm(q.y, p.y, 0x07060302u));
        }
    }
}

template <int FMT, int OP>
__global__ __launch_bounds__(256) void xh_pack_kernel(const float* __restrict__ x, const float* __restrict__ w, uint32_t ldx,
                                                       uint32_t k, uint32_t M, uint32_t M_pad, uint32_t nblk_pad,
                                                       const float* __restrict__ rowmul, uint4* __restrict__ xh) {
    const uint32_t tid = threadIdx.x, m0 = blockIdx.x * 16;
    const uint32_t j = tid & 15u, c = tid >> 4, m = m0 + j;
    const bool live = m < M;
    const float mul = live ? rowmul[m] : 0.0f;
    for (uint32_t blk = blockIdx.y; blk < nblk_pad; blk += gridDim.y) {
        uint4 o = make_uint4(0, 0, 0, 0);
        if (live && blk * 128 < k) o = pack_item<FMT, OP>(x + (size_t)m * ldx, w, k, blk, c, mul);
        xh[(size_t)(blk * 16 + c) * M_pad + m] = o;
    }
}

// ---------------------------------------------------------------------------
// GEMM.
// ---------------------------------------------------------------------------
// How a kernel expands its weights (template FMT): by the matrix's format, and one more for a ternary matrix with a scale of 2^15 or
// more, twice which fp16 does not hold (decode_step).
enum { GEMM_TQ2_LOUD = OXB_FMT_TQ2 + 1 };
static_assert(OXB_FMT_Q1 == 0 && OXB_FMT_TQ2 == 1, "the forms of a matrix's weights");

// Codes and scales of one row tile for half a superblock (two 128-weight blocks), as loaded: the unit of the
// in-place register ring (half 0 is reloaded for the next superblock while half 1 is still being consumed).
template <int FMT>
struct HalfRegs {
    uint32_t c[FMT == OXB_FMT_Q1 ? 2 : 4];  // Q1: dword e = sign bits of block e; TQ2: dwords 2e, 2e+1 = fields of block e
    uint32_t d[2];                          // fp16 scale bits of blocks 0, 1 of the half (this lane's row)
};

template <int FMT>
__device__ __forceinline__ void load_half(HalfRegs<FMT>& H, __amdgpu_buffer_rsrc_t rc, __amdgpu_buffer_rsrc_t rs,
                                          uint32_t tile, bool ok, uint32_t n_sb, uint32_t sb, int half, uint32_t lane) {
    const uint32_t r = lane & 15u;
    const uint32_t unit = tile * n_sb + sb;  // wave-uniform
    ok = ok && sb < n_sb;
    if (FMT == OXB_FMT_Q1) {
        const v2u v = __builtin_amdgcn_raw_buffer_load_b64(rc, (int)(ok ? lane * 16u : OXB_OOB), (int)(unit * 1024u + half * 8u), 0);
        H.c[0] = v.x, H.c[1] = v.y;
    } else {
        const v4i v = buf_load_b128(rc, ok ? lane * 16u : OXB_OOB, unit * 2048u + half * 1024u);
        H.c[0] = (uint32_t)v.x, H.c[1] = (uint32_t)v.y, H.c[FMT == OXB_FMT_Q1 ? 0 : 2] = (uint32_t)v.z,
        H.c[FMT == OXB_FMT_Q1 ? 1 : 3] = (uint32_t)v.w;
    }
    // scales of blocks 2 * half and 2 * half + 1 of this lane's row lie side by side
    const uint32_t sv = __builtin_amdgcn_raw_buffer_load_b32(rs, (int)(ok ? r * 8u : OXB_OOB), (int)(unit * 128u + half * 4u), 0);
    H.d[0] = sv & 0xFFFFu;
    H.d[1] = sv >> 16;
}

// Per (row tile, block) state prepared once and used by the four MFMA steps of the block.
struct BlockDec {
    uint32_t w0, w1;  // Q1: w0 = inverted sign bits (xor the scale's sign); TQ2: fields of the 16-weight halves as sign and magnitude bits
    uint32_t d2;      // Q1: |d| in both halves of the dword; TQ2: d in both halves
};

// TQ2.  A field with both bits inverted is a sign bit above a magnitude bit (-1 = 3, 0 = 2, which is minus 0, +1 = 1); those at in-byte
// position 3 are that as they are (two's complement: 3, 0, 1).  Shifted to the top of a half and masked it is the fp16 number +-2 or
// +-0, and one packed multiplication by d makes the weight, twice as large as it is: three instructions for two weights where
// building 1024 + field, subtracting 1025 and multiplying takes four.  The factor goes into the row's exponent (row_exp).
// A matrix with a scale of 2^15 or more (GEMM_TQ2_LOUD) has these numbers halved first, which is exact, and the weights as they are:
// an instruction more.  (Half the scale instead would round the ones below 2^-13.)
// us, TQ2, four instructions / three: 19456 x 2560 at 64 / 301 / 512 / 2048 rows 16.8 / 37.5 / 51.3 / 190 and 14.8 / 35.2 / 50.8 / 186, the
// same as gate || up with SwiGLU 20.2 / 42.6 / 61.0 / 198 and 18.3 / 39.0 / 57.7 / 188; 12288 x 2048 with SwiGLU at 200 / 512 / 2048 24.2 /
// 34.5 / 100.5 and 22.1 / 32.9 / 95.8; 2560 x 9728 at 16 / 128 / 512 6.3 / 18.9 / 40.6 and 5.85 / 17.6 / 38.1; 5120 x 2560 at 23 / 301 / 512
// 5.7 / 16.6 / 23.2 and 5.15 / 14.9 / 21.5.  Equal up to 2 % slower with two row tiles and seven token tiles (97 to 112 rows of 6144 x
// 4096 12.1 and 12.3, of 12288 x 2048 13.9 and 14.3).

template <int FMT>
__device__ __forceinline__ BlockDec prepare_block(const HalfRegs<FMT>& H, int e) {
    BlockDec B;
    const uint32_t dbits = H.d[e];
    const uint32_t dd = (dbits & 0xFFFFu) * 0x00010001u;
    if (FMT == OXB_FMT_Q1) {
        // weight = bit ? d : -d  ->  sign bit = ~bit ^ sign(d)
        const uint32_t flip = (uint32_t)((int32_t)(dbits << 16) >> 31);
        B.w0 = ~H.c[e] ^ flip;
        B.w1 = 0;
        B.d2 = dd & 0x7FFF7FFFu;
    } else {
        B.w0 = H.c[FMT == OXB_FMT_Q1 ? 0 : 2 * e] ^ 0x3F3F3F3Fu;
        B.w1 = H.c[FMT == OXB_FMT_Q1 ? 0 : 2 * e + 1] ^ 0x3F3F3F3Fu;
        // (Opaque, or the inversion moves into the masks that take it and the loaded codes live on: up to 30 registers more, with which
        // three of the wide kernel's forms and <2, 7> of the narrow one spill or lose a workgroup a CU: 6144 x 4096 at 97 rows 15.0 us
        // against 12.3, 24576 x 4096 at 400 84.7 against 71.7, gate || up 12288 x 2048 at 700 47.3 against 44.2.)
        asm("" : "+v"(B.w0), "+v"(B.w1));
        B.d2 = dd;
    }
    return B;
}

// The A operands of MFMA step s (0..3) of the block for all row tiles.  Written operation by operation across
// the RT x 4 independent dwords, so that consecutive VALU instructions do not depend on each other.
template <int FMT, int RT>
__device__ __forceinline__ void decode_step(const BlockDec (&B)[RT], int s, v8h (&A)[RT]) {
    uint32_t o[RT][4];
    // The masks live in registers (VOP3 encodings take no literal), opaque to the compiler so that
    // (x & mask) | y stays one v_and_or_b32.
    uint32_t kmask;
    if (FMT == OXB_FMT_Q1) {
        asm volatile("s_mov_b32 %0, 0x80008000" : "=s"(kmask));
#pragma unroll
        for (int p = 0; p < 4; p++)
#pragma unroll
            for (int rt = 0; rt < RT; rt++) o[rt][p] = B[rt].w0 << (15 - (4 * s + p));
#pragma unroll
        for (int p = 0; p < 4; p++)
#pragma unroll
            for (int rt = 0; rt < RT; rt++) o[rt][p] = (o[rt][p] & kmask) | B[rt].d2;
    } else {
        asm volatile("s_mov_b32 %0, 0xC000C000" : "=s"(kmask));
#pragma unroll
        for (int p = 0; p < 4; p++)
#pragma unroll
            for (int rt = 0; rt < RT; rt++) o[rt][p] = ((s >> 1) ? B[rt].w1 : B[rt].w0) << (14 - 2 * (4 * (s & 1) + p));
#pragma unroll
        for (int p = 0; p < 4; p++)
#pragma unroll
            for (int rt = 0; rt < RT; rt++) o[rt][p] &= kmask;  // fp16 2, -2, 0 or -0
        if (FMT == GEMM_TQ2_LOUD) {
            const v2h half = {(_Float16)0.5f, (_Float16)0.5f};
#pragma unroll
            for (int p = 0; p < 4; p++)
#pragma unroll
                for (int rt = 0; rt < RT; rt++) o[rt][p] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(v2h, o[rt][p]) * half);
        }
#pragma unroll
        for (int p = 0; p < 4; p++)
#pragma unroll
            for (int rt = 0; rt < RT; rt++) o[rt][p] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(v2h, o[rt][p]) * __builtin_bit_cast(v2h, B[rt].d2));
    }
#pragma unroll
    for (int rt = 0; rt < RT; rt++) {
        const v4u u = {o[rt][0], o[rt][1], o[rt][2], o[rt][3]};
        A[rt] = __builtin_bit_cast(v8h, u);
    }
}

typedef __attribute__((address_space(3))) void* lds_ptr_t;

// One 128-weight block of the K loop: 4 MFMA steps over the staged token tile `xsb`.  The A operands of the
// step after the current one are expanded while the current step's MFMAs run (for the last step: the first
// step of the next block, from `bdn`), and each B operand is reloaded for the next step right after its last use.
template <int FMT, int RT, int CT>
__device__ __forceinline__ void block_steps(const v8h* __restrict__ xsb, v8h (&A)[RT], const BlockDec (&bd)[RT],
                                            const BlockDec (&bdn)[RT], v4f (&acc)[RT][CT], uint32_t boff) {
    constexpr int BM = 16 * CT;
    constexpr int NV = FMT == OXB_FMT_Q1 ? 1 : 2;  // VALU instructions issued after each MFMA, while there are any (a step has 8 or 12 a row tile)
    v8h B[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ct++) B[ct] = xsb[boff + ct * 16];
    // all B operands of the first step are requested at once, so their LDS latency is paid once per block
    __builtin_amdgcn_sched_group_barrier(0x100, CT, 0);
#pragma unroll
    for (int s = 0; s < 4; s++) {
        v8h An[RT];
        if (s < 3)
            decode_step<FMT, RT>(bd, s + 1, An);
        else
            decode_step<FMT, RT>(bdn, 0, An);
#pragma unroll
        for (int ct = 0; ct < CT; ct++) {
#pragma unroll
            for (int rt = 0; rt < RT; rt++)  // row tiles past the range hold zero weights
                acc[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[rt], B[ct], acc[rt][ct], 0, 0, 0);
            if (s < 3) B[ct] = xsb[boff + (s + 1) * BM + ct * 16];
        }
#pragma unroll
        for (int rt = 0; rt < RT; rt++) A[rt] = An[rt];
        // issue order: one MFMA, then the VALU work that expands the next A operand, a B reload per token tile
#pragma unroll
        for (int i = 0; i < RT * CT; i++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            // (the first step also absorbs the per-block preparation of the next block's codes)
            if (s == 0)
                __builtin_amdgcn_sched_group_barrier(0x002, NV + 1, 0);
            else
                __builtin_amdgcn_sched_group_barrier(0x002, NV, 0);
            if (s < 3 && i % RT == RT - 1) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_barrier(0);  // one scheduling region per step keeps compile time bounded
    }
}

// Exponent that undoes the scaling of token row m, INT32_MIN for a row that holds something non-finite.
template <int FMT>
__device__ __forceinline__ int row_exp(const OxbGemmParams& p, uint32_t m) {
    const int e = p.xsh ? p.xsh[m] : p.x_exp;
    return e == INT32_MIN || FMT != OXB_FMT_TQ2 ? e : e - 1;
}

// SWIGLU with the next product's operand as the output: |silu(gate) up| <= |gate up| <= w_mant 2^w_exp norm2 (Cauchy-Schwarz), so that
// times 2^shift it lies below 2^15: a factor of two from fp16's end for the roundings on the way.
__device__ __forceinline__ int swiglu_shift(const OxbGemmParams& p, uint32_t m) {
    int e;
    (void)frexpf(p.w_mant * p.norm2[m], &e);
    return 15 - p.w_exp - e;
}

// What else the operand of n_rows / 2 values a row needs: the rows' exponents, and zeros in the blocks up to a whole superblock.
// By one workgroup for `rows` rows from m0 on.
__device__ __forceinline__ void finish_operand(const OxbGemmParams& p, uint32_t m0, uint32_t rows, uint32_t tid, uint32_t threads) {
    for (uint32_t j = tid; j < rows && m0 + j < p.M; j += threads) p.xsh_out[m0 + j] = -swiglu_shift(p, m0 + j);
    const uint32_t blocks = p.n_rows / 256u, pad = ((blocks + 3u) & ~3u) - blocks;
    for (uint32_t i = tid; i < pad * 16u * rows; i += threads)
        reinterpret_cast<uint4*>(p.xh_out)[(size_t)(blocks * 16u + i / rows) * p.M_pad + m0 + i % rows] = make_uint4(0, 0, 0, 0);
}

template <int FMT, int RT, int CT>
__global__ __launch_bounds__(OXB_GEMM_THREADS, RT == 3 ? 2 : 1) void gemm_mfma_kernel(const OxbGemmParams p) {
    constexpr int BM = 16 * CT;
    // two stages of the token tile: [chunk 4g+s][token] x 16 bytes.  Separate arrays, so that loads in flight
    // into one stage do not make reads of the other wait.
    __shared__ __attribute__((aligned(16))) uint4 xs0[16 * BM];
    __shared__ __attribute__((aligned(16))) uint4 xs1[16 * BM];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, r = lane & 15u, g = lane >> 4;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));  // keeps unit offsets in SGPRs
    const uint32_t m_t = blockIdx.x % p.n_mt, n_g = (blockIdx.x / p.n_mt) % p.n_ng, ks = blockIdx.x / (p.n_mt * p.n_ng);
    const uint32_t m0 = m_t * BM;
    // K slice of this workgroup, in superblocks
    const uint32_t sb0 = ks * p.sb_per_split, sb1 = min(sb0 + p.sb_per_split, p.n_sb);
    // row tiles: the workgroup's [wg_t0, wg_t1), split evenly over the four waves
    const uint32_t wg_t0 = n_g * p.tpw, wg_t1 = min(wg_t0 + p.tpw, p.n_tiles);
    // SWIGLU mode (the matrix is gate || up).  Two tiles per wave: a gate tile and the up tile of the same rows.  Three (the
    // count that still runs two workgroups per CU): waves 0 and 1 take three gate tiles each, waves 2 and 3 the up tiles of
    // the same rows.  The factors meet in the LDS stages once the K loop is done.
    const bool sw = p.mode == OXB_GEMM_SWIGLU;
    constexpr bool SPLIT = RT == 3;  // (of the SWIGLU mode; other odd counts are never launched in it)
    auto tile_of = [&](uint32_t u) -> uint32_t { return sw ? ((u & 1u) ? p.n_tiles / 2 + (u >> 1) : (u >> 1)) : u; };
    uint32_t t0 = 0, n_valid = 0, up_base = 0;  // first tile index of this wave (an index into tile_of, or with SPLIT a gate tile)
    if (sw && SPLIT) {
        const uint32_t half_tiles = p.n_tiles / 2, g_first = n_g * (2 * RT) + (wave & 1u) * RT;
        t0 = g_first;
        n_valid = g_first < half_tiles ? min((uint32_t)RT, half_tiles - g_first) : 0u;
        up_base = (wave >> 1) ? half_tiles : 0u;
    } else {
        const uint32_t per = (p.tpw + 3u) / 4u;  // <= RT
        t0 = wg_t0 + wave * per;
        const uint32_t t1 = min(t0 + per, wg_t1);
        n_valid = t1 > t0 ? t1 - t0 : 0u;
    }
    auto tile_at = [&](uint32_t rt) -> uint32_t { return (sw && SPLIT) ? up_base + t0 + rt : tile_of(t0 + rt); };

    const __amdgpu_buffer_rsrc_t rc = make_rsrc(p.codes, p.codes_bytes), rs = make_rsrc(p.scales, p.scales_bytes);
    const __amdgpu_buffer_rsrc_t rx = make_rsrc(p.xh, p.xh_bytes);

    v4f acc[RT][CT];
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
        for (int ct = 0; ct < CT; ct++) acc[rt][ct] = (v4f){0.f, 0.f, 0.f, 0.f};

    // this thread's share of an X stage: CT items of 16 bytes; item id = it*256 + tid -> chunk id / BM, token id % BM.
    // The loads write LDS directly: lane l of a wave fills bytes [16 l, 16 l + 16) after the wave's base.
    uint32_t xoff[CT];
#pragma unroll
    for (int it = 0; it < CT; it++) {
        const uint32_t id = it * OXB_GEMM_THREADS + tid, c = id / BM, j = id % BM;
        xoff[it] = m0 + j < p.M_pad ? (c * p.M_pad + m0 + j) * 16u : OXB_OOB;
    }
    const uint32_t blk_stride = 16u * p.M_pad * 16u;  // bytes of xh per block
    const uint32_t nblk = p.n_sb * 4u;
    auto stage_x = [&](uint32_t blk, uint4* xs) {
        const uint32_t soff = (blk < nblk ? blk : nblk - 1) * blk_stride;  // past the end: restage the last block
#pragma unroll
        for (int it = 0; it < CT; it++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_ptr_t)(xs + it * OXB_GEMM_THREADS + wave * 64), 16,
                                                     (int)xoff[it], (int)soff, 0, 0);
    };
    auto publish = [&]() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
    // In the blocks that also request the next superblock's weights, those 2 RT loads (codes and scales of each row
    // tile, load_half) are issued after the stage's loads (memory reads return in order) and stay in flight across
    // the barrier: they come from HBM and have until the end of the following block, instead of stalling the whole
    // workgroup at the end of this one.  The count must be exactly the weight loads: one more, and a piece of the
    // token-tile stage may still be on its way when the next block reads it.
    // Measured: three row tiles per wave gain 19 % from it (QKV 6144 x 4096 at 2048 tokens: 105 -> 85 us); with two, four
    // or five tiles the time does not change or gets 3 % worse, so those keep the plain wait.
    constexpr bool KEEP_W = RT == 3;
    auto publish_keep_weights = [&]() {
        if (KEEP_W)
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * RT) : "memory");
        else
            publish();
    };

    HalfRegs<FMT> H[RT][2];
    stage_x(sb0 * 4, xs0);
#pragma unroll
    for (int rt = 0; rt < RT; rt++) {
        load_half<FMT>(H[rt][0], rc, rs, tile_at(rt), (uint32_t)rt < n_valid, p.n_sb, sb0, 0, lane);
        load_half<FMT>(H[rt][1], rc, rs, tile_at(rt), (uint32_t)rt < n_valid, p.n_sb, sb0, 1, lane);
    }
    publish();
    BlockDec bd[RT], bdn[RT];
    v8h A[RT];
#pragma unroll
    for (int rt = 0; rt < RT; rt++) bd[rt] = prepare_block<FMT>(H[rt][0], 0);
    decode_step<FMT, RT>(bd, 0, A);
    const uint32_t boff = g * 4 * BM + r;  // this lane's B operand of step s, token tile ct: xs[boff + s*BM + 16 ct]
    const v8h* x0 = reinterpret_cast<const v8h*>(xs0);
    const v8h* x1 = reinterpret_cast<const v8h*>(xs1);

    for (uint32_t sb = sb0; sb < sb1; sb++) {
        // block 0 of the superblock
        stage_x(sb * 4 + 1, xs1);
#pragma unroll
        for (int rt = 0; rt < RT; rt++) bdn[rt] = prepare_block<FMT>(H[rt][0], 1);
        block_steps<FMT, RT, CT>(x0, A, bd, bdn, acc, boff);
        publish();
        // block 1: half 0 is consumed; reload it for the next superblock
        stage_x(sb * 4 + 2, xs0);
        if (KEEP_W) __builtin_amdgcn_sched_barrier(0);  // the stage's loads first, then the weights (see publish_keep_weights)
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
            bd[rt] = bdn[rt];
            bdn[rt] = prepare_block<FMT>(H[rt][1], 0);
        }
#pragma unroll
        for (int rt = 0; rt < RT; rt++) load_half<FMT>(H[rt][0], rc, rs, tile_at(rt), (uint32_t)rt < n_valid, p.n_sb, sb + 1, 0, lane);
        if (KEEP_W) __builtin_amdgcn_sched_barrier(0);
        block_steps<FMT, RT, CT>(x1, A, bd, bdn, acc, boff);
        publish_keep_weights();
        // block 2
        stage_x(sb * 4 + 3, xs1);
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
            bd[rt] = bdn[rt];
            bdn[rt] = prepare_block<FMT>(H[rt][1], 1);
        }
        block_steps<FMT, RT, CT>(x0, A, bd, bdn, acc, boff);
        publish();
        // block 3: half 1 is consumed; the next block is block 0 of the next superblock (half 0, already reloaded)
        stage_x(sb * 4 + 4, xs0);
        if (KEEP_W) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
            bd[rt] = bdn[rt];
            bdn[rt] = prepare_block<FMT>(H[rt][0], 0);
        }
#pragma unroll
        for (int rt = 0; rt < RT; rt++) load_half<FMT>(H[rt][1], rc, rs, tile_at(rt), (uint32_t)rt < n_valid, p.n_sb, sb + 1, 1, lane);
        if (KEEP_W) __builtin_amdgcn_sched_barrier(0);
        block_steps<FMT, RT, CT>(x1, A, bd, bdn, acc, boff);
        publish_keep_weights();
#pragma unroll
        for (int rt = 0; rt < RT; rt++) bd[rt] = bdn[rt];
    }

    // epilogue: lane holds rows 4g..4g+3 of the row tile for token 16ct + r
    const bool vec_ok = (p.ldy & 3u) == 0;
    if constexpr (RT == 2 || RT == 3) {  // (the counts that are launched in SWIGLU mode)
        if (sw) {
            // The K loop ended behind a barrier with no stage load in flight: both stages are free.  Half of the token tiles at
            // a time the waves leave their factors there (already scaled back by the row's power of two), tile by tile as
            // [tile][ct][lane] float4, gate in the first stage and up in the second, and then take pairs of gate tiles in
            // turn: two tiles are 32 output rows, whole pieces of the next product's operand.
            constexpr int CH = (CT + 1) / 2, TILES = SPLIT ? 2 * RT : 4;  // token tiles a pass, gate tiles of the workgroup
            static_assert((size_t)TILES * CH * 64 * 16 <= sizeof(xs0), "the factors of half the token tiles fit the stages");
            const uint32_t half_tiles = p.n_tiles / 2, g_first = n_g * TILES;
            float4* const gx = reinterpret_cast<float4*>(xs0);
            float4* const ux = reinterpret_cast<float4*>(xs1);
#pragma unroll
            for (int ps = 0; ps < 2; ps++) {
                if (ps) __syncthreads();
#pragma unroll
                for (int ci = 0; ci < CH; ci++) {
                    const int ct = ps * CH + ci;
                    if (ct >= CT) continue;
                    const uint32_t m = m0 + ct * 16 + r;
                    const int e = m < p.M ? row_exp<FMT>(p, m) : 0;
#pragma unroll
                    for (int rt = 0; rt < RT; rt++) {
                        float o[4];
#pragma unroll
                        for (int v = 0; v < 4; v++) o[v] = e == INT32_MIN ? __int_as_float(0x7FC00000) : ldexpf(acc[rt][ct < CT ? ct : 0][v], e);
                        const uint32_t slot = SPLIT ? (wave & 1u) * RT + rt : wave;
                        (( SPLIT ? wave >> 1 : (uint32_t)rt) ? ux : gx)[(slot * CH + ci) * 64 + lane] = make_float4(o[0], o[1], o[2], o[3]);
                    }
                }
                __syncthreads();
                for (uint32_t u = wave; u < TILES / 2 * CH; u += 4) {
                    const uint32_t pr = u / CH, ci = u % CH, ct = ps * CH + ci, m = m0 + ct * 16 + r;
                    if (ct >= CT || m >= p.M) continue;
                    auto four = [&](uint32_t t, uint32_t ln) -> float4 {  // rows 4g..4g+3 of tile 2 pr + t for lane ln = 16 g + r
                        const uint32_t at = ((2 * pr + t) * CH + ci) * 64 + ln;
                        const float4 a = gx[at], b = ux[at];
                        return make_float4(silu_mul(a.x, b.x), silu_mul(a.y, b.y), silu_mul(a.z, b.z), silu_mul(a.w, b.w));
                    };
                    if (p.xh_out) {
                        if (g_first + 2 * pr >= half_tiles) continue;  // (whole blocks of 128 rows: pairs are complete)
                        const OxbOperandOut out = {(_Float16*)p.xh_out, FMT == OXB_FMT_Q1 ? OXB_FMT_Q1 : OXB_FMT_TQ2, p.M_pad, swiglu_shift(p, m)};
                        // lane 16 s + r writes piece s of the 32 rows
                        const uint32_t k0 = (g_first + 2 * pr) * 16;
                        if constexpr (FMT == OXB_FMT_Q1) operand_store8(out, k0 + 4 * g, m, four(0, lane), four(1, lane));
                        else operand_store8(out, k0 + 16 * (g >> 1) + 4 * (g & 1u), m, four(g >> 1, (g & 1u) * 16 + r), four(g >> 1, ((g & 1u) + 2) * 16 + r));
                        continue;
                    }
#pragma unroll
                    for (uint32_t t = 0; t < 2; t++) {
                        const uint32_t tile = g_first + 2 * pr + t, n = tile * 16 + 4 * g;
                        if (tile >= half_tiles) continue;
                        const float4 o = four(t, lane);
                        float* yr = p.y + (size_t)m * p.ldy + n;
                        if (vec_ok) *reinterpret_cast<float4*>(yr) = o;
                        else yr[0] = o.x, yr[1] = o.y, yr[2] = o.z, yr[3] = o.w;
                    }
                }
            }
            if (p.xh_out && n_g == 0) finish_operand(p, m0, min((uint32_t)BM, p.M_pad - m0), tid, OXB_GEMM_THREADS);
            return;
        }
    }
#pragma unroll
    for (int ct = 0; ct < CT; ct++) {
        const uint32_t m = m0 + ct * 16 + r;
        if (m >= p.M) continue;
        const int e = row_exp<FMT>(p, m);
        // with K split over workgroups, slice ks writes its partial sums to plane ks of the workspace
        float* yr = p.ksplit > 1 ? p.part + ((size_t)ks * p.M + m) * p.ldy : p.y + (size_t)m * p.ldy;
        const float* rr = (p.mode == OXB_GEMM_RESIDUAL && p.ksplit == 1) ? p.residual + (size_t)m * p.ldy : nullptr;
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
            if ((uint32_t)rt >= n_valid) continue;
            const uint32_t n = (t0 + rt) * 16 + 4 * g, n_lim = p.n_rows;
            float o[4];
#pragma unroll
            for (int v = 0; v < 4; v++) o[v] = e == INT32_MIN ? __int_as_float(0x7FC00000) : ldexpf(acc[rt][ct][v], e);
            if (vec_ok && n + 3 < n_lim) {
                if (rr) {
                    const float4 q4 = *reinterpret_cast<const float4*>(rr + n);
                    o[0] += q4.x, o[1] += q4.y, o[2] += q4.z, o[3] += q4.w;
                }
                *reinterpret_cast<float4*>(yr + n) = make_float4(o[0], o[1], o[2], o[3]);
            } else {
#pragma unroll
                for (int v = 0; v < 4; v++)
                    if (n + v < n_lim) yr[n + v] = rr ? rr[n + v] + o[v] : o[v];
            }
        }
    }
}

// ---------------------------------------------------------------------------
// GEMM for up to 128 token rows (decode batches, short prompts).  The wide kernel above would spend its time on barriers
// and on MFMAs over padding; here the weights stream once at GEMV-like rates.  A workgroup = 8 waves owns RT row
// tiles; the waves split K (contiguous runs of half superblocks, 256 values), each expands its weights and multiplies them
// with B operands read straight from the packed activations (they stay in L2, no LDS stage, no barrier in the loop),
// requested D - 1 steps ahead; the eight partial sums meet in LDS and are added in wave order.  What bounds it is the
// activations' way into the CU: every workgroup takes in all of them, 16 CT rows of K at 64 bytes a clock.
// Runs of halves and no request past a run against runs of superblocks: 2048 x 6144 (TQ2) at 16 / 77 rows 5.3 -> 4.8 /
// 10.8 -> 10.0 us, 4096 x 4096 at 77 9.3 -> 8.6, 6144 x 4096 at 16 4.8 -> 4.4; the LM head 151936 x 4096 at 16 rows with
// the plan below 53 -> 40, 19456 x 2560 (TQ2) at 16 14.1 -> 8.4.
// Beyond 32 rows against the wide kernel with its 64-token tiles (kernel alone): 4096 x 4096 at 64 / 128 rows 14.9 -> 8.7 /
// 15.5 -> 13.5 us, 6144 x 4096 at 77 15.8 -> 9.7, 4096 x 2048 (TQ2) at 64 / 128 10.5 -> 5.6 / 11.0 -> 8.2.
// ---------------------------------------------------------------------------
#define OXB_GEMM_NARROW_THREADS 512

template <int FMT, int RT, int CT>
__global__ __launch_bounds__(OXB_GEMM_NARROW_THREADS) void gemm_narrow_kernel(const OxbGemmParams p) {
    // The partial sums meet in LDS in passes of PT row tiles: all of them where that takes 64 KB at most, else pairs (48 KB with
    // three token tiles to 112 with seven): in SWIGLU mode a pass holds gate tiles and the up tiles of the same rows.
    constexpr int PT = RT * CT <= 8 || RT == 1 ? RT : 2, NPASS = RT / PT;
    static_assert(RT % PT == 0, "row tiles per pass");
    constexpr int D = CT <= 2 && RT <= 4 ? 8 : 4;  // steps of B operands in registers (16 D CT registers)
    __shared__ float red[8][PT * CT * 4][64];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, r = lane & 15u, g = lane >> 4;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    // Row tiles of this workgroup.  Plain modes: RT consecutive tiles.  SWIGLU mode (the matrix is gate || up,
    // RT even): RT/2 consecutive gate tiles and the up tiles of the same rows, so the epilogue holds both factors.
    const bool sw = p.mode == OXB_GEMM_SWIGLU;
    constexpr uint32_t HP = RT > 1 ? RT / 2 : 1;
    const uint32_t ng = blockIdx.x, ks = blockIdx.y;  // row group, K slice
    const uint32_t t0 = sw ? ng * HP : ng * RT;
    const uint32_t t_lim = sw ? p.n_tiles / 2 : p.n_tiles;
    auto tile_of = [&](int rt) -> uint32_t { return sw ? ((uint32_t)rt < HP ? t0 + rt : p.n_tiles / 2 + t0 + rt - HP) : t0 + rt; };
    auto valid = [&](int rt) -> bool { return sw ? t0 + ((uint32_t)rt % HP) < t_lim : t0 + rt < t_lim; };
    // the wave's run of half superblocks (two blocks each) of the slice: with 2048 values of K every wave has one
    const uint32_t s0 = ks * p.sb_per_split * 2u, s1 = min(s0 + p.sb_per_split * 2u, p.n_sb * 2u);
    const uint32_t per = (s1 - s0 + 7u) / 8u, h0 = s0 + wave * per, h1 = min(h0 + per, s1);
    const __amdgpu_buffer_rsrc_t rc = make_rsrc(p.codes, p.codes_bytes), rs = make_rsrc(p.scales, p.scales_bytes);
    const __amdgpu_buffer_rsrc_t rx = make_rsrc(p.xh, p.xh_bytes);

    v4f acc[RT][CT];
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
        for (int ct = 0; ct < CT; ct++) acc[rt][ct] = (v4f){0.f, 0.f, 0.f, 0.f};

    if (h0 < h1) {
        const uint32_t blk_stride = 16u * p.M_pad * 16u;  // bytes of xh per block
        const uint32_t blk_end = h1 * 2u;
        // B operands of step s, token tile ct of a block: chunk 4g + s, token 16 ct + r.  A ring of D steps, D - 1 ahead.
        v8h B[D][CT];
        // One lane offset; step and block go into the wave-uniform part, the token tile into the instruction's constant.
        const uint32_t b_off = (4u * g * p.M_pad + r) * 16u;
        auto load_b = [&](uint32_t blk, int s, v8h (&dst)[CT]) {
            const uint32_t at = blk < blk_end ? b_off : OXB_OOB_BASE;  // (past the slice)
#pragma unroll
            for (int ct = 0; ct < CT; ct++) dst[ct] = __builtin_bit_cast(v8h, buf_load_b128(rx, at + ct * 256u, blk * blk_stride + s * p.M_pad * 16u));
        };
        // Two halves of weights in registers: a half is requested again, for the one after next, as soon as both its blocks
        // have been prepared (with many row tiles only once the second one has: there is no room for two prepared blocks; nor with
        // seven token tiles of a ternary matrix, 4096 x 4096 at 97 rows 11.9 against 11.5 us, while with eight the two are equal).
        constexpr bool EARLY = RT <= 4 && RT * CT <= 12 && (FMT == OXB_FMT_Q1 || CT != 7);
        HalfRegs<FMT> H[RT][2];
#pragma unroll
        for (int rt = 0; rt < RT; rt++)
#pragma unroll
            for (int hh = 0; hh < 2; hh++) load_half<FMT>(H[rt][hh], rc, rs, tile_of(rt), valid(rt) && h0 + hh < h1, p.n_sb, (h0 + hh) >> 1, (int)((h0 + hh) & 1u), lane);
        // (two blocks in registers: the next block's steps are requested together; else step by step)
        constexpr bool BLOCKS = D == 8;
#pragma unroll
        for (int j = 0; j < (BLOCKS ? 4 : D - 1); j++) load_b(h0 * 2u + (j >> 2), j & 3, B[j]);
        // The two blocks of half superblock h, weights in set hh.  Where the registers allow the last half its own copy (PEEL),
        // nothing is requested past the run: a load that is out of range still takes its turn on the way into the CU, which is
        // what the kernel waits for (with K = 6144 a wave has three halves: 2048 x 6144, TQ2, 16 rows 5.3 -> 4.8 us).
        constexpr bool PEEL = CT <= 6 && (RT * CT <= 8 || (FMT == OXB_FMT_Q1 && (RT * CT <= 10 || CT <= 3)));
        auto half = [&](auto hh_c, auto refill_c, auto last_c, uint32_t h) {
            constexpr int hh = hh_c;
            constexpr bool REFILL = refill_c, LAST = last_c;
            BlockDec bd[EARLY ? 2 : 1][RT];
            auto refill = [&]() {
#pragma unroll
                for (int rt = 0; rt < RT; rt++) load_half<FMT>(H[rt][hh], rc, rs, tile_of(rt), valid(rt) && h + 2 < h1, p.n_sb, (h + 2) >> 1, (int)(h & 1u), lane);
            };
            if (EARLY) {
#pragma unroll
                for (int bi = 0; bi < 2; bi++)
#pragma unroll
                    for (int rt = 0; rt < RT; rt++) bd[EARLY ? bi : 0][rt] = prepare_block<FMT>(H[rt][hh], bi);
                if (REFILL) refill();
            }
#pragma unroll
            for (int bi = 0; bi < 2; bi++) {
                if (BLOCKS && !(LAST && bi)) {
#pragma unroll
                    for (int s = 0; s < 4; s++) load_b(h * 2u + bi + 1, s, B[(4 * (bi + 1) + s) % D]);
                }
                if (!EARLY) {
#pragma unroll
                    for (int rt = 0; rt < RT; rt++) bd[0][rt] = prepare_block<FMT>(H[rt][hh], bi);
                    if (REFILL && bi) refill();
                }
#pragma unroll
                for (int s = 0; s < 4; s++) {
                    const int j = 4 * bi + s, jn = j + D - 1;
                    if (!BLOCKS && !(LAST && jn >= 8)) load_b(h * 2u + (jn >> 2), jn & 3, B[jn % D]);
                    v8h A[RT];
                    decode_step<FMT, RT>(bd[EARLY ? bi : 0], s, A);
#pragma unroll
                    for (int ct = 0; ct < CT; ct++)
#pragma unroll
                        for (int rt = 0; rt < RT; rt++)  // row tiles past the range hold zero weights
                            acc[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[rt], B[j % D][ct], acc[rt][ct], 0, 0, 0);
                }
            }
        };
        constexpr std::integral_constant<int, 0> set0{};
        constexpr std::integral_constant<int, 1> set1{};
        constexpr std::true_type yes{};
        constexpr std::false_type no{};
        uint32_t h = h0;
        for (; h + 2 < (PEEL ? h1 : h1 + 1); h += 2) {
            half(set0, yes, no, h);
            half(set1, yes, no, h + 1);
        }
        if (PEEL && h + 1 < h1) {
            half(set0, no, no, h);
            half(set1, no, yes, h + 1);
        } else if (h < h1)
            half(set0, no, yes, h);
    }
    // row tile behind slot q of pass ps: all tiles in order with a single pass; with pairs, SWIGLU mode takes a gate
    // tile and the up tile of the same rows, the plain modes two neighbours
    auto pass_rt = [&](int ps, int q) -> int { return NPASS == 1 ? q : (sw ? ps + q * (int)HP : ps * PT + q); };
#pragma unroll
    for (int ps = 0; ps < NPASS; ps++) {
    if (ps) __syncthreads();  // the last pass has been read
#pragma unroll
    for (int q = 0; q < PT; q++)
#pragma unroll
        for (int ct = 0; ct < CT; ct++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                // (constant register indices in both arms: the choice is a select, not an indexed array)
                const int rt_sw = NPASS == 1 ? q : ps + q * (int)HP, rt_pl = NPASS == 1 ? q : ps * PT + q;
                red[wave][(q * CT + ct) * 4 + v][lane] = sw ? acc[rt_sw < RT ? rt_sw : 0][ct][v] : acc[rt_pl][ct][v];
            }
    __syncthreads();
    // wave w finishes the accumulator tiles w, w + 8, ...: lane holds rows 4g..4g+3 of row tile rt for token 16ct + r
    const bool vec_ok = (p.ldy & 3u) == 0;
    auto total = [&](uint32_t idx, float (&o)[4], int e) {
#pragma unroll
        for (int v = 0; v < 4; v++) {
            float a = red[0][idx * 4 + v][lane];
#pragma unroll
            for (int w = 1; w < 8; w++) a += red[w][idx * 4 + v][lane];
            o[v] = e == INT32_MIN ? __int_as_float(0x7FC00000) : ldexpf(a, e);
        }
    };
    // slots of a pass that hold output rows: all of them; in SWIGLU mode the gate slots (half of a single pass, slot 0 of a pair)
    const uint32_t q_out = sw ? (NPASS == 1 ? HP : 1u) : (uint32_t)PT, q_up = NPASS == 1 ? HP : 1u;
    for (uint32_t idx = wave; idx < q_out * CT; idx += 8) {
        const uint32_t q = idx / CT, ct = idx % CT, m = ct * 16 + r;
        const uint32_t rt = (uint32_t)pass_rt(ps, (int)q);
        if (!valid((int)rt) || m >= p.M) continue;
        const int e = row_exp<FMT>(p, m);
        float o[4];
        total(idx, o, e);
        if (sw) {  // y[m][row] = silu(gate) * up, rows counted within the gate half
            float u[4];
            total((q + q_up) * CT + ct, u, e);
#pragma unroll
            for (int v = 0; v < 4; v++) o[v] = silu_mul(o[v], u[v]);
            if (p.xh_out) {
                operand_store4({(_Float16*)p.xh_out, FMT == OXB_FMT_Q1 ? OXB_FMT_Q1 : OXB_FMT_TQ2, p.M_pad, swiglu_shift(p, m)}, (t0 + rt) * 16 + 4 * g, m, o[0], o[1], o[2], o[3]);
                continue;
            }
        }
        // (with K split over workgroups, slice ks writes its partial sums to plane ks of the workspace)
        float* yr = p.ksplit > 1 ? p.part + ((size_t)ks * p.M + m) * p.ldy : p.y + (size_t)m * p.ldy;
        const float* rr = p.mode == OXB_GEMM_RESIDUAL && p.ksplit == 1 ? p.residual + (size_t)m * p.ldy : nullptr;
        const uint32_t n = (t0 + rt) * 16 + 4 * g, n_lim = sw ? p.n_rows / 2 : p.n_rows;
        if (vec_ok && n + 3 < n_lim) {
            if (rr) {
                const float4 q4 = *reinterpret_cast<const float4*>(rr + n);
                o[0] += q4.x, o[1] += q4.y, o[2] += q4.z, o[3] += q4.w;
            }
            *reinterpret_cast<float4*>(yr + n) = make_float4(o[0], o[1], o[2], o[3]);
        } else {
#pragma unroll
            for (int v = 0; v < 4; v++)
                if (n + v < n_lim) yr[n + v] = rr ? rr[n + v] + o[v] : o[v];
        }
    }
    }
    if (sw && p.xh_out && ng == 0) finish_operand(p, 0, p.M_pad, tid, OXB_GEMM_NARROW_THREADS);
}

// ---------------------------------------------------------------------------
// The same for matrices of many rows (an LM head) and 17 to 32 token rows, K up to 4096.  With a workgroup for each group of row tiles the
// kernel above takes all of the activations in again and waits for its first weights every time, one workgroup on a CU: 11 us
// each.  Here one workgroup per CU stays: a wave keeps the activations of its superblock in registers (64 for each 16 token rows) and its
// share of the tiles streams past in pairs, RING tiles ahead.  The waves' sums of a pair meet in LDS as [token][row], two pairs' worth,
// a barrier for each; every thread adds up a few outputs and stores them, 16 rows of a token side by side.  Reads of the sums
// one behind the other cost 5 us of 56, stores in branches, whose number nobody knows where the next weights are waited for, 3.
// us, 32 rows, kernel above / this one: Q1 151936 x 4096 65.4 / 50.7, x 2048 46.2 / 34.8, TQ2 84.2 / 57.3 and 52.3 / 38.3;
// 65536 x 2560 25.3 / 21.9 and 33.7 / 25.5.
// ---------------------------------------------------------------------------
template <int FMT>
__global__ __launch_bounds__(OXB_GEMM_NARROW_THREADS) void gemm_tall_kernel(const OxbGemmParams p) {
    constexpr int CT = 2, RING = 4;  // token tiles; row tiles in flight
    __shared__ __attribute__((aligned(16))) float red[2][8][2][CT * 256];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, r = lane & 15u, g = lane >> 4, threads = blockDim.x, S = threads >> 6;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));  // its superblock
    const uint32_t t_begin = blockIdx.x * p.tpw, t_end = min(t_begin + p.tpw, p.n_tiles);
    const __amdgpu_buffer_rsrc_t rc = make_rsrc(p.codes, p.codes_bytes), rs = make_rsrc(p.scales, p.scales_bytes);
    const __amdgpu_buffer_rsrc_t rx = make_rsrc(p.xh, p.xh_bytes);
    const __amdgpu_buffer_rsrc_t ry = make_rsrc(p.y, ((p.M - 1) * p.ldy + p.n_rows) * 4u);
    const uint32_t b_off = (4u * g * p.M_pad + r) * 16u, blk_stride = 16u * p.M_pad * 16u;
    v8h B[4][4][CT];  // [block][step][token tile]
#pragma unroll
    for (int b = 0; b < 4; b++)
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int ct = 0; ct < CT; ct++) B[b][s][ct] = __builtin_bit_cast(v8h, buf_load_b128(rx, b_off + ct * 256u, (wave * 4u + b) * blk_stride + s * p.M_pad * 16u));
    HalfRegs<FMT> H[RING][2];
    auto request = [&](HalfRegs<FMT> (&h)[2], uint32_t t) __attribute__((always_inline)) {
#pragma unroll
        for (int hh = 0; hh < 2; hh++) load_half<FMT>(h[hh], rc, rs, t, t < t_end, p.n_sb, wave, hh, lane);
    };
#pragma unroll
    for (int i = 0; i < RING; i++) request(H[i], t_begin + i);
    // the outputs of this thread: value o = tid + i threads of a tile, row o % 16 of token o / 16
    int e[CT];
#pragma unroll
    for (int i = 0; i < CT; i++) {
        const uint32_t m = (tid + i * threads) / 16u;
        e[i] = m < p.M ? row_exp<FMT>(p, m) : 0;
    }
    for (uint32_t t0 = t_begin, pair = 0; t0 < t_end; t0 += RING) {
#pragma unroll
        for (int i = 0; i < RING; i += 2, pair++) {
            const uint32_t t = t0 + i;
            if (t >= t_end) break;  // (the same for all waves)
            v4f acc[2][CT];
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int ct = 0; ct < CT; ct++) acc[j][ct] = (v4f){0.f, 0.f, 0.f, 0.f};
            // a step's weights are expanded while the products of the one before run: one product, then its share of the expansion
            BlockDec bd[2] = {prepare_block<FMT>(H[i][0], 0), prepare_block<FMT>(H[i + 1][0], 0)};
            v8h A[2];
            decode_step<FMT, 2>(bd, 0, A);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int st = 0; st < 16; st++) {
                const int b = st >> 2, s = st & 3;
                v8h An[2];
                if (s == 3 && b < 3) {
                    bd[0] = prepare_block<FMT>(H[i][(b + 1) >> 1], (b + 1) & 1);
                    bd[1] = prepare_block<FMT>(H[i + 1][(b + 1) >> 1], (b + 1) & 1);
                }
                if (st < 15) decode_step<FMT, 2>(bd, (s + 1) & 3, An);
#pragma unroll
                for (int ct = 0; ct < CT; ct++)
#pragma unroll
                    for (int j = 0; j < 2; j++) acc[j][ct] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[j], B[b][s][ct], acc[j][ct], 0, 0, 0);
                if (st < 15) A[0] = An[0], A[1] = An[1];
#pragma unroll
                for (int k = 0; k < 2 * CT; k++) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, (FMT == OXB_FMT_Q1 ? 16 : 24) / (2 * CT), 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            request(H[i], t + RING);
            request(H[i + 1], t + RING + 1);
            float(*const mine)[CT * 256] = red[pair & 1u][wave];
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int ct = 0; ct < CT; ct++) *reinterpret_cast<v4f*>(&mine[j][ct * 256 + r * 16 + 4 * g]) = acc[j][ct];
            // (one barrier a pair: a wave writes the pair after next here only when all have added this one up)
            lds_barrier();
            // (all the reads before the first sum; a wave that does not exist adds nothing)
            float v[2][CT][8];
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int k = 0; k < CT; k++)
#pragma unroll
                    for (uint32_t w = 0; w < 8; w++) v[j][k][w] = red[pair & 1u][w < S ? w : 0u][j][min(tid + k * threads, CT * 256u - 1)];
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int k = 0; k < CT; k++) {
                    const uint32_t o = tid + k * threads, m = o / 16u, n = (t + j) * 16u + (o & 15u);
                    float a = v[j][k][0];
#pragma unroll
                    for (uint32_t w = 1; w < 8; w++) a += w < S ? v[j][k][w] : 0.f;
                    a = e[k] == INT32_MIN ? __int_as_float(0x7FC00000) : ldexpf(a, e[k]);
                    // (no branch: how many stores are under way is known where the next weights are waited for)
                    const bool there = m < p.M && n < p.n_rows && t + j < t_end;
                    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(a), ry, (int)(there ? (m * p.ldy + n) * 4u : OXB_OOB_BASE), 0, 0);
                }
        }
    }
}

// y = (residual +) the K slices' partial sums, added in slice order (deterministic): where no pack of the result follows.
__global__ __launch_bounds__(256) void gemm_splitk_reduce_kernel(const float* __restrict__ part, uint32_t ksplit, size_t plane,
                                                                  const float* __restrict__ residual, float* __restrict__ y,
                                                                  size_t n4) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n4) return;
    float4 a = reinterpret_cast<const float4*>(part)[i];
    for (uint32_t s = 1; s < ksplit; s++) {
        const float4 b = reinterpret_cast<const float4*>(part + s * plane)[i];
        a.x += b.x, a.y += b.y, a.z += b.z, a.w += b.w;
    }
    if (residual) {
        const float4 r = reinterpret_cast<const float4*>(residual)[i];
        a.x += r.x, a.y += r.y, a.z += r.z, a.w += r.w;
    }
    reinterpret_cast<float4*>(y)[i] = a;
}

// The square of the 2-norm of each row of a tile (weights are +-d or 0: with zeros among them a bound), in threads 0 .. 15: the sum
// over its blocks of the scale's square times weight(block), 128 where all inputs count alike.
template <class F>
__device__ __forceinline__ float tile_row_norms2(const uint16_t* __restrict__ scales, uint32_t n_sb, uint32_t tile, float (&part)[16][17], F weight) {
    const uint32_t tid = threadIdx.x, r = tid & 15u, j = tid >> 4;
    const _Float16* s = reinterpret_cast<const _Float16*>(scales) + (size_t)tile * n_sb * 64u + r * 4u;
    float a = 0.f;
    for (uint32_t sb = j; sb < n_sb; sb += 16)
        for (uint32_t q = 0; q < 4; q++) {
            const float d = (float)s[sb * 64u + q];
            a = fmaf(d * d, weight(sb * 4u + q), a);
        }
    __syncthreads();
    part[j][r] = a;
    __syncthreads();
    a = 0.f;
    if (tid < 16)
        for (int i = 0; i < 16; i++) a += part[i][tid];
    return a;
}
__device__ __forceinline__ float norm_or_inf(float n) { return n == n ? n : __builtin_inff(); }

__global__ __launch_bounds__(256) void pair_norms_kernel(const uint16_t* __restrict__ scales, uint32_t n_sb, uint32_t pair_tiles, float* __restrict__ out) {
    __shared__ float part[16][17];
    auto all = [](uint32_t) -> float { return 128.f; };
    const float a = tile_row_norms2(scales, n_sb, blockIdx.x, part, all), b = tile_row_norms2(scales, n_sb, blockIdx.x + pair_tiles, part, all);
    if (threadIdx.x < 16) out[blockIdx.x * 16u + threadIdx.x] = norm_or_inf(sqrtf(a) * sqrtf(b));
}

__global__ __launch_bounds__(256) void weighted_norms_kernel(const uint16_t* __restrict__ scales, uint32_t n_sb, uint32_t t0, const float* __restrict__ w,
                                                             uint32_t k, float typical, float* __restrict__ out) {
    __shared__ float part[16][17];
    for (uint32_t f = 0; f < 2; f++) {
        const float most = f ? typical : __builtin_inff();
        const float a = tile_row_norms2(scales, n_sb, t0 + blockIdx.x, part, [&](uint32_t blk) -> float {
            float s = 0.f;
            for (uint32_t i = blk * 128u; i < blk * 128u + 128u && i < k; i++) {
                const float v = fabsf(w[i]) > most ? most : w[i];
                s = fmaf(v, v, s);
            }
            return s;
        });
        if (threadIdx.x < 16) out[(f * gridDim.x + blockIdx.x) * 16u + threadIdx.x] = norm_or_inf(sqrtf(a));
    }
}

// ---------------------------------------------------------------------------
// Host-side launchers.
// ---------------------------------------------------------------------------
hipError_t oxb_launch_pair_norms(const uint16_t* d_scales, uint32_t n_sb, uint32_t n, float* d_out, hipStream_t st) {
    if ((n & 15u) != 0 || n == 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(pair_norms_kernel, dim3(n / 16), dim3(256), 0, st, d_scales, n_sb, n / 16, d_out);
    return hipGetLastError();
}

hipError_t oxb_launch_weighted_norms(const uint16_t* d_scales, uint32_t n_sb, uint32_t row0, uint32_t n, const float* d_w, uint32_t k, float typical, float* d_out, hipStream_t st) {
    if (((row0 | n) & 15u) != 0 || n == 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(weighted_norms_kernel, dim3(n / 16), dim3(256), 0, st, d_scales, n_sb, row0 / 16, d_w, k, typical, d_out);
    return hipGetLastError();
}

size_t oxb_xh_bytes(uint32_t k, uint32_t M) {
    const size_t nblk_pad = ((k + 511u) / 512u) * 4u, M_pad = (M + 15u) / 16u * 16u;
    return nblk_pad * 16 * M_pad * 16;
}

#define OXB_PACK_ROWS_MAX 64  // up to this many token rows (of at most 16384 values) the one-launch packer is used

template <int OP, bool SUM>
static void launch_pack_op(int fmt, float* d_x, const float* d_w, uint32_t ldx, uint32_t k, uint32_t M, uint32_t M_pad,
                           uint32_t nblk_pad, float eps, float* d_rowmul, uint32_t* d_xh, int32_t* d_xsh, OxbPackNorm norm, const OxbPackSum& sum, hipStream_t st) {
    const uint32_t per_thread = (nblk_pad * 16 + 255) / 256;  // items of a row per thread of the one-launch packer
    if (M <= OXB_PACK_ROWS_MAX && per_thread <= 8) {
#define OXB_ROWS_CASE(NI)                                                                                                      \
    if (per_thread <= NI) {                                                                                                    \
        if (fmt == OXB_FMT_Q1)                                                                                                 \
            hipLaunchKernelGGL((xh_pack_rows_kernel<OXB_FMT_Q1, OP, NI, SUM>), dim3(M_pad), dim3(256), 0, st, d_x, d_w, ldx, k, eps, M, \
                               M_pad, nblk_pad, d_xsh, norm, reinterpret_cast<uint4*>(d_xh), sum);                                   \
        else                                                                                                                   \
            hipLaunchKernelGGL((xh_pack_rows_kernel<OXB_FMT_TQ2, OP, NI, SUM>), dim3(M_pad), dim3(256), 0, st, d_x, d_w, ldx, k, eps, M, \
                               M_pad, nblk_pad, d_xsh, norm, reinterpret_cast<uint4*>(d_xh), sum);                                   \
        return;                                                                                                                \
    }
        OXB_ROWS_CASE(1) OXB_ROWS_CASE(2) OXB_ROWS_CASE(4)
        if constexpr (!SUM) { OXB_ROWS_CASE(6) OXB_ROWS_CASE(8) }
#undef OXB_ROWS_CASE
    }
    // Four rows per workgroup, two where four would leave half the CUs idle; eight for long rows where each of 256 CUs has
    // a workgroup all the same (2048 rows of 12288: 25 us against 28 with four and 36 with two; of 4096: 11, 10 and 12).
    // Long rows with sums to add: two, or the registers of the planes spill (600 rows of 10240 33 us against 60, 1700 of 8320
    // 60 against 100).
    const uint32_t rpw = OP == OXB_PACK_IDENT && k > 8192 && M_pad >= 2048 ? 8 : M_pad >= 512 && !(SUM && k > 8192) ? 4 : 2, per_lane = (nblk_pad * 4 * rpw + 63) / 64;  // pieces of four values per lane
#define OXB_WIDE_CASE(RPW, NI)                                                                                                     \
    if (rpw == RPW && per_lane <= NI) {                                                                                            \
        if (fmt == OXB_FMT_Q1)                                                                                                     \
            hipLaunchKernelGGL((xh_pack_wide_kernel<OXB_FMT_Q1, OP, RPW, NI, SUM>), dim3(M_pad / RPW), dim3(512), 0, st, d_x, d_w, ldx, \
                               k, eps, M, M_pad, nblk_pad, d_xsh, norm, reinterpret_cast<uint4*>(d_xh), sum);                            \
        else                                                                                                                       \
            hipLaunchKernelGGL((xh_pack_wide_kernel<OXB_FMT_TQ2, OP, RPW, NI, SUM>), dim3(M_pad / RPW), dim3(512), 0, st, d_x, d_w, ldx, \
                               k, eps, M, M_pad, nblk_pad, d_xsh, norm, reinterpret_cast<uint4*>(d_xh), sum);                            \
        return;                                                                                                                    \
    }
    OXB_WIDE_CASE(4, 8) OXB_WIDE_CASE(4, 16)
    if constexpr (!SUM) { OXB_WIDE_CASE(4, 24) }
    OXB_WIDE_CASE(2, 4) OXB_WIDE_CASE(2, 8) OXB_WIDE_CASE(2, 12)
    if constexpr (OP == OXB_PACK_IDENT) { OXB_WIDE_CASE(8, 48) }
    // (rows of more than 12288 values take two launches)
#undef OXB_WIDE_CASE
    if constexpr (!SUM) {
        hipLaunchKernelGGL(row_stats_kernel<OP>, dim3(M), dim3(256), 0, st, d_x, d_w, ldx, k, eps, d_rowmul, d_xsh, norm);
        const dim3 grid(M_pad / 16, nblk_pad < 16 ? nblk_pad : 16);
        if (fmt == OXB_FMT_Q1)
            hipLaunchKernelGGL((xh_pack_kernel<OXB_FMT_Q1, OP>), grid, dim3(256), 0, st, d_x, d_w, ldx, k, M, M_pad, nblk_pad, d_rowmul,
                               reinterpret_cast<uint4*>(d_xh));
        else
            hipLaunchKernelGGL((xh_pack_kernel<OXB_FMT_TQ2, OP>), grid, dim3(256), 0, st, d_x, d_w, ldx, k, M, M_pad, nblk_pad, d_rowmul,
                               reinterpret_cast<uint4*>(d_xh));
    }
}

bool oxb_pack_can_sum(uint32_t k, uint32_t M) { return k <= (M <= OXB_PACK_ROWS_MAX ? 8192u : 12288u) && (k % OXB_QK) == 0; }

hipError_t oxb_launch_xh_pack(int fmt, int op, const float* d_x, const float* d_w, uint32_t ldx, uint32_t k, float eps,
                              uint32_t M, float* d_rowmul, uint32_t* d_xh, int32_t* d_xsh, hipStream_t st, const OxbPackSum* sum, OxbPackNorm norm) {
    if (M == 0 || k == 0 || (k % OXB_QK) != 0 || (ldx & 3u) != 0) return hipErrorInvalidValue;
    if (op == OXB_PACK_RMSNORM && !d_w) return hipErrorInvalidValue;
    const uint32_t nblk_pad = ((k + 511u) / 512u) * 4u, M_pad = (M + 15u) / 16u * 16u;
    if (oxb_xh_bytes(k, M) >= 0xFFFFFFF0ull) return hipErrorInvalidValue;
    float* x = const_cast<float*>(d_x);  // (written with `sum` only)
    if (sum && sum->n > 1) {
        if (op != OXB_PACK_RMSNORM || !oxb_pack_can_sum(k, M) || ldx != k) return hipErrorInvalidValue;
        launch_pack_op<OXB_PACK_RMSNORM, true>(fmt, x, d_w, ldx, k, M, M_pad, nblk_pad, eps, d_rowmul, d_xh, d_xsh, norm, *sum, st);
        return hipGetLastError();
    }
    const OxbPackSum none = {nullptr, 0, 0};
    switch (op) {
        case OXB_PACK_IDENT: launch_pack_op<OXB_PACK_IDENT, false>(fmt, x, d_w, ldx, k, M, M_pad, nblk_pad, eps, d_rowmul, d_xh, d_xsh, norm, none, st); break;
        case OXB_PACK_RMSNORM: launch_pack_op<OXB_PACK_RMSNORM, false>(fmt, x, d_w, ldx, k, M, M_pad, nblk_pad, eps, d_rowmul, d_xh, d_xsh, norm, none, st); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <int FMT, int RT, int CT>
static hipError_t launch_gemm_case(const OxbGemmParams& p, uint32_t grid, hipStream_t st) {
    hipLaunchKernelGGL((gemm_mfma_kernel<FMT, RT, CT>), dim3(grid), dim3(OXB_GEMM_THREADS), 0, st, p);
    return hipGetLastError();
}

// Time of a wide plan in us, from 19 000 measured (shape, tokens, plan) triples - both formats, 1280 .. 24576 rows, K 1280 ..
// 12288, 33 .. 2048 tokens - whose best plan it names within 2 % on average (the rule before it, 128-token tiles by rounds
// of workgroups: 12 %).  Per 128-weight block a workgroup alone on its CU needs `lone`, a latency; workgroups that share
// one need `busy` each, a rate.  More tokens per tile amortise the expansion of the weights, more row tiles the reading of
// the token tile out of LDS; small tiles make more workgroups and less padding.  (The ternary times here and in narrow_cost are those of
// four instructions for two weights; with three (BlockDec) a plan takes up to 10 % less, 4 % on average, and the choice was not fitted again.)
static float wide_cost(bool tq2, const OxbGemmParams& p, const OxbGemmPlan& g, uint32_t n_cus) {
    // [format][ct = 4, 5, 8][rt - 1]; rt = 5 goes with ct = 8 only, rt = 1 not with it (smaller token tiles always beat it)
    static const float lone_us[2][3][5] = {{{0.34f, 0.50f, 0.68f, 0.82f}, {0.40f, 0.59f, 0.81f, 0.96f}, {0.66f, 0.86f, 1.18f, 1.42f, 1.69f}},
                                           {{0.39f, 0.59f, 0.85f, 1.05f}, {0.45f, 0.70f, 0.96f, 1.19f}, {0.69f, 0.99f, 1.30f, 1.60f, 1.83f}}};
    static const float busy_us[2][3][5] = {{{0.25f, 0.41f, 0.58f, 0.77f}, {0.31f, 0.51f, 0.70f, 0.92f}, {0.54f, 0.83f, 1.09f, 1.42f, 1.69f}},
                                           {{0.28f, 0.49f, 0.68f, 0.94f}, {0.34f, 0.60f, 0.84f, 1.06f}, {0.57f, 0.85f, 1.17f, 1.60f, 1.83f}}};
    static const float long_k_us[3][5] = {{0.14f, 0.05f, 0.03f, 0.02f}, {0.14f, 0.05f, 0.03f, 0.02f}, {0.03f, 0.03f}};  // on top of lone, K > 4608: the token panel leaves L2
    static const uint32_t resident[3][5] = {{5, 4, 3, 2}, {4, 3, 3, 2}, {2, 2, 2, 1, 1}};  // workgroups per CU (registers, LDS)
    const uint32_t ci = g.ct == 4 ? 0 : g.ct == 5 ? 1 : 2, ri = g.rt - 1, R = resident[ci][ri];
    const uint32_t n_mt = (p.M + 16 * g.ct - 1) / (16 * g.ct), n_ng = (p.n_tiles + g.tpw - 1) / g.tpw;
    const uint32_t q = (n_ng * n_mt * g.ksplit + n_cus - 1) / n_cus;  // workgroups on the CU that gets most
    const float lone = lone_us[tq2][ci][ri] + (p.n_sb > 9 ? long_k_us[ci][ri] : 0.f), busy = busy_us[tq2][ci][ri];
    auto round = [&](uint32_t w) { const float b = w * busy; return w == 0 ? 0.f : b > lone ? b : lone; };
    const float us = 4.4f + 4.f * g.sb_per_split * ((float)(q / R) * round(R) + round(q % R)) + 0.158f * q * g.rt * g.ct;
    // a K split writes its partial sums and adds them in a launch of its own, or leaves them to the next pack
    return g.ksplit > 1 ? 1.04f * (us + (p.sum_later ? 0.6f : 2.2f) + 0.73e-6f * g.ksplit * p.M * (float)p.n_rows) : us;
}

// Time of a narrow plan in us, from 1900 measured (shape, tokens, plan) triples - both formats, 1280 .. 151936 rows, K 1280 ..
// 12288, 8 .. 128 tokens; rms 4 %; the plan it names is within 1 % of the best on average.  A workgroup's eight waves have a
// latency (a round trip per half superblock, longer with more row tiles in flight); workgroups that share a CU queue for what
// each takes in: all of the packed activations and its weights.  What counts is the fullest CU: 384 workgroups of one tile
// leave half the CUs with two (QKV 6144 x 4096, 32 rows: 8.2 us against 5.9 as 192 workgroups of two tiles), six tiles make
// gate || up 24576 x 4096 one workgroup per CU (11.8 us; as 384 of four: 16.6), while the LM head's 9496 tiles run best in
// fours at 16 rows, two workgroups resident (39.6 us against 53 in sixes).
static float narrow_cost(bool tq2, const OxbGemmParams& p, uint32_t rt, uint32_t ksplit, uint32_t n_cus) {
    static const uint8_t resident[2][2][2] = {{{4, 2}, {2, 1}}, {{3, 2}, {2, 1}}};  // [format][rt = 1, 2][ct = 1, 2]: workgroups per CU (registers); else one
    const uint32_t ct = (p.M + 15) / 16, R = rt > 2 || ct > 2 ? 1 : resident[tq2][rt - 1][ct - 1], spk = (p.n_sb + ksplit - 1) / ksplit;
    const uint32_t wgs = (p.mode == OXB_GEMM_SWIGLU ? (p.n_tiles / 2 + rt / 2 - 1) / (rt / 2) : (p.n_tiles + rt - 1) / rt) * ksplit;
    const uint32_t q = (wgs + n_cus - 1) / n_cus;  // workgroups on the CU that gets most
    const float w_rt = rt * (tq2 ? 1.48f : 1.f), busy = spk * (0.096f * ct + 0.035f * w_rt + 0.012f * rt * ct) + 0.119f * rt * ct;
    const float lat = 0.18f + (float)((2 * spk + 7) / 8) * 0.192f * w_rt;
    return 1.91f + (float)(q / R) * (lat + R * busy) + (q % R ? lat + (q % R) * busy : 0.f);
}

// 16 row tiles and more for every CU, two token tiles and a wave for every superblock (four to eight).  With half the rows, 32768, the two
// kernels are about equal (Q1 x 4096 15.2 / 15.6 us, x 2048 10.7 / 10.9, TQ2 19.6 / 17.8 and 12.2 / 12.1), with one token tile often the
// other is faster (Q1 65536 x 2560 16.4 / 17.8 us, 151936 x 4096 42.6 / 41.5).
static bool tall(const OxbGemmParams& p, uint32_t n_cus) {
    return p.mode == OXB_GEMM_STORE && p.M > 16 && p.M <= 32 && p.n_sb >= 4 && p.n_sb <= 8 && p.n_tiles >= 16 * n_cus &&
           (uint64_t)p.M * p.ldy * 4 < OXB_OOB_BASE;
}

// The narrow kernel up to OXB_GEMM_NARROW_MAX_M token rows (the wide one would spend its time on barriers and padding),
// the cheaper of the two up to 128, the wide one beyond.
OxbGemmPlan oxb_gemm_plan(int fmt, const OxbGemmParams& p, uint32_t n_cus) {
    const bool tq2 = fmt == OXB_FMT_TQ2, sw = p.mode == OXB_GEMM_SWIGLU;
    OxbGemmPlan best = {true, 0, 0, 0, 1, p.n_sb};
    float best_us = 1e30f;
    if (tall(p, n_cus)) {
        best.ct = (p.M + 15) / 16, best.tpw = (p.n_tiles + n_cus - 1) / n_cus;
        return best;
    }
    if (p.M <= 128) {
        // row tiles per workgroup: as many as the registers hold next to the token tiles (six: Q1 only), two or more with SWIGLU
        static const uint32_t choices[4] = {1, 2, 4, 6};
        const uint32_t ct = best.ct = (p.M + 15) / 16, most = ct <= 2 && !tq2 ? 6 : ct <= 4 ? 4 : ct <= 7 ? 2 : 1;
        for (uint32_t rt : choices) {
            if (rt > most || (sw && rt == 1)) continue;
            // K in slices where the next pack adds them anyway: with few row tiles they fill the chip, and a workgroup takes in
            // its slice of the activations only (4096 x 12288, 32 rows: 9.6 us whole, 7.7 in four slices of 64 workgroups)
            for (uint32_t ks = 1; ks <= (p.sum_later ? 4u : 1u); ks++) {
                const uint32_t spk = (p.n_sb + ks - 1) / ks;
                if ((p.n_sb + spk - 1) / spk != ks || (ks > 1 && (p.n_tiles + rt - 1) / rt * ks > 2 * n_cus)) continue;
                const float us = narrow_cost(tq2, p, rt, ks, n_cus) + (ks > 1 ? 0.3f + 0.3f * ks : 0.f);
                if (us < best_us) best_us = us, best.rt = rt, best.ksplit = ks, best.sb_per_split = spk;
            }
        }
        if (p.M <= OXB_GEMM_NARROW_MAX_M) return best;
    }
    static const uint32_t cts[3] = {8, 5, 4}, splits[5] = {1, 2, 3, 4, 6};
    const bool can_split = (p.ldy & 3u) == 0 && !sw && !p.no_split;  // (the SwiGLU epilogue is not linear)
    for (uint32_t ks : splits) {
        if (ks > (can_split ? p.n_sb : 1u)) break;
        const uint32_t spk = (p.n_sb + ks - 1) / ks;
        if ((p.n_sb + spk - 1) / spk != ks) continue;  // same slices as a smaller count
        for (uint32_t ct : cts)
            for (uint32_t rt = ct == 8 ? 2 : 1; rt <= (ct == 8 ? 5u : 4u); rt++) {
                if (sw && rt != 2 && rt != 3) continue;  // a gate and an up tile per wave, or three tiles of either kind
                const OxbGemmPlan g = {false, rt, 4 * rt, ct, ks, spk};
                const float us = wide_cost(tq2, p, g, n_cus);
                if (us < best_us) best_us = us, best = g;
            }
    }
    return best;
}

template <int FMT, int RT, int CT>
static hipError_t launch_narrow_case(const OxbGemmParams& p, hipStream_t st) {
    hipLaunchKernelGGL((gemm_narrow_kernel<FMT, RT, CT>), dim3(p.n_ng, p.ksplit), dim3(OXB_GEMM_NARROW_THREADS), 0, st, p);
    return hipGetLastError();
}

// (fmt: OXB_FMT_* or GEMM_TQ2_LOUD)
static hipError_t launch_gemm_narrow(int fmt, OxbGemmParams p, uint32_t rt, hipStream_t st) {
    p.n_ng = p.mode == OXB_GEMM_SWIGLU ? (p.n_tiles / 2 + rt / 2 - 1) / (rt > 1 ? rt / 2 : 1) : (p.n_tiles + rt - 1) / rt;
    const uint32_t ct = p.M_pad / 16;
#define OXB_NARROW_CASE(F, R, C) \
    if (fmt == F && rt == R && ct == C) return launch_narrow_case<F, R, C>(p, st);
#define OXB_NARROW_CASES(R, C) OXB_NARROW_CASE(OXB_FMT_Q1, R, C) OXB_NARROW_CASE(OXB_FMT_TQ2, R, C) OXB_NARROW_CASE(GEMM_TQ2_LOUD, R, C)
    OXB_NARROW_CASES(1, 1) OXB_NARROW_CASES(2, 1) OXB_NARROW_CASES(4, 1) OXB_NARROW_CASE(OXB_FMT_Q1, 6, 1)
    OXB_NARROW_CASES(1, 2) OXB_NARROW_CASES(2, 2) OXB_NARROW_CASES(4, 2) OXB_NARROW_CASE(OXB_FMT_Q1, 6, 2)
    OXB_NARROW_CASES(1, 3) OXB_NARROW_CASES(2, 3) OXB_NARROW_CASES(4, 3)
    OXB_NARROW_CASES(1, 4) OXB_NARROW_CASES(2, 4) OXB_NARROW_CASES(4, 4)
    OXB_NARROW_CASES(1, 5) OXB_NARROW_CASES(2, 5)
    OXB_NARROW_CASES(1, 6) OXB_NARROW_CASES(2, 6)
    OXB_NARROW_CASES(1, 7) OXB_NARROW_CASES(2, 7)
    OXB_NARROW_CASES(1, 8)
#undef OXB_NARROW_CASES
#undef OXB_NARROW_CASE
    return hipErrorInvalidValue;
}


uint32_t oxb_gemm_ksplit(int fmt, const OxbGemmParams& p, uint32_t n_cus) {
    if (p.M == 0 || p.n_rows == 0 || p.n_sb == 0) return 1;
    return oxb_gemm_plan(fmt, p, n_cus).ksplit;
}

hipError_t oxb_launch_gemm(int fmt, OxbGemmParams p, uint32_t n_cus, hipStream_t st) {
    if (p.M == 0 || p.n_rows == 0) return hipSuccess;
    if (p.n_sb == 0 || (uint64_t)p.n_tiles * p.n_sb * 2048ull >= 0xFFFFFFF0ull) return hipErrorInvalidValue;
    if (p.mode == OXB_GEMM_SWIGLU && (p.n_rows & 31u) != 0) return hipErrorInvalidValue;  // whole gate and up row tiles
    if (p.xh_out && (p.mode != OXB_GEMM_SWIGLU || (p.n_rows & 255u) != 0 || !p.xsh_out || !p.norm2)) return hipErrorInvalidValue;  // whole blocks
    p.M_pad = (p.M + 15u) / 16u * 16u;
    const OxbGemmPlan plan = oxb_gemm_plan(fmt, p, n_cus);
    p.ksplit = plan.ksplit;
    p.sb_per_split = plan.sb_per_split;
    if (p.ksplit > 1 && !p.part) return hipErrorInvalidValue;
    if (p.loud && fmt == OXB_FMT_TQ2) fmt = GEMM_TQ2_LOUD;
    if (plan.narrow && plan.rt == 0) {
        p.tpw = plan.tpw;
        const dim3 grid((p.n_tiles + p.tpw - 1) / p.tpw), block(64 * p.n_sb);
        if (fmt == OXB_FMT_Q1) hipLaunchKernelGGL(gemm_tall_kernel<OXB_FMT_Q1>, grid, block, 0, st, p);
        else if (fmt == OXB_FMT_TQ2) hipLaunchKernelGGL(gemm_tall_kernel<OXB_FMT_TQ2>, grid, block, 0, st, p);
        else hipLaunchKernelGGL(gemm_tall_kernel<GEMM_TQ2_LOUD>, grid, block, 0, st, p);
        return hipGetLastError();
    }
    if (plan.narrow) return launch_gemm_narrow(fmt, p, plan.rt, st);
    p.n_mt = (p.M + 16 * plan.ct - 1) / (16 * plan.ct);
    p.tpw = plan.tpw;
    p.n_ng = (p.n_tiles + p.tpw - 1) / p.tpw;
    const uint32_t grid = p.n_ng * p.n_mt * p.ksplit;
    hipError_t err = hipErrorInvalidValue;
#define OXB_GEMM_CASE(R, C)                                                                        \
    if (plan.rt == R && plan.ct == C)                                                              \
        err = fmt == OXB_FMT_Q1 ? launch_gemm_case<OXB_FMT_Q1, R, C>(p, grid, st) : fmt == OXB_FMT_TQ2 ? launch_gemm_case<OXB_FMT_TQ2, R, C>(p, grid, st) : launch_gemm_case<GEMM_TQ2_LOUD, R, C>(p, grid, st);
    OXB_GEMM_CASE(2, 8) OXB_GEMM_CASE(3, 8) OXB_GEMM_CASE(4, 8) OXB_GEMM_CASE(5, 8)
    OXB_GEMM_CASE(1, 5) OXB_GEMM_CASE(2, 5) OXB_GEMM_CASE(3, 5) OXB_GEMM_CASE(4, 5)
    OXB_GEMM_CASE(1, 4) OXB_GEMM_CASE(2, 4) OXB_GEMM_CASE(3, 4) OXB_GEMM_CASE(4, 4)
#undef OXB_GEMM_CASE
    if (err != hipSuccess || p.ksplit == 1 || p.sum_later) return err;
    const size_t plane = (size_t)p.M * p.ldy, n4 = plane / 4;
    hipLaunchKernelGGL(gemm_splitk_reduce_kernel, dim3((uint32_t)((n4 + 255) / 256)), dim3(256), 0, st, p.part, p.ksplit, plane,
                       p.mode == OXB_GEMM_RESIDUAL ? p.residual : nullptr, p.y, n4);
    return hipGetLastError();
}
