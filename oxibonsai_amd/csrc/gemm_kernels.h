// gemm_kernels.h — launch interface of the prefill GEMM (fp16 MFMA) and its activation packer.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "layout.h"

// STORE: y = W a;  RESIDUAL: y = residual + W a;  SWIGLU: W = gate || up (n_rows = 2 * inter, a multiple of 32),
// y[m][i] = silu(gate_i . a) * (up_i . a) for i < inter, ldy >= inter.
enum { OXB_GEMM_STORE = 0, OXB_GEMM_RESIDUAL = 2, OXB_GEMM_SWIGLU = 3 };
#define OXB_GEMM_NARROW_MAX_M 32  // up to this many token rows the narrow kernel (K split over waves) is always used

struct OxbGemmParams {
    const uint32_t* codes;   // resident codes section
    const uint16_t* scales;  // resident scales section
    const uint32_t* xh;      // packed fp16 activations (oxb_launch_xh_pack)
    const int32_t* xsh;      // [M] exponent that undoes the row scaling, INT32_MIN for a non-finite row; null: x_exp for all rows
    int32_t x_exp;
    int32_t loud;            // TQ2: 1 where a scale is 2^15 or more: the weights then do not enter the products twice as large
    float* y;                // [M][ldy]
    const float* residual;   // [M][ldy], mode RESIDUAL only
    uint32_t n_rows, n_tiles, n_sb;
    uint32_t M, M_pad;       // token rows, and that count rounded up to 16
    uint32_t ldy;
    uint32_t tpw;            // row tiles per workgroup   (filled by the launcher)
    uint32_t n_mt;           // token tiles of the launch (filled by the launcher)
    uint32_t n_ng;           // row groups of the launch  (filled by the launcher)
    uint32_t ksplit, sb_per_split;  // K slices and superblocks per slice (filled by the launcher)
    float* part;             // [ksplit][M][ldy] partial sums, needed when oxb_gemm_ksplit(...) > 1
    uint32_t codes_bytes, scales_bytes, xh_bytes;  // buffer extents (loads beyond them read 0)
    int mode;
    // Mode SWIGLU, optional: instead of y the packed activations of the product that follows (n_rows / 2 values a row, a multiple
    // of 128; its format is this matrix's) and their exponents.  norm2: |a|_2^2 of every row at most (OxbPackNorm);
    // |gate row j|_2 |up row j|_2 <= w_mant 2^w_exp for every j, w_mant in [0.5, 1).
    uint32_t* xh_out;
    int32_t* xsh_out;
    const float* norm2;
    float w_mant;
    int32_t w_exp;
    bool no_split;           // keep K in one piece (a caller without room for partial sums)
    bool sum_later;          // mode RESIDUAL: with K in slices leave the sums in `part`, the next pack of y adds them (OxbPackSum)
};

// Bytes of the packed activation buffer for M token rows of length k.
size_t oxb_xh_bytes(uint32_t k, uint32_t M);

// Activations a[M][k] -> fp16 in MFMA B-operand order, each row scaled by a power of two so that its largest
// element lies in [2^14, 2^15).  The activations are computed on the fly from x[M][ldx] by `op`:
//   IDENT: a = x;  RMSNORM: a = w * x / rms(x) (w = d_w[k]).
// d_rowmul: M floats of scratch (the multiplier applied to every row).
enum { OXB_PACK_IDENT = 0, OXB_PACK_RMSNORM = 1 };
// With `sum` (RMSNORM, ldx = k, a shape that oxb_pack_can_sum takes) x lacks the K slices' sums of the product it is the
// result of: x += planes 0 .. n - 1, in that order, then as above; x is written back.
struct OxbPackSum { const float* part; uint32_t n; size_t plane; };
bool oxb_pack_can_sum(uint32_t k, uint32_t M);
// RMSNORM, optional: norm2[m] is no less than the square of the 2-norm of row m's activations (and never 0); cap is such a bound for
// every row, from the norm weights: max |w|^2 k.
struct OxbPackNorm { float* norm2; float cap; };
hipError_t oxb_launch_xh_pack(int fmt, int op, const float* d_x, const float* d_w, uint32_t ldx, uint32_t k, float eps,
                              uint32_t M, float* d_rowmul, uint32_t* d_xh, int32_t* d_xsh, hipStream_t st, const OxbPackSum* sum = nullptr,
                              OxbPackNorm norm = {nullptr, 0.f});
// d_out[i] = the 2-norm of matrix row i times that of row n + i, i < n (bounds: weights are +-d or 0), infinity where a scale is not
// finite.  n is a multiple of 16.
hipError_t oxb_launch_pair_norms(const uint16_t* d_scales, uint32_t n_sb, uint32_t n, float* d_out, hipStream_t st);
// d_out[i] = the 2-norm of matrix row row0 + i with column j times w[j], i < n, and d_out[n + i] the same with no |w[j]| taken as more
// than `typical`.  row0 and n are multiples of 16.
hipError_t oxb_launch_weighted_norms(const uint16_t* d_scales, uint32_t n_sb, uint32_t row0, uint32_t n, const float* d_w, uint32_t k, float typical, float* d_out, hipStream_t st);
// What the launcher runs for p: the narrow kernel with rt row tiles per workgroup and ct token tiles of 16 (rt 0: the tall one with
// tpw row tiles per workgroup), or the wide one
// with rt row tiles per wave, tpw per workgroup, 16 ct tokens per tile; K in ksplit slices of sb_per_split superblocks.
struct OxbGemmPlan { bool narrow; uint32_t rt, tpw, ct, ksplit, sb_per_split; };
OxbGemmPlan oxb_gemm_plan(int fmt, const OxbGemmParams& p, uint32_t n_cus);
// Number of K slices the launcher will use for this shape (1: no workspace needed).
uint32_t oxb_gemm_ksplit(int fmt, const OxbGemmParams& p, uint32_t n_cus);
hipError_t oxb_launch_gemm(int fmt, OxbGemmParams p, uint32_t n_cus, hipStream_t st);
