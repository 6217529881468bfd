// operand_device.h — where value k of token row m lies in the GEMM's packed activations (gemm_kernels.hip), for the kernels
// that leave their results there for the product that follows instead of fp32 rows for a pack launch.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "layout.h"

// The packed activations of M token rows: value v of the producer is stored as fp16(v 2^shift).  The shift comes from a
// bound on |v| (find_bounds, model.hip; for gate times up also the row's own norm, OxbPackNorm), so that nothing overflows: the
// bound times 2^shift lies below 2^15.  A value is stored to 2^-12 of itself, or where it lies below 2^-14 to 2^-25.  Between
// matrices that are even enough for it to be used (kEvenRows) and random rows of activations the largest value of a row lies
// 2^10 (h = 4096, equally loud rows) to 2^14 (one row 16 times as loud) below the bound, where fewer than one value in 10^4 to
// one in 400 is that small.  xh == nullptr: off.
// What it saves is two of the four pack launches of a layer and the fp32 rows in front of them (kernel traces, us per layer):
// 2048 tokens of the 8B shape 35.5 (25.7 of them for 12288 values a row), 301 tokens 13.2, 32 sequences 10.0 of 87, 23 tokens
// of the ternary 1.7B shape 6.1 of 50.  Against the CPU reference (24
// models of four layers, h 1024 to 2048, prompts of 7 to 150 tokens and steps of 12 or 20 sequences): 6.04e-4 / 5.48e-4 off, with packs
// throughout 6.05e-4 / 5.50e-4.
struct OxbOperandOut {
    _Float16* xh;
    uint32_t fmt, M_pad;
    int32_t shift;
};

// Index (in halves) of value k of row m; the next three values, where k is a multiple of four, follow at 2, 4 and 6.
OXB_HD size_t oxb_operand_index(uint32_t fmt, uint32_t k, uint32_t m, uint32_t M_pad) {
    const uint32_t blk = k >> 7, g = (k >> 5) & 3u, r = k & 31u;
    const uint32_t s = fmt == OXB_FMT_Q1 ? (r >> 2) & 3u : 2u * (r >> 4) + ((r >> 2) & 1u);
    const uint32_t h = fmt == OXB_FMT_Q1 ? r >> 4 : (r >> 3) & 1u;
    return ((size_t)(blk * 16u + 4u * g + s) * M_pad + m) * 8u + 2u * (r & 3u) + h;
}

#ifdef __HIPCC__
// Four consecutive values of row m from k (a multiple of four) on.
__device__ __forceinline__ void operand_store4(const OxbOperandOut& o, uint32_t k, uint32_t m, float a, float b, float c, float d) {
    _Float16* q = o.xh + oxb_operand_index(o.fmt, k, m, o.M_pad);
    q[0] = (_Float16)ldexpf(a, o.shift), q[2] = (_Float16)ldexpf(b, o.shift), q[4] = (_Float16)ldexpf(c, o.shift), q[6] = (_Float16)ldexpf(d, o.shift);
}
// The eight values of row m that share 16 bytes with value k (a multiple of four, the first of the piece): lo the four from k on, hi
// the four `OXB_OPERAND_STEP` further.
#define OXB_OPERAND_STEP(fmt) ((fmt) == OXB_FMT_Q1 ? 16u : 8u)
__device__ __forceinline__ void operand_store8(const OxbOperandOut& o, uint32_t k, uint32_t m, const float4& lo, const float4& hi) {
    typedef _Float16 v8h_op __attribute__((ext_vector_type(8)));
    const v8h_op v = {(_Float16)ldexpf(lo.x, o.shift), (_Float16)ldexpf(hi.x, o.shift), (_Float16)ldexpf(lo.y, o.shift), (_Float16)ldexpf(hi.y, o.shift),
                      (_Float16)ldexpf(lo.z, o.shift), (_Float16)ldexpf(hi.z, o.shift), (_Float16)ldexpf(lo.w, o.shift), (_Float16)ldexpf(hi.w, o.shift)};
    *reinterpret_cast<v8h_op*>(o.xh + oxb_operand_index(o.fmt, k, m, o.M_pad)) = v;
}
#endif
