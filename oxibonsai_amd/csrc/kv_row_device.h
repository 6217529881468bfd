// kv_row_device.h — a new position's K and V row of one kv head from the raw projection: per-head RMSNorm and RoPE of K
// (fused_qk_norm_rope + fused_kv_store, gpu_backend/cuda_attn_kernels.rs:160-251), the values or one-byte codes that the cache
// holds.  HD / 4 lanes share a row: lane j has elements 4 j .. 4 j + 3, the other half of its RoPE pairs lies HD / 8 lanes away.
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stdint.h>

#include "device_utils.h"
#include "kv_quant_device.h"

// The sum / largest over groups of L lanes, in every lane.
template <int L>
__device__ __forceinline__ float group_sum(float v) {
    v += dpp_f32<0xB1>(v);
    v += dpp_f32<0x4E>(v);
    v += dpp_f32<0x141>(v);
    if constexpr (L >= 16) v += dpp_f32<0x140>(v);
    if constexpr (L >= 32) {
        const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    }
    if constexpr (L >= 64) {
        const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    }
    return v;
}
template <int L>
__device__ __forceinline__ float group_max(float v) {
    v = fmaxf(v, dpp_f32<0xB1>(v));
    v = fmaxf(v, dpp_f32<0x4E>(v));
    v = fmaxf(v, dpp_f32<0x141>(v));
    if constexpr (L >= 16) v = fmaxf(v, dpp_f32<0x140>(v));
    if constexpr (L >= 32) {
        const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    }
    if constexpr (L >= 64) {
        const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    }
    return v;
}

struct KvRowIn { float4 k, v, cs, sn; };
// row_in: the token's q heads | k heads | v heads
template <int HD>
__device__ __forceinline__ KvRowIn kv_row_load(const float* __restrict__ row_in, uint32_t nq, uint32_t nkv, uint32_t head, uint32_t j,
                                               const float* __restrict__ cos_t, const float* __restrict__ sin_t, uint32_t pos) {
    const uint32_t at = (4 * j) % (HD / 2);  // the pair's place
    const float* k = row_in + (size_t)(nq + head) * HD + 4 * j;
    return {*reinterpret_cast<const float4*>(k), *reinterpret_cast<const float4*>(k + (size_t)nkv * HD),
            *reinterpret_cast<const float4*>(cos_t + (size_t)pos * (HD / 2) + at), *reinterpret_cast<const float4*>(sin_t + (size_t)pos * (HD / 2) + at)};
}

// The lane's four values of K and V: four fp16 numbers, or four codes in .x and the row's scale.
struct KvRowOut { uint2 k, v; float ks, vs; };
template <int HD, int KVM>
__device__ __forceinline__ KvRowOut kv_row_make(const KvRowIn& in, const float4& w, float eps, uint32_t j) {
    constexpr int L = HD / 4;
    const float ss = group_sum<L>(fmaf(in.k.x, in.k.x, fmaf(in.k.y, in.k.y, fmaf(in.k.z, in.k.z, in.k.w * in.k.w))));
    const float inv_rms = 1.0f / sqrtf(ss / (float)HD + eps);
    const float a[4] = {w.x * in.k.x * inv_rms, w.y * in.k.y * inv_rms, w.z * in.k.z * inv_rms, w.w * in.k.w * inv_rms};
    const float c4[4] = {in.cs.x, in.cs.y, in.cs.z, in.cs.w}, s4[4] = {in.sn.x, in.sn.y, in.sn.z, in.sn.w}, v4[4] = {in.v.x, in.v.y, in.v.z, in.v.w};
    float o[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float other = __shfl_xor(a[i], L / 2, 64);
        // (written out, and an fp32 number before it becomes anything else: the same bits wherever this is inlined - the compiler
        // rounds some of these sums to fp16 inside the multiply-add)
        o[i] = fmaf(j < L / 2 ? -other : other, s4[i], a[i] * c4[i]);
        asm("" : "+v"(o[i]));
    }
    KvRowOut r = {make_uint2(0, 0), make_uint2(0, 0), 1.f, 1.f};
    if constexpr (KVM != OXB_KV_F16) {
        r.ks = kv_row_scale<KVM>(group_max<L>(fmaxf(fmaxf(fabsf(o[0]), fabsf(o[1])), fmaxf(fabsf(o[2]), fabsf(o[3])))));
        r.vs = kv_row_scale<KVM>(group_max<L>(fmaxf(fmaxf(fabsf(v4[0]), fabsf(v4[1])), fmaxf(fabsf(v4[2]), fabsf(v4[3])))));
#pragma unroll
        for (int i = 0; i < 4; i++) r.k.x |= kv_encode<KVM>(o[i], r.ks) << (8 * i), r.v.x |= kv_encode<KVM>(v4[i], r.vs) << (8 * i);
    } else {
        typedef _Float16 h4 __attribute__((ext_vector_type(4)));
        r.k = __builtin_bit_cast(uint2, (h4){(_Float16)o[0], (_Float16)o[1], (_Float16)o[2], (_Float16)o[3]});
        r.v = __builtin_bit_cast(uint2, (h4){(_Float16)v4[0], (_Float16)v4[1], (_Float16)v4[2], (_Float16)v4[3]});
    }
    return r;
}

template <int HD, int KVM>
__device__ __forceinline__ void kv_row_store(const KvRowOut& r, void* k_cache, void* v_cache, float* k_scale, float* v_scale, size_t row, uint32_t j) {
    constexpr int L = HD / 4;
    if constexpr (KVM != OXB_KV_F16) {
        reinterpret_cast<uint32_t*>(k_cache)[row * L + j] = r.k.x;
        reinterpret_cast<uint32_t*>(v_cache)[row * L + j] = r.v.x;
        if (j == 0) k_scale[row] = r.ks, v_scale[row] = r.vs;
    } else {
        reinterpret_cast<uint2*>(k_cache)[row * L + j] = r.k;
        reinterpret_cast<uint2*>(v_cache)[row * L + j] = r.v;
    }
}
