// kore_attn_device.h - device helpers shared by the attention kernels.
// Internal to libkore_attn.so.
#pragma once

#include <hip/hip_runtime.h>

namespace kore_attn_gpu {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = 4;

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float4 ld4(const float *p) { return *reinterpret_cast<const float4 *>(p); }
__device__ __forceinline__ void st4(float *p, float4 v) { *reinterpret_cast<float4 *>(p) = v; }
__device__ __forceinline__ float4 zero4() { return make_float4(0.f, 0.f, 0.f, 0.f); }
__device__ __forceinline__ float comp(const float4 &v, int e) {
    return e == 0 ? v.x : (e == 1 ? v.y : (e == 2 ? v.z : v.w));
}


// Cross-lane moves inside a 16-lane DPP row (no LDS traffic).  CTRL is a
// DPP control word: 0x121..0x12F rotate the row right by 1..15 lanes,
// 0x141 mirrors each half-row of 8 lanes, 0x00..0xFF permute within quads.
template <int CTRL>
__device__ __forceinline__ float dpp(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xF, 0xF, false));
}
// Max over each 16-lane row; every lane of the row receives it.
__device__ __forceinline__ float row16_max(float x) {
    x = fmaxf(x, dpp<0x128>(x));
    x = fmaxf(x, dpp<0x124>(x));
    x = fmaxf(x, dpp<0x122>(x));
    return fmaxf(x, dpp<0x121>(x));
}
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// NEOX rotation of the pair (x0, x1) = (x[i], x[i + hd/2]) by (c, s)
// (kore.cpp:1379-1382): products rounded, then difference / sum rounded.
__device__ __forceinline__ void rope_pair(float x0, float x1, float2 cs, float &y0, float &y1) {
#pragma clang fp contract(off)
    const float a = x0 * cs.x, b = x1 * cs.y;
    const float c = x0 * cs.y, d = x1 * cs.x;
    y0 = a - b;
    y1 = c + d;
}

// x of lane l and of lane l ^ 16 (v_permlane16_swap with x as both operands
// returns the even 16-lane rows in one result and the odd rows in the other),
// and likewise of lane l ^ 32 (v_permlane32_swap).  The results are copied
// to integers before the bit casts: a bit cast applied to an element of the
// returned vector directly is compiled as the first element by this hipcc
// (ROCm 7.2) for either index.
__device__ __forceinline__ void pair16(float x, float &a, float &b) {
    const unsigned xb = __builtin_bit_cast(unsigned, x);
    const auto r = __builtin_amdgcn_permlane16_swap(xb, xb, false, false);
    const unsigned r0 = r[0], r1 = r[1];
    a = __builtin_bit_cast(float, r0);
    b = __builtin_bit_cast(float, r1);
}
__device__ __forceinline__ void pair32(float x, float &a, float &b) {
    const unsigned xb = __builtin_bit_cast(unsigned, x);
    const auto r = __builtin_amdgcn_permlane32_swap(xb, xb, false, false);
    const unsigned r0 = r[0], r1 = r[1];
    a = __builtin_bit_cast(float, r0);
    b = __builtin_bit_cast(float, r1);
}

}  // namespace
}  // namespace kore_attn_gpu
