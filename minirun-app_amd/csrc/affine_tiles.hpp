// What the MFMA kernels over 4-bit affine rows share (skinny.hip,
// affine_gemm.hip): buffer offsets past every row, nibbles as bf16 operands,
// scales, and one output from dequantized weights.
#pragma once
#include "mr_kernels.hpp"

namespace mr {

namespace {

// byte offsets outside every buffer (host check: buffers under 2^30 bytes), of
// a lane's row and of a k-block past the row's end; their sum is outside too
constexpr uint32_t SK_OOB_ROW = 0x40000000u, SK_OOB_K = 0x80000000u;

// the resource in scalar registers (its inputs are uniform, but may have been
// computed in vector registers)
__device__ __forceinline__ i32x4 uniform_rsrc(const void* base, uint32_t bytes) {
    i32x4 r = buffer_rsrc(base, bytes);
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = __builtin_amdgcn_readfirstlane(r[i]);
    return r;
}

// eight nibbles of a word as bf16 0..15, in their order
__device__ __forceinline__ bf16x8 nibbles_bf16(uint32_t w) {
    const uint32_t lo = w & 0x0F0F0F0Fu, hi = (w >> 4) & 0x0F0F0F0Fu;  // nibbles 0,2,4,6 / 1,3,5,7
    const uint32_t a = __builtin_amdgcn_perm(hi, lo, 0x05010400u), b = __builtin_amdgcn_perm(hi, lo, 0x07030602u);
    const u32x4 v = {__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(a, 512.f, false)),
                     __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(a, 512.f, true)),
                     __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(b, 512.f, false)),
                     __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(b, 512.f, true))};
    return __builtin_bit_cast(bf16x8, v);
}

template <int SDT>
__device__ __forceinline__ float sk_scale(uint32_t v) {
    return SDT == 0 ? __uint_as_float(v << 16) : (SDT == 1 ? f16_bits_to_f32((uint16_t)v) : __uint_as_float(v));
}

// one output from dequantized weights, in order
template <int SDT>
__device__ __forceinline__ float sk_affine_dot(const uint16_t* x, const uint32_t* packed, const void* scales,
                                               const void* biases, int K, int group) {
    float acc = 0.f;
#pragma unroll 1
    for (int i = 0; i < K; ++i) {
        const int g = i / group;
        const float s = sk_scale<SDT>(SDT == 2 ? ((const uint32_t*)scales)[g] : ((const uint16_t*)scales)[g]);
        const float b = sk_scale<SDT>(SDT == 2 ? ((const uint32_t*)biases)[g] : ((const uint16_t*)biases)[g]);
        const float qv = (float)((packed[i >> 3] >> (4 * (i & 7))) & 15u);
        acc = fmaf(bf16_bits_to_f32(x[i]), add_rn(mul_rn(s, qv), b), acc);
    }
    return acc;
}

__device__ __forceinline__ void dma4_buf(i32x4 rsrc, uint32_t voff, const void* lds_dst_wave_base) {
    const uint32_t m0 = (uint32_t)(uintptr_t)lds_dst_wave_base;
    asm volatile("buffer_load_dword %0, %1, 0 offen lds" ::"v"(voff), "s"(rsrc), "{m0}"(m0) : "memory");
}

}  // namespace

}  // namespace mr
