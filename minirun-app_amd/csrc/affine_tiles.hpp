// What the MFMA kernels over 4-bit affine rows share (skinny.hip,
// affine_gemm.hip): buffer offsets past every row, nibbles as bf16 operands,
// scales, and outputs from dequantized weights.
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

// One token's outputs again, from dequantized weights, by a whole wave: lane j's
// is weight row j of `packed` / `scales` / `biases` (rows of wrow / srow bytes),
// where bit j of `rows` (the same in every lane) is set.  `finite` is the lane's
// note of its row's weights: -1 unknown, which is what the caller starts with.
//
// For outputs that are not finite.  A NaN in x makes them all NaN, and with
// infinities in x only those products count (if every weight is finite): both
// take one read of the row of x.  What is left, sums of finite values that
// overflow without their scales, or more infinities than 64, is summed by the
// wave, one output after the other.  (7168 x 16384, finite / every x NaN / one
// infinity in each row: 13 tokens 27 / 32 / 119 us, 300 tokens 194 / 243 / 795,
// 1111 tokens 363 / 387 / 948; each output by one lane took 10.6, 202 and 692 ms
// for both.)
constexpr int SK_INFS = 64;

template <int SDT>
__device__ float sk_affine_again(uint64_t rows, const uint16_t* x, const char* packed, const char* scales,
                                 const char* biases, uint32_t wrow, uint32_t srow, int K, int group, int& finite) {
    int l = threadIdx.x & 63;
    asm volatile("" : "+v"(l));  // no address of this is worth a register outside
    const bool mine = (rows >> l) & 1;
    auto scale = [&](const char* p, int g) {
        return sk_scale<SDT>(SDT == 2 ? ((const uint32_t*)p)[g] : ((const uint16_t*)p)[g]);
    };
    auto weight = [&](float s, float b, uint32_t q) { return add_rn(mul_rn(s, (float)(q & 15u)), b); };
    const char *wl = packed + (int64_t)l * wrow, *sl = scales + (int64_t)l * srow, *bl = biases + (int64_t)l * srow;
    float acc = 0.f;
    int infs = 0;
#pragma unroll 1
    for (int k0 = 0; k0 < K; k0 += 2048) {
        u32x4 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int k = k0 + 512 * u + 8 * l;
            v[u] = k < K ? *(const u32x4*)(x + k) : u32x4{};
        }
        bool nan = false;
        uint32_t inf = 0;  // bit 8 u + i: value i of chunk u
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint32_t e = (v[u][i >> 1] >> (16 * (i & 1))) & 0x7fffu;
                nan |= e > 0x7f80u;
                inf |= e == 0x7f80u ? 1u << (8 * u + i) : 0u;
            }
        if (__ballot(nan)) return NAN;
        uint64_t lanes = __ballot(inf != 0);
#pragma unroll 1
        while (lanes && infs < SK_INFS) {
            const int from = __builtin_ctzll(lanes);
            lanes &= lanes - 1;
            uint32_t bits = __builtin_amdgcn_readlane(inf, from);
#pragma unroll 1
            while (bits && infs < SK_INFS) {
                const int at = __builtin_ctz(bits);
                bits &= bits - 1;
                ++infs;
                const int k = k0 + 512 * (at >> 3) + 8 * from + (at & 7);
                if (mine) {
                    const uint32_t word = ((const uint32_t*)wl)[k >> 3];
                    const int g = k / group;
                    acc = fmaf(bf16_bits_to_f32(x[k]), weight(scale(sl, g), scale(bl, g), word >> (4 * (k & 7))), acc);
                }
                if (!__ballot(mine && acc == acc)) return acc;
            }
        }
    }
    bool open = mine && acc == acc;
    if (open && infs > 0 && infs < SK_INFS) {
        if (finite < 0) {
            finite = 1;
#pragma unroll 4
            for (int g = 0; g < K / group; ++g)
                finite &= fmaf(fabsf(scale(sl, g)), 15.f, fabsf(scale(bl, g))) < INFINITY;
        }
        open = !finite;
    }
    uint64_t left = __ballot(open);
#pragma unroll 1
    while (left) {
        const int j = __builtin_ctzll(left);
        left &= left - 1;
        const uint32_t* wj = (const uint32_t*)(packed + (int64_t)j * wrow);
        const char *sj = scales + (int64_t)j * srow, *bj = biases + (int64_t)j * srow;
        float d = 0.f;
#pragma unroll 1
        for (int k = 8 * l; k < K; k += 512) {
            const u32x4 v = *(const u32x4*)(x + k);
            const uint32_t word = wj[k >> 3];
            const int g = k / group;
            const float s = scale(sj, g), b = scale(bj, g);
#pragma unroll
            for (int i = 0; i < 8; ++i)
                d = fmaf(__uint_as_float(i & 1 ? v[i >> 1] & 0xffff0000u : v[i >> 1] << 16), weight(s, b, word >> (4 * i)), d);
        }
        d = wave_sum(d);
        if (l == j) acc = d;
    }
    return acc;
}

__device__ __forceinline__ void dma4_buf(i32x4 rsrc, uint32_t voff, const void* lds_dst_wave_base) {
    const uint32_t m0 = (uint32_t)(uintptr_t)lds_dst_wave_base;
    asm volatile("buffer_load_dword %0, %1, 0 offen lds" ::"v"(voff), "s"(rsrc), "{m0}"(m0) : "memory");
}

}  // namespace

}  // namespace mr
