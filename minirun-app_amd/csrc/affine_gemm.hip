// 4-bit affine projections of many tokens on MFMA: y[T][N] = x[T][K] . W[N][K]^T
// for the prefill-sized calls of affineMM (AffineWeights.swift:239-254), groups
// of a multiple of 64.
//
// As in skinny.hip the weights are not dequantized: with one scale and one bias
// per weight row and group,
//   y_o += s_og * (sum_{i in g} x_i q_oi) + b_og * (sum_{i in g} x_i),
// q = 0..15 exact in bf16, so a product takes one MFMA where a dequantized
// weight takes two (bf16 parts hi and lo), and the only work per (output,
// group) is the multiply-add of the scale.  The second term is a product over
// groups: its factors, split into three bf16 parts each (24 bits), go to MFMA
// too, four groups at a time (bf16 biases: one part, 3 of 16 k-slots a group;
// else the six part products down to 2^-24).
//
// What bounds it: LDS and the DMA that fills it, then the matrix pipe (busy 35% of
// the cycles).  7168 x 16384, 1111 tokens: 356 us (698 before: two MFMAs per product,
// weights dequantized by every workgroup between barriers); copies of the kernel
// without its LDS reads of x took 285, without those and the DMA 207, without the
// scale multiply-adds 360.  Others, before -> now: 24576 x 1536, 1111 tokens 192 ->
// 161 us, 300 tokens 131 -> 51; 12288 x 7168, 1111 tokens 571 -> 311.  f32 outputs
// against 64 bits 1.1e-6 -> 2.6e-7 (K = 16384), 2.8e-7 -> 1.1e-7 (K = 1536).
//
// A workgroup of 8 waves owns 32 MI tokens x 256 weight rows (MI = 4 or 2):
// wave (h, c) takes rows 64 c .. + 63 of every second group (h), so each
// weight is unpacked by one wave only, in registers, and each x is read from
// LDS by four waves.  The two halves' sums meet in LDS at the end.
// An iteration takes 128 k (both halves' group): its x, packed words and scales
// come by DMA while the one before is used, with one barrier.
// v_mfma_f32_32x32x16_bf16, A = x (row = token), B = W (column = weight row): a
// lane holds one weight row, so its scale is one register.
// Within a group the k order is the packed words' own: lane half l / 32 takes
// words 4 (l / 32) .. + 3, and x chunks to match.
//
// The sums of x: wave w multiplies tokens 16 w .. + 15 (8 waves, 128 tokens)
// with ones and writes the three bf16 parts per (token, group) to LDS; after
// four iterations every wave adds its rows' biases times them.
//
// Outputs that are not finite are computed again from dequantized weights, by
// the wave that holds them, as in skinny.hip.  Rows past T or N read zeros and are not stored.
#include <algorithm>

#include "affine_tiles.hpp"
#include "mr_kernels.hpp"

namespace mr {

namespace {

constexpr int AG_TN = 256, AG_NW = 8, AG_THREADS = 64 * AG_NW;

template <int MI>
struct AgShape {
    static constexpr int TM = 32 * MI;
    static constexpr int XB = TM * 256, WB = AG_TN * 64, SB = AG_TN * 8;  // bytes per stage: x, words, scales (= biases)
    static constexpr int WOFF = 3 * XB, WSTAGE = WB + 2 * SB;  // three x stages, then two of words and scales
    static constexpr int XSOFF = WOFF + 2 * WSTAGE;
    static constexpr int XS = 2 * TM * 32;  // sums of x: [half][token][4 groups][4 bf16], double-buffered
    static constexpr int EXCH = AG_NW * (MI / 2) * 2 * 16 * 64 * 4;
    static constexpr size_t LDS = std::max(XSOFF + 2 * XS, EXCH);
    static_assert(LDS <= 163840, "LDS");
};

// the three bf16 parts of v, in the low halves of two words: {h | m << 16, l}
__device__ __forceinline__ u32x2 bf16_parts(float v) {
    const uint32_t h = pack_bf16x2_hw(v, 0.f);
    const float r = v - __uint_as_float(h << 16);  // exact
    const uint32_t m = pack_bf16x2_hw(r, 0.f);
    return u32x2{h | (m << 16), pack_bf16x2_hw(r - __uint_as_float(m << 16), 0.f)};
}

template <int MI, int SDT>
__global__ void __launch_bounds__(AG_THREADS) affine_gemm_kernel(ProjGemmStack ps) {
    using S = AgShape<MI>;
    constexpr int TM = S::TM;
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int tid = threadIdx.x, l = tid & 63, h = l >> 5, r32 = l & 31, lr = l & 15, q = l >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), kh = w >> 2, wc = w & 3;

    // tile order as in gemm.hip: the 8 XCDs take consecutive runs of groups of
    // 4 M tiles, N tiles outer
    const int m_tiles = (ps.seg[0].M + TM - 1) / TM, n_tiles = ps.tile_end[ps.nseg - 1];
    const int total = m_tiles * n_tiles;
    int bid = blockIdx.x;
    bid = (bid & 7) * (total >> 3) + min(bid & 7, total & 7) + (bid >> 3);
    constexpr int GM = 4;
    const int first_m = bid / (GM * n_tiles) * GM, gsize = min(m_tiles - first_m, GM);
    const int mt = first_m + (bid % (GM * n_tiles)) % gsize;
    const int nt_all = (bid % (GM * n_tiles)) / gsize;
    const int seg = (nt_all >= ps.tile_end[0]) + (nt_all >= ps.tile_end[1]);
    const ProjGemmParams p = ps.seg[seg];
    const int n0 = (nt_all - (seg ? ps.tile_end[seg - 1] : 0)) * AG_TN, m0 = mt * TM;
    const int rows = min(AG_TN, p.N - n0), toks = min(TM, p.M - m0);
    const int G = p.K / 64, gpl = p.group / 64, iters = (G + 7) / 8 * 4;  // by four: the biases'
    const uint32_t wrow = (uint32_t)p.K / 2, srow = (uint32_t)(p.K / p.group) * (SDT == 2 ? 4 : 2);
    const char* wbase = (const char*)p.packed + (int64_t)n0 * wrow;
    const char *sbase = (const char*)p.scales + (int64_t)n0 * srow, *bbase = (const char*)p.biases + (int64_t)n0 * srow;
    const uint16_t* xb = p.x + (int64_t)m0 * p.ldx;
    const i32x4 xres = uniform_rsrc(xb, (uint32_t)(((int64_t)(toks - 1) * p.ldx + p.K) * 2));
    const i32x4 wres = uniform_rsrc(wbase, (uint32_t)rows * wrow);
    // (2-byte scales: through the dword that holds the last one)
    const i32x4 sres = uniform_rsrc(sbase, ((uint32_t)rows * srow + 3u) & ~3u);
    const i32x4 bres = uniform_rsrc(bbase, ((uint32_t)rows * srow + 3u) & ~3u);

    // A row past the last reads zeros (its offset is past the buffer).
    // x rows of 256 bytes, chunk c of row r in slot c ^ (r % 16); DMA u of wave
    // w: rows 32 u + 4 w + l / 16, slot l % 16
    const int xtok = 4 * w + q, xk = 8 * (lr ^ (xtok & 15));  // xk: the chunk's first k
    const uint32_t xo = (uint32_t)(xtok * p.ldx * 2) + 2u * xk, x32 = (uint32_t)(64 * p.ldx);
    // words: rows of 64 bytes, chunk c of row r in slot c ^ ((r >> 2) & 3); DMA
    // u of wave w: rows 128 u + 16 w + l / 4, slot l % 4
    const int wk = 32 * ((l & 3) ^ ((l >> 4) & 3));
    const uint32_t wo = (uint32_t)(16 * w + (l >> 2)) * wrow + (uint32_t)wk / 2;
    // scales and biases: [row][2 groups] dwords that hold them; lane l of wave
    // w: row 32 w + l / 2, group l % 2
    const uint32_t so = (uint32_t)(32 * w + (l >> 1)) * srow;
    // g / gpl, exact (affine_gemm_ok)
    const uint32_t inv = gpl == 1 ? 0u : (uint32_t)((0x100000000ull + gpl - 1) / gpl);
    auto scale_of = [&](int g) { return gpl == 1 ? (uint32_t)g : __umulhi((uint32_t)g, inv); };
    auto issue = [&](int it, int xstage) {
        char* sx = lds + xstage * S::XB;
        char* st = lds + S::WOFF + (it & 1) * S::WSTAGE;
        const int k0 = 128 * it;  // (a chunk past the row's end: out of range)
        const uint32_t xv = k0 + xk < p.K ? xo + 2u * k0 : SK_OOB_K, wv = k0 + wk < p.K ? wo + (uint32_t)k0 / 2 : SK_OOB_K;
#pragma unroll
        for (int u = 0; u < MI; ++u)
            dma16_buf(xres, xv + u * x32, sx + 8192 * u + 1024 * w);
#pragma unroll
        for (int u = 0; u < 2; ++u)
            dma16_buf(wres, wv + u * 128 * wrow, st + 8192 * u + 1024 * w);
        const int g = min(2 * it + (l & 1), G - 1);  // a group past the last is not used
        const uint32_t sv = (so + scale_of(g) * (SDT == 2 ? 4 : 2)) & ~3u;
        dma4_buf(sres, sv, st + S::WB + 256 * w);
        dma4_buf(bres, sv, st + S::WB + S::SB + 256 * w);
    };

    f32x16 acc[MI][2];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = f32x16{};
    const bf16x8 ones = __builtin_bit_cast(bf16x8, u32x4{0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u});
    char* const xs = lds + S::XSOFF;
    // the lane's two of the last four groups' biases: 2h, 2h + 1 (bf16), or h, 2 + h
    float bias[2][2] = {};
    auto add_biases = [&](int buf) {
        int l = tid & 63;
        asm volatile("" : "+v"(l));
        const int h = l >> 5, r32 = l & 31;
        const char* xa = xs + buf * S::XS + kh * TM * 32;
        bf16x8 fb[2][2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            if constexpr (SDT == 0) {  // lane half: groups 2h, 2h + 1, k-slots {h, m, l, 0} of each
                const uint32_t b0 = __float_as_uint(bias[j][0]) >> 16;
                const uint32_t b1 = __float_as_uint(bias[j][1]) >> 16;
                fb[j][0] = __builtin_bit_cast(bf16x8, u32x4{b0 | (b0 << 16), b0, b1 | (b1 << 16), b1});
            } else {  // lane half: group 2m + h, k-slots {hh, hm, hl, mh, mm, lh, 0, 0} (bias part, x part)
#pragma unroll
                for (int m = 0; m < 2; ++m) {
                    const u32x2 b = bf16_parts(bias[j][m]);
                    const uint32_t bh = b[0] & 0xffffu, bm = b[0] >> 16;
                    fb[j][m] = __builtin_bit_cast(bf16x8, u32x4{bh | (bh << 16), bh | (bm << 16), bm | (b[1] << 16), 0u});
                }
            }
        }
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            const char* xt = xa + 32 * (32 * i + r32);
            if constexpr (SDT == 0) {
                const bf16x8 fx = *(const bf16x8*)(xt + 16 * h);
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] = mfma32(fx, fb[j][0], acc[i][j]);
            } else {
#pragma unroll
                for (int m = 0; m < 2; ++m) {
                    const u32x2 v = *(const u32x2*)(xt + 16 * m + 8 * h);
                    const uint32_t xh = v[0] & 0xffffu, xm = v[0] >> 16;
                    const bf16x8 fx = __builtin_bit_cast(bf16x8, u32x4{v[0], v[1] | (xh << 16), xm | (xh << 16), 0u});
#pragma unroll
                    for (int j = 0; j < 2; ++j) acc[i][j] = mfma32(fx, fb[j][m], acc[i][j]);
                }
            }
        }
    };

    // this half's group of iteration `it`: scales, biases and words of the
    // lane's two rows; and the sums of x of both groups
    float sc[2];
    bf16x8 fw[2][4];
    // (lane-dependent addresses are computed again each time: kept in
    // registers across the loop they would not fit beside the accumulators)
    auto unpack = [&](int it, int xstage) {
        int l = tid & 63;
        asm volatile("" : "+v"(l));
        const int h = l >> 5, r32 = l & 31, lr = l & 15, q = l >> 4;
        const int c = it >> 2, c4 = it & 3;
        const char* st = lds + S::WOFF + (it & 1) * S::WSTAGE;
        const int g = 2 * it + kh;
        const bool live = g < G;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int row = 64 * wc + 32 * j + r32;
            uint32_t sw = *(const uint32_t*)(st + S::WB + 8 * row + 4 * kh);
            uint32_t bw = *(const uint32_t*)(st + S::WB + S::SB + 8 * row + 4 * kh);
            if (SDT != 2) {  // the half that holds it
                const uint32_t sh = (((uint32_t)row * (srow >> 1) + scale_of(g)) & 1u) * 16u;
                sw = (sw >> sh) & 0xffffu;
                bw = (bw >> sh) & 0xffffu;
            }
            sc[j] = live ? sk_scale<SDT>(sw) : 0.f;
            const float b = live ? sk_scale<SDT>(bw) : 0.f;
#pragma unroll
            for (int k = 0; k < 2; ++k) bias[j][k] = c4 == (SDT == 0 ? 2 * h + k : 2 * k + h) ? b : bias[j][k];
            const u32x4 words = *(const u32x4*)(st + 64 * row + 16 * ((2 * kh + h) ^ ((row >> 2) & 3)));
#pragma unroll
            for (int k = 0; k < 4; ++k) fw[j][k] = nibbles_bf16(words[k]);
        }
        if (16 * w < TM) {
            const uint32_t a = (uint32_t)(xstage * S::XB + 256 * (16 * w + lr) + 16 * (q ^ lr));
#pragma unroll
            for (int g2 = 0; g2 < 2; ++g2) {
                f32x4 v = f32x4{};
#pragma unroll
                for (int s = 0; s < 2; ++s)
                    v = mfma16(*(const bf16x8*)(lds + (a ^ (128u * g2 + 64u * s))), ones, v);
                // lane lr < 4 of each quarter: token 16 w + 4 q + lr
                const float t = lr & 2 ? (lr & 1 ? v[3] : v[2]) : (lr & 1 ? v[1] : v[0]);
                if (lr < 4)
                    *(u32x2*)(xs + (c & 1) * S::XS + g2 * TM * 32 + 32 * (16 * w + 4 * q + lr) + 8 * c4) = bf16_parts(t);
            }
        }
    };
    // its products: those of tile t while the multiply-adds of tile t - 1 run
    auto products = [&](int xstage) {
        f32x16 d[2];
        bf16x8 fx[2][4];
        int l = tid & 63;
        asm volatile("" : "+v"(l));
        const uint32_t a = (uint32_t)(xstage * S::XB + 256 * (l & 31) + 16 * ((8 * kh + 4 * (l >> 5)) ^ (l & 15)));
        auto read_x = [&](int i) {
#pragma unroll
            for (int k = 0; k < 4; ++k) fx[i & 1][k] = *(const bf16x8*)(lds + (a ^ (16u * k)) + 8192 * i);
        };
        read_x(0);
#pragma unroll
        for (int t = 0; t <= 2 * MI; ++t) {
            if (t < 2 * MI) {
                const int i = t >> 1, j = t & 1;
                if (j == 0 && i + 1 < MI) read_x(i + 1);
                d[j] = mfma32(fx[i & 1][0], fw[j][0], f32x16{});
#pragma unroll
                for (int k = 1; k < 4; ++k) d[j] = mfma32(fx[i & 1][k], fw[j][k], d[j]);
            }
            if (t > 0) {
                const int i = (t - 1) >> 1, j = (t - 1) & 1;
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[i][j][e] = fmaf(sc[j], d[j][e], acc[i][j][e]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // Waves w and w + 4 share a SIMD.  Half 0 unpacks, then multiplies; half 1
    // multiplies the last iteration's group, then unpacks: one's vector work
    // runs beside the other's products.
    issue(0, 0);
    int cur = 0, nxt = 1, prv = 2;  // x stages
#pragma unroll 1
    for (int it = 0; it < iters; ++it) {
        wait_vmcnt<0>();  // this wave's part of the stage
        lds_barrier();    // every wave's; every wave done with the stages written next
        issue(it + 1, nxt);
        if ((it & 3) == 0 && it > 0) add_biases(((it >> 2) - 1) & 1);
        if (kh == 1 && it > 0) products(prv);
        unpack(it, cur);
        if (kh == 0) products(cur);
        const int t = prv;
        prv = cur;
        cur = nxt;
        nxt = t;
    }
    if (kh == 1) products(prv);
    wait_vmcnt<0>();
    lds_barrier();
    add_biases(((iters >> 2) - 1) & 1);
    __syncthreads();  // the stages and sums are free

    // half h finishes token tiles h MI / 2 .. of both halves' sums
    f32x4* ex = (f32x4*)lds;
    auto finish = [&](auto half) {
        constexpr int KH = decltype(half)::value, OWN = KH * (MI / 2), OTHER = (1 - KH) * (MI / 2);
#pragma unroll
        for (int i = 0; i < MI / 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const f32x16& a = acc[OTHER + i][j];
                    ex[((w * (MI / 2) + i) * 8 + j * 4 + g) * 64 + l] = f32x4{a[4 * g], a[4 * g + 1], a[4 * g + 2], a[4 * g + 3]};
                }
        __syncthreads();
        uint64_t again = 0;  // values that are not finite
        auto store = [&](int m, int nn, float y) {
            const int64_t at = (int64_t)(m0 + m) * p.ldy + n0 + nn;
            if (p.y_f32)
                ((float*)p.y)[at] = y;
            else
                ((uint16_t*)p.y)[at] = f32_to_bf16_bits(y);
        };
#pragma unroll
        for (int v = 0; v < MI * 16; ++v) {
            const int i = v >> 5, j = (v >> 4) & 1, e = v & 15;
            const int m = 32 * (OWN + i) + 8 * (e >> 2) + 4 * h + (e & 3), nn = 64 * wc + 32 * j + r32;
            const float y = acc[OWN + i][j][e] + ((const float*)&ex[(((w ^ 4) * (MI / 2) + i) * 8 + j * 4 + (e >> 2)) * 64 + l])[e & 3];
            if (m >= toks || nn >= rows) continue;
            if (fabsf(y) < INFINITY)
                store(m, nn, y);
            else
                again |= 1ull << v;
        }
        if (!__ballot(again != 0)) return;
        int finite = -1;
        // token by token: lane half b of bit (i, j, e) holds row 32 j + its lane
        // for token 32 i + 8 (e / 4) + 4 b + e % 4
#pragma unroll 1
        for (int t = 0; t < 16 * MI; ++t) {
            const int v = (t & ~31) + 4 * ((t & 31) >> 3) + (t & 3), up = 32 * ((t >> 2) & 1);
            const uint64_t lo = __ballot((again >> v) & 1), hi = __ballot((again >> (v + 16)) & 1);
            const uint64_t which = ((lo >> up) & 0xffffffffull) | ((hi >> up) << 32);
            if (!which) continue;
            const int m = 32 * OWN + t;
            const int64_t r0 = 64 * wc;
            const float y = sk_affine_again<SDT>(which, xb + m * p.ldx, wbase + r0 * wrow, sbase + r0 * srow, bbase + r0 * srow,
                                                 wrow, srow, p.K, p.group, finite);
            if ((which >> l) & 1) store(m, 64 * wc + l, y);
        }
    };
    if (kh == 0)
        finish(std::integral_constant<int, 0>{});
    else
        finish(std::integral_constant<int, 1>{});
}

template <int MI, int SDT>
hipError_t launch_mi(const ProjGemmStack& ps, hipStream_t st) {
    using S = AgShape<MI>;
    const int m_tiles = (ps.seg[0].M + S::TM - 1) / S::TM, n_tiles = ps.tile_end[ps.nseg - 1];
    const auto kern = affine_gemm_kernel<MI, SDT>;
    const hipError_t attr = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)S::LDS);
    if (attr != hipSuccess) return attr;
    hipLaunchKernelGGL(kern, dim3((unsigned)(m_tiles * n_tiles)), dim3(AG_THREADS), S::LDS, st, ps);
    return hipGetLastError();
}

template <int MI>
hipError_t launch_sdt(const ProjGemmStack& ps, hipStream_t st) {
    if (ps.seg[0].scale_dtype == 0) return launch_mi<MI, 0>(ps, st);
    if (ps.seg[0].scale_dtype == 1) return launch_mi<MI, 1>(ps, st);
    return launch_mi<MI, 2>(ps, st);
}

}  // namespace

// beyond proj_gemm_ok: whole 64-groups, and buffers within the out-of-range offsets
bool affine_gemm_ok(const ProjGemmParams& p) {
    return p.packed && p.group % 64 == 0 && (int64_t)AG_TN * (p.K / 2) < (1 << 30) && (int64_t)128 * p.ldx * 2 < (1 << 30) &&
           (int64_t)(p.K / 64) * (p.group / 64) < INT32_MAX;
}

namespace {

// us of a launch with tiles of 32 MI tokens: workgroups run in rounds of one
// per CU; a round of MI = 2 takes 12.1 ns per k (7168 x 16384, 64 to 500 tokens:
// 191 to 209 us), of MI = 4 22.3 ns (1111 tokens: 372 us), and 6 us to fill,
// exchange and store
double tiles_cost(int64_t n_tiles, int m, int k, int mi, int cus) {
    const int64_t wgs = n_tiles * ((m + 32 * mi - 1) / (32 * mi));
    return (double)((wgs + cus - 1) / cus) * (k * (mi == 2 ? 12.1e-3 : 22.3e-3) + 6.);
}

}  // namespace

double affine_gemm_cost(int64_t n, int m, int k, int cus) {
    const int64_t n_tiles = (n + AG_TN - 1) / AG_TN;
    return std::min(tiles_cost(n_tiles, m, k, 2, cus), tiles_cost(n_tiles, m, k, 4, cus));
}

int affine_gemm_rows(int64_t n_tiles, int m, int k, int cus) {
    return tiles_cost(n_tiles, m, k, 4, cus) < tiles_cost(n_tiles, m, k, 2, cus) ? 128 : 64;
}

hipError_t launch_affine_gemm(const ProjGemmStack& ps, int cu_count, hipStream_t st) {
    const int n_tiles = ps.tile_end[ps.nseg - 1], m = ps.seg[0].M, k = ps.seg[0].K;
    return affine_gemm_rows(n_tiles, m, k, cu_count) == 128 ? launch_sdt<4>(ps, st) : launch_sdt<2>(ps, st);
}

}  // namespace mr
