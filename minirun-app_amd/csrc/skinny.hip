// Projections of a few tokens on MFMA: y[T][N] = x[T][K] . W[N][K]^T for the
// calls between one token (the GEMV kernels) and a prompt (gemm.hip): a batch
// of decodes, speculative tokens, short prompts.  k3Linear (Linear.swift:55-57).
//
// What bounds it: the weights' bytes from HBM while T is small (each weight is
// read once per 16 TT tokens), the activations' bytes from L2 after that
// (every workgroup reads all of its tokens' rows).  A workgroup of 8 waves
// owns 16 RT weight rows and 16 TT tokens, and its waves split K: wave w takes
// ring entries w, w + 8, ... of 32 k.  Each wave
// streams its own entries into its own LDS ring of S entries by DMA and waits
// for its own vmcnt, so the loop has no barrier; an entry's fragments are read
// to registers, the slot is refilled at once, then the products run.  The
// waves' partial sums meet in LDS once, at the end, in a fixed order.
// Workgroups of one row tile and several token blocks sit 8 apart, on one XCD.
//
// Why DMA and not loads straight to the operand registers: those need 16 rows
// in neighbouring lanes, so every four lanes touch four lines, and such loads
// reach 9 TB/s from L2 where lanes that cover whole 64-byte pieces of a row
// reach 25-30 (one 14336-byte row set read by 256 workgroups).
//
// v_mfma_f32_16x16x32_bf16 with A = x (row = token) and B = W (column =
// weight row): lane l holds weight row l % 16 and tokens 4 (l / 16) + 0..3.
// Short chains of MFMAs start from zero and are added to the running sums by
// fp32 adds: fewer roundings at the size of the whole sum (with one chain per
// wave the error against 64 bits is a third larger).
#include <algorithm>

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

// row tile and token block of this workgroup: consecutive workgroups go to
// the 8 XCDs in turn
__device__ __forceinline__ void sk_tile(int bid, int blocks, int& tile, int& tb) {
    const int lo = bid & 7, hi = bid >> 3;
    tb = hi % blocks;
    tile = (hi / blocks) * 8 + lo;
}

// partial sums of the waves -> LDS -> one f32x4 per (tile, lane): emit(r, t,
// lane, value) of row tile r, token tile t
template <int RT, int TT, int NW, typename F>
__device__ __forceinline__ void sk_reduce(char* lds, const f32x4 (&acc)[RT][TT], F emit) {
    const int tid = threadIdx.x, w = tid >> 6, l = tid & 63;
    constexpr int P = RT * TT * 64;
    f32x4* d = (f32x4*)lds;
    __syncthreads();  // every wave is done with its ring
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int t = 0; t < TT; ++t) d[w * P + (r * TT + t) * 64 + l] = acc[r][t];
    __syncthreads();
    for (int i = tid; i < P; i += 64 * NW) {
        f32x4 v[NW];
#pragma unroll
        for (int k = 0; k < NW; ++k) v[k] = d[k * P + i];
#pragma unroll
        for (int n = 1; n < NW; n *= 2)
#pragma unroll
            for (int k = 0; k + n < NW; k += 2 * n) v[k] += v[k + n];
        emit((i >> 6) / TT, (i >> 6) % TT, i & 63, v[0]);
    }
}

// ---------------------------------------------------------------- dense
// Ring entry: 32 k; W [16 RT rows][64 B], then x [16 TT rows][64 B]; 16-byte
// chunk c of row r in slot c ^ ((r >> 2) & 3), so the 16 rows of a ds_read_b128
// phase hit 16 bank groups.
//
// Measured, one call among others (rotating weights), before (token-tile GEMV,
// or the 128-row tiles of gemm.hip from 64 tokens) -> now: 12288 x 7168, 24
// tokens 497 -> 41 us (4.3 TB/s of weights), 2 tokens 70 -> 34 us (5.2 TB/s),
// 64 tokens 128 -> 52 us; 7168 x 16384, 24 tokens 899 -> 64 us; 576 x 7168, 24
// tokens 61 -> 11 us.
template <int RT, int TT, int S, int NW>
__global__ void __launch_bounds__(64 * NW) skinny_dense_kernel(ProjGemmParams p, int blocks) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    constexpr int NI = RT + TT, ENTRY = 1024 * NI;
    static_assert((S - 1) * NI < 64, "vmcnt range");
    const int l = threadIdx.x & 63, q = l >> 4;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int tile, tb;
    sk_tile(blockIdx.x, blocks, tile, tb);
    const int n0 = tile * 16 * RT, m0 = tb * 16 * TT;
    if (n0 >= p.N) return;
    const int rows = min(16 * RT, p.N - n0), toks = min(16 * TT, p.M - m0);
    const i32x4 wres = uniform_rsrc(p.w + (int64_t)n0 * p.ldw, (uint32_t)(((int64_t)(rows - 1) * p.ldw + p.K) * 2));
    const i32x4 xres = uniform_rsrc(p.x + (int64_t)m0 * p.ldx, (uint32_t)(((int64_t)(toks - 1) * p.ldx + p.K) * 2));
    // lane l of a DMA fills slot l % 4 of row l / 4
    uint32_t wo[RT], xo[TT];
    const uint32_t ch = 16u * ((l & 3) ^ ((l >> 4) & 3));
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        const int row = 16 * r + (l >> 2);
        wo[r] = row < rows ? (uint32_t)(row * p.ldw * 2) + ch : SK_OOB_ROW;
    }
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        const int tok = 16 * t + (l >> 2);
        xo[t] = tok < toks ? (uint32_t)(tok * p.ldx * 2) + ch : SK_OOB_ROW;
    }
    char* ring = lds + w * S * ENTRY;
    const int nk = p.K / 32;
    const int n = w < nk ? (nk - 1 - w) / NW + 1 : 0;  // this wave's entries
    auto issue = [&](int i, int slot) {
        const uint32_t o = i < n ? 64u * (uint32_t)(w + NW * i) : SK_OOB_K;
        char* e = ring + slot * ENTRY;
#pragma unroll
        for (int r = 0; r < RT; ++r) dma16_buf(wres, wo[r] + o, e + 1024 * r);
#pragma unroll
        for (int t = 0; t < TT; ++t) dma16_buf(xres, xo[t] + o, e + 1024 * (RT + t));
    };
    f32x4 acc[RT][TT], part[RT][TT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int t = 0; t < TT; ++t) acc[r][t] = part[r][t] = f32x4{};
#pragma unroll
    for (int s = 0; s < S; ++s) issue(s, s);
    const uint32_t fo = 64u * (l & 15) + 16u * (q ^ ((l >> 2) & 3));
    int slot = 0;
    for (int i = 0; i < n; ++i) {
        wait_vmcnt<(S - 1) * NI>();
        const char* e = ring + slot * ENTRY + fo;
        bf16x8 fw[RT], fx[TT];
#pragma unroll
        for (int r = 0; r < RT; ++r) fw[r] = *(const bf16x8*)(e + 1024 * r);
#pragma unroll
        for (int t = 0; t < TT; ++t) fx[t] = *(const bf16x8*)(e + 1024 * (RT + t));
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0xc07f);  // the same, known to the compiler
        __builtin_amdgcn_sched_barrier(0);
        issue(i + S, slot);
        slot = slot + 1 == S ? 0 : slot + 1;
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int t = 0; t < TT; ++t) part[r][t] = mfma16(fx[t], fw[r], part[r][t]);
        if (i & 1) {
#pragma unroll
            for (int r = 0; r < RT; ++r)
#pragma unroll
                for (int t = 0; t < TT; ++t) {
                    acc[r][t] += part[r][t];
                    part[r][t] = f32x4{};
                }
        }
    }
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int t = 0; t < TT; ++t) acc[r][t] += part[r][t];
    wait_vmcnt<0>();
    sk_reduce<RT, TT, NW>(lds, acc, [&](int r, int t, int lane, f32x4 v) {
        const int n = n0 + 16 * r + (lane & 15);
        if (n >= p.N) return;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int m = m0 + 16 * t + 4 * (lane >> 4) + e;
            if (m >= p.M) break;
            const int64_t o = (int64_t)m * p.ldy + n;
            if (p.y_f32)
                ((float*)p.y)[o] = v[e];
            else
                ((uint16_t*)p.y)[o] = f32_to_bf16_bits(v[e]);
        }
    });
}

template <typename K>
hipError_t set_lds(K kern, size_t lds) {
    return lds > 65536 ? hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds)
                       : hipSuccess;
}

template <int RT, int TT, int S, int NW>
hipError_t launch_dense(const ProjGemmParams& p, hipStream_t st) {
    constexpr size_t lds = std::max<size_t>((size_t)NW * S * (RT + TT) * 1024, (size_t)NW * RT * TT * 1024);
    static_assert(lds <= 163840, "LDS");
    const auto kern = skinny_dense_kernel<RT, TT, S, NW>;
    const hipError_t e = set_lds(kern, lds);
    if (e != hipSuccess) return e;
    const int tiles = (p.N + 16 * RT - 1) / (16 * RT), blocks = (p.M + 16 * TT - 1) / (16 * TT);
    hipLaunchKernelGGL(kern, dim3((unsigned)((tiles + 7) / 8 * 8 * blocks)), dim3(64 * NW), lds, st, p, blocks);
    return hipGetLastError();
}

}  // namespace

bool skinny_gemm_ok(const ProjGemmParams& p) {
    if (p.M <= 0 || p.N <= 0 || p.K < 32 || p.K % 32 || ((uintptr_t)p.x & 15) || p.ldx % 8 || p.ldx < p.K) return false;
    if ((int64_t)64 * p.ldx * 2 >= (1 << 30)) return false;  // byte offsets of one token block's rows
    if (((int64_t)p.N / 16 + 8) * ((int64_t)p.M / 16 + 1) > INT32_MAX) return false;  // workgroups
    return !p.packed && p.w && ((uintptr_t)p.w & 15) == 0 && p.ldw % 8 == 0 && p.ldw >= p.K && (int64_t)64 * p.ldw * 2 < (1 << 30);
}

namespace {

// Token tiles of 16 per workgroup
int token_tiles(int m) { return m <= 16 ? 1 : (m <= 32 ? 2 : 4); }

// Time of a dense launch with RT row tiles per workgroup, in units of one row
// tile's weights per CU: workgroups run in rounds of one per CU, and a token
// tile's activations (from L2) cost about 0.3 of a row tile's weights
double dense_cost(int64_t n, int m, int rt, int cus) {
    const int tt = token_tiles(m);
    const int64_t wgs = (int64_t)((n + 16 * rt - 1) / (16 * rt)) * ((m + 16 * tt - 1) / (16 * tt));
    return (double)((wgs + cus - 1) / cus) * (rt + 0.3 * tt);
}

// RT with the least cost, the larger one of equals (12288 rows, 24 tokens: 3
// row tiles 41 us, 2 54 us; 7168 rows: 2 64 us, 3 77 us; 576 rows: 1 11 us, 2
// 15 us)
int dense_rt(int64_t n, int m, int cus) {
    int best = 3;
    for (int rt = 2; rt >= 1; --rt)
        if (dense_cost(n, m, rt, cus) < dense_cost(n, m, best, cus)) best = rt;
    return best;
}

}  // namespace

// Against gemm.hip's tiles, both in rounds of one workgroup per CU.  Dense: a
// unit of dense_cost takes 1.65 ns per k (52 us at 12288 x 7168, 64 tokens),
// a round of 128-row tiles 17.5 ns per k (128 us there).
bool skinny_gemm_better(int64_t n, int m, int cus) {
    if (m < PROJ_GEMM_MIN_TOKENS) return true;
    const int64_t tiles = (int64_t)((m + 127) / 128) * ((n + 255) / 256), rounds = (tiles + cus - 1) / cus;
    return dense_cost(n, m, dense_rt(n, m, cus), cus) * 1.65 < 17.5 * rounds;
}

hipError_t launch_skinny_gemm(const ProjGemmParams& p, int cu_count, hipStream_t st) {
    const int tt = token_tiles(p.M);
    const int rt = dense_rt(p.N, p.M, cu_count);
    if (tt == 1) return rt == 1 ? launch_dense<1, 1, 4, 8>(p, st) : (rt == 2 ? launch_dense<2, 1, 3, 8>(p, st) : launch_dense<3, 1, 2, 8>(p, st));
    if (tt == 2) return rt == 1 ? launch_dense<1, 2, 3, 8>(p, st) : (rt == 2 ? launch_dense<2, 2, 2, 8>(p, st) : launch_dense<3, 2, 2, 8>(p, st));
    return rt == 1 ? launch_dense<1, 4, 2, 8>(p, st) : (rt == 2 ? launch_dense<2, 4, 3, 8>(p, st) : launch_dense<3, 4, 2, 8>(p, st));
}

}  // namespace mr
