// Projections of a few tokens on MFMA: y[T][N] = x[T][K] . W[N][K]^T for the
// calls between one token (the GEMV kernels) and a prompt (gemm.hip): a batch
// of decodes, speculative tokens, short prompts, and the tokens that a router
// sends to one expert.  k3Linear (Linear.swift:55-57), affineMM
// (AffineWeights.swift:239-254), affineGatherMM (AffineWeights.swift:255-318).
//
// What bounds it: the weights' bytes from HBM while T is small (each weight is
// read once per 16 TT tokens), the activations' bytes from L2 after that
// (every workgroup reads all of its tokens' rows).  A workgroup of 8 waves
// owns 16 RT weight rows and 16 TT tokens, and its waves split K: wave w takes
// ring entries w, w + 8, ... of 32 k (dense) or 128 k (4-bit).  Each wave
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
//
// Affine weights are not dequantized: a lane's weight row has one scale and
// one bias per group, so
//   y_o += s_og * (sum_{i in g} x_i q_oi) + b_og * (sum_{i in g} x_i)
// with both inner sums on MFMA (q = 0..15 is exact in bf16; the sum of x is a
// product with ones) and the two multiply-adds in fp32.  A nibble becomes bf16
// by v_cvt_scalef32_pk_bf16_fp8: the e4m3 codes 0..15 are q * 2^-9 (0..7
// subnormal), and the scale 2^9 makes them q.  An output that is not finite
// that way (an infinite activation, or a sum that overflows without its
// scale) is computed again from dequantized weights, so it holds what those
// give.
#include <algorithm>

#include "affine_tiles.hpp"
#include "mr_kernels.hpp"

namespace mr {

namespace {

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
        const int rt = __builtin_amdgcn_readfirstlane(i >> 6);
        emit(rt / TT, rt % TT, i & 63, v[0]);
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

// ---------------------------------------------------------------- 4-bit affine
constexpr int SK_IDS = 32;            // routed: ids per thread and scan
constexpr int SK_WINDOW_MAX_LOG2 = 9;  // pairs per workgroup
constexpr int SK_MAX_EXPERTS = 3072;   // bins in the ring of sk_find_window

// Routed, pairs lo .. hi - 1 of expert e, as the scans find them, into `list`
// (expert index `experts`: the ids out of range); how many there are.  Every
// workgroup that asks for an expert finds its pairs in one order, so the windows
// of an expert do not overlap.  sums: an int per wave.
//
// A scan costs its instructions: each of the workgroups looks at every id, four
// instructions an id here (with a ballot and a count per 64 ids it was a fifth
// of the whole call at 4096 pairs).
template <int NW>
__device__ __forceinline__ int sk_collect(const SkinnyRoute& route, int e, int lo, int hi, int32_t* list, int32_t* sums) {
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
    // ids from e, or all from `experts` up as unsigned numbers
    const uint32_t span = e == route.experts ? 0u - (uint32_t)e : 1u;
    int seen = 0;  // of the expert's pairs, before this scan
#pragma unroll 1
    for (int base = 0; base < route.pairs && seen < hi; base += 64 * NW * SK_IDS) {
        // a wave takes `per` runs of 64 pairs, one after the other
        const int left = min(route.pairs - base, 64 * NW * SK_IDS), per = (left + 64 * NW - 1) / (64 * NW);
        const int first = 64 * per * w + l;
        const __amdgpu_buffer_rsrc_t ids =
            __builtin_amdgcn_make_buffer_rsrc((void*)(route.ids + base), 0, 4 * left, 0x00020000);
        uint32_t id[SK_IDS], hit = 0;  // bit u: pair first + 64 u is the expert's
#pragma unroll
        for (int u0 = 0; u0 < SK_IDS; u0 += 8)
            if (u0 < per) {
#pragma unroll
                for (int u = u0; u < u0 + 8; ++u) id[u] = __builtin_amdgcn_raw_buffer_load_b32(ids, 4 * first + 256 * u, 0, 0);
            }
#pragma unroll
        for (int u0 = SK_IDS - 8; u0 >= 0; u0 -= 8)
            if (u0 < per) {
#pragma unroll
                for (int u = u0 + 7; u >= u0; --u) hit = (hit << 1) | (id[u] - (uint32_t)e < span ? 1u : 0u);
            }
        const int valid = min(per, (left - first + 63) / 64);  // past it: zeros, or another wave's pairs
        hit &= valid <= 0 ? 0u : ~0u >> (32 - valid);
        const int mine = __popc(hit), incl = (int)wave_scan_incl((uint32_t)mine);
        if (l == 63) sums[w] = incl;
        __syncthreads();
        int r = seen - lo + incl - mine;
#pragma unroll
        for (int k = 0; k < NW; ++k) {
            const int c = __builtin_amdgcn_readfirstlane(sums[k]);
            if (k < w) r += c;
            seen += c;
        }
        while (hit) {
            if (r >= 0 && r < hi - lo) list[r] = base + first + 64 * __builtin_ctz(hit);
            hit &= hit - 1;
            ++r;
        }
        __syncthreads();  // the list is whole; the sums are free
    }
    return max(0, min(seen, hi) - lo);
}

// Routed: the o-th window, of 2^shift pairs, after the first of each expert:
// {expert, which of its windows}, or {-1, ..} past the last.  bins: an int per
// expert and one more; sums: NW + 2.
template <int NW>
__device__ __forceinline__ int2 sk_find_window(const SkinnyRoute& route, int o, int32_t* bins, int32_t* sums) {
    constexpr int NT = 64 * NW;
    const int tid = threadIdx.x, l = tid & 63, w = tid >> 6, n = route.experts + 1;
    for (int i = tid; i < n; i += NT) bins[i] = 0;
    if (tid == 0) sums[NW] = -1;
    __syncthreads();
    auto load = [&](int (&id)[8], int base) {
#pragma unroll
        for (int u = 0; u < 8; ++u) id[u] = route.ids[min(base + NT * u + tid, route.pairs - 1)];
    };
    int id[8], next[8];
    load(id, 0);
#pragma unroll 1
    for (int base = 0; base < route.pairs; base += 8 * NT) {
        if (base + 8 * NT < route.pairs) load(next, base + 8 * NT);
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int bin = (int)min((uint32_t)id[u], (uint32_t)route.experts);
            // lane 0 adds for all lanes of its expert: the ids of a hot one
            // would be 64 adds to one word, one after the other
            const bool in = base + NT * u + tid < route.pairs, same = bin == __builtin_amdgcn_readfirstlane(bin);
            const int n = __popcll(__ballot(in && same));
            if (in && (!same || l == 0)) atomicAdd(&bins[bin], same ? n : 1);
            id[u] = next[u];
        }
    }
    __syncthreads();
    // a thread takes `run` experts one after the other
    const int run = (n + NT - 1) / NT;
    int mine = 0;
    for (int j = tid * run; j < min(n, (tid + 1) * run); ++j) mine += max(0, bins[j] - 1) >> route.shift;
    int incl = (int)wave_scan_incl((uint32_t)mine);
    if (l == 63) sums[w] = incl;
    __syncthreads();
    for (int k = 0; k < w; ++k) incl += sums[k];
    if (o >= incl - mine && o < incl) {
        int at = incl - mine, j = tid * run;
        for (;; ++j) {
            const int more = max(0, bins[j] - 1) >> route.shift;
            if (o < at + more) break;
            at += more;
        }
        sums[NW] = j;
        sums[NW + 1] = o - at + 1;
    }
    __syncthreads();
    const int2 r = make_int2(__builtin_amdgcn_readfirstlane(sums[NW]), __builtin_amdgcn_readfirstlane(sums[NW + 1]));
    __syncthreads();  // bins and sums are free
    return r;
}

// Ring entry: two groups (128 k); W [16 RT rows][64 B] (chunk c of row r in
// slot c ^ ((r >> 2) & 3)), x [16 TT rows][256 B] (slot c ^ (r % 16)), then per
// (row, group) the dword that holds its scale and the one that holds its bias.
//
// Measured as above, before (one wave per output, or the 128-row tiles of
// gemm.hip) -> now: 7168 x 16384, 13 tokens 2280 -> 22 us, 24 tokens 4150 -> 27
// us, 64 tokens 661 -> 44 us; 24576 x 1536, 13 tokens 780 -> 11 us.  One ring
// entry per wave (S = 1, all 8 waves' entries in flight) is as fast as three.
//
// Routed: workgroup (expert, row tile).  It scans the ids for the first window of
// its expert's (token, slot) pairs and takes them 16 TT at a time; expert index
// `experts` stands for the ids out of range, whose outputs are zeros.  Further
// workgroups take the windows that follow a first one: each counts every expert's
// pairs and finds every route.slots-th of them, so that a hot expert is no chain
// of passes.  They cost nothing that could be measured where no expert is hot.
//
// 2 waves and 16 tokens, six workgroups a CU (three waves a SIMD, at most 168
// registers; at 128 and four waves 768 x 2048 takes 1 us more, 2048 x 768 5 less,
// without a bound both are slower): a workgroup is a chain of waits (ids, rows,
// sums).  768 x 2048, 128 experts, 200 tokens of 8 slots, a GEMV per pair -> now:
// spread 207 -> 44 us, half of the slots on one expert 193 -> 54, all on one 190 ->
// 45 (318 and 609 when an expert was one workgroup per row tile).  2048 x 768: 249
// -> 48; 256 experts of 256 x 512, 2048 tokens 263 -> 50.  4 or 8 waves, 32 tokens,
// 64 or 128 rows each were slower with one workgroup per expert.
template <int RT, int TT, int S, int SDT, bool ROUTED, int NW>
__global__ void __launch_bounds__(64 * NW, ROUTED ? 3 : 1) skinny_affine_kernel(ProjGemmParams p, SkinnyRoute route, int blocks) {
    static_assert(RT <= 2, "one DMA of scales per entry");
    extern __shared__ __attribute__((aligned(16))) char lds[];
    constexpr int NI = RT + 4 * TT + 2, XOFF = 1024 * RT, SOFF = XOFF + 4096 * TT, ENTRY = SOFF + 512;
    static_assert((S - 1) * NI < 64, "vmcnt range");
    static_assert(!ROUTED || 4 * (SK_MAX_EXPERTS + 1) <= NW * S * ENTRY, "bins");
    const int tid = threadIdx.x, l = tid & 63, q = l >> 4, lr = l & 15;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    int tile, tb = 0, e = 0;
    const int n_tiles = (p.N + 16 * RT - 1) / (16 * RT);
    int32_t* const list = (int32_t*)(lds + std::max(NW * S * ENTRY, NW * RT * TT * 1024));
    if constexpr (ROUTED) {
        e = blockIdx.x / n_tiles;
        tile = blockIdx.x - e * n_tiles;
    } else {
        sk_tile(blockIdx.x, blocks, tile, tb);
        if (tile >= n_tiles) return;
    }
    const int n0 = tile * 16 * RT, rows = min(16 * RT, p.N - n0);
    const int G = p.K / 64, nblk = (G + 1) / 2;
    const uint32_t wrow = (uint32_t)p.K / 2, srow = (uint32_t)(p.K / p.group) * (SDT == 2 ? 4 : 2);
    const int gpl = p.group / 64;  // 64-groups per scale
    const int n = w < nblk ? (nblk - 1 - w) / NW + 1 : 0;  // this wave's entries
    const char *wbase, *sbase, *bbase;
    i32x4 wres, sres, bres;
    auto set_rows = [&](int64_t first) {  // the weight rows of this workgroup: first + n0 ..
        wbase = (const char*)p.packed + (first + n0) * wrow;
        sbase = (const char*)p.scales + (first + n0) * srow;
        bbase = (const char*)p.biases + (first + n0) * srow;
        wres = uniform_rsrc(wbase, (uint32_t)rows * wrow);
        // (2-byte scales: through the dword that holds the last one)
        sres = uniform_rsrc(sbase, ((uint32_t)rows * srow + 3u) & ~3u);
        bres = uniform_rsrc(bbase, ((uint32_t)rows * srow + 3u) & ~3u);
    };
    if constexpr (!ROUTED) set_rows(0);
    const bf16x8 ones = __builtin_bit_cast(bf16x8, u32x4{0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u});
    f32x4 tot[RT][TT];
    // the products of `toks` tokens: x row and y row of token i from row_of
    auto tokens = [&](int toks, const uint16_t* xb, int64_t xbytes, auto xrow_of, auto yrow_of) {
        uint32_t wo[RT];
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const int row = 16 * r + (l >> 2);
            wo[r] = row < rows ? (uint32_t)row * wrow + 16u * ((l & 3) ^ ((l >> 4) & 3)) : SK_OOB_ROW;
        }
        // lane l of the scale DMA: row l / 2, group l % 2 of the entry
        const uint32_t so = (l >> 1) < rows ? (uint32_t)(l >> 1) * srow : SK_OOB_ROW;
        char* ring = lds + w * S * ENTRY;
        auto issue_w = [&](int i, char* ent) {
            const int blk = w + NW * i;
            const uint32_t o = i < n ? 64u * blk : SK_OOB_K;
#pragma unroll
            for (int r = 0; r < RT; ++r) dma16_buf(wres, wo[r] + o, ent + 1024 * r);
            const int g = min(2 * blk + (l & 1), G - 1);  // a group past the last is not used
            const uint32_t gs = (uint32_t)(gpl == 1 ? g : g / gpl) * (SDT == 2 ? 4 : 2);
            const uint32_t sv = i < n ? (so + gs) & ~3u : SK_OOB_K;
            dma4_buf(sres, sv, ent + SOFF);
            dma4_buf(bres, sv, ent + SOFF + 256);
        };
        const i32x4 xres = uniform_rsrc(xb, (uint32_t)xbytes);
        // lane l of DMA u: row 4 u + l / 16, slot l % 16, chunk slot ^ (row % 16)
        uint32_t xo[TT][4];
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int rt = 4 * u + q, tok = 16 * t + rt;
                xo[t][u] = tok < toks ? (uint32_t)(xrow_of(tok) * p.ldx * 2) + 16u * (lr ^ rt) : SK_OOB_ROW;
            }
        auto issue = [&](int i, int slot) {
            char* ent = ring + slot * ENTRY;
            issue_w(i, ent);
            const int blk = w + NW * i;
            const uint32_t o = i < n ? 256u * (uint32_t)blk : SK_OOB_K;
            // an odd last group: the entry's second half is past the row's
            // end, where the next row or padding may hold a NaN
            const bool half = 2 * blk + 1 == G;
            const uint32_t o2[2] = {half && lr >= 8 ? SK_OOB_K : o, half && lr < 8 ? SK_OOB_K : o};  // u < 2, u >= 2
#pragma unroll
            for (int t = 0; t < TT; ++t)
#pragma unroll
                for (int u = 0; u < 4; ++u) dma16_buf(xres, xo[t][u] + o2[u >> 1], ent + XOFF + 4096 * t + 1024 * u);
        };
        f32x4 part[RT][TT];
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int t = 0; t < TT; ++t) tot[r][t] = part[r][t] = f32x4{};
#pragma unroll
        for (int s = 0; s < S; ++s) issue(s, s);
        int slot = 0;
        for (int i = 0; i < n; ++i) {
            wait_vmcnt<(S - 1) * NI>();
            const char* ent = ring + slot * ENTRY;
            const int blk = w + NW * i;
            u32x2 fw[RT][2], sv[RT], bv[RT];
            bf16x8 fx[TT][2][2];
#pragma unroll
            for (int r = 0; r < RT; ++r) {
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    fw[r][j] = *(const u32x2*)(ent + 1024 * r + 64 * lr + 16 * ((2 * j + (q >> 1)) ^ (lr >> 2)) + 8 * (q & 1));
                sv[r] = *(const u32x2*)(ent + SOFF + 128 * r + 8 * lr);
                bv[r] = *(const u32x2*)(ent + SOFF + 256 + 128 * r + 8 * lr);
            }
#pragma unroll
            for (int t = 0; t < TT; ++t)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int s = 0; s < 2; ++s)
                        fx[t][j][s] = *(const bf16x8*)(ent + XOFF + 4096 * t + 256 * lr + 16 * ((8 * j + 2 * q + s) ^ lr));
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_waitcnt(0xc07f);  // the same, known to the compiler
            __builtin_amdgcn_sched_barrier(0);
            issue(i + S, slot);
            slot = slot + 1 == S ? 0 : slot + 1;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int g = 2 * blk + j;
                const bool live = g < G;
                f32x4 xs[TT];
#pragma unroll
                for (int t = 0; t < TT; ++t) xs[t] = mfma16(fx[t][j][1], ones, mfma16(fx[t][j][0], ones, f32x4{}));
#pragma unroll
                for (int r = 0; r < RT; ++r) {
                    uint32_t sw = sv[r][j], bw = bv[r][j];
                    if (SDT != 2) {  // the half that holds it
                        const uint32_t sh =
                            (((16 * r + lr) * (srow >> 1) + (uint32_t)(gpl == 1 ? g : g / gpl)) & 1u) * 16u;
                        sw = (sw >> sh) & 0xffffu;
                        bw = (bw >> sh) & 0xffffu;
                    }
                    const float s = live ? sk_scale<SDT>(sw) : 0.f, b = live ? sk_scale<SDT>(bw) : 0.f;
                    const bf16x8 w0 = nibbles_bf16(fw[r][j][0]), w1 = nibbles_bf16(fw[r][j][1]);
#pragma unroll
                    for (int t = 0; t < TT; ++t) {
                        const f32x4 d = mfma16(fx[t][j][1], w1, mfma16(fx[t][j][0], w0, f32x4{}));
#pragma unroll
                        for (int k = 0; k < 4; ++k) part[r][t][k] = fmaf(b, xs[t][k], fmaf(s, d[k], part[r][t][k]));
                    }
                }
            }
            if ((i & 3) == 3 || i + 1 == n) {
#pragma unroll
                for (int r = 0; r < RT; ++r)
#pragma unroll
                    for (int t = 0; t < TT; ++t) {
                        tot[r][t] += part[r][t];
                        part[r][t] = f32x4{};
                    }
            }
        }
        wait_vmcnt<0>();
        sk_reduce<RT, TT, NW>(lds, tot, [&](int r, int t, int lane, f32x4 v) {
            const int nn = 16 * r + (lane & 15);
            auto store = [&](int m, int row, float y) {
                const int64_t o = yrow_of(m) * p.ldy + n0 + row;
                if (p.y_f32)
                    ((float*)p.y)[o] = y;
                else
                    ((uint16_t*)p.y)[o] = f32_to_bf16_bits(y);
            };
            uint32_t again = 0;  // values that are not finite
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int m = 16 * t + 4 * (lane >> 4) + i;
                if (nn >= rows || m >= toks) continue;
                if (fabsf(v[i]) < INFINITY)
                    store(m, nn, v[i]);
                else
                    again |= 1u << i;
            }
            if (__builtin_expect(!__ballot(again), 1)) return;
            int finite = -1;
#pragma unroll 1
            for (int i = 0; i < 16; ++i) {
                const uint64_t lanes = __ballot((again >> (i & 3)) & 1u), which = (lanes >> (16 * (i >> 2))) & 0xffffu;
                if (!which) continue;
                const int m = 16 * t + i;
                const float y = sk_affine_again<SDT>(which, xb + xrow_of(m) * p.ldx, wbase + (int64_t)(16 * r) * wrow,
                                                     sbase + (int64_t)(16 * r) * srow, bbase + (int64_t)(16 * r) * srow,
                                                     wrow, srow, p.K, p.group, finite);
                if ((which >> lane) & 1) store(m, 16 * r + lane, y);
            }
        });
    };
    if constexpr (!ROUTED) {
        const int m0 = tb * 16 * TT, toks = min(16 * TT, p.M - m0);
        tokens(toks, p.x + (int64_t)m0 * p.ldx, ((int64_t)(toks - 1) * p.ldx + p.K) * 2,
               [](int i) { return (int64_t)i; }, [&](int i) { return (int64_t)(m0 + i); });
    } else {
        const int32_t* pairs = list + NW;
        // the first window of expert e; or, past the experts, every
        // route.slots-th of the windows that follow a first one
        const bool later = e > route.experts;
#pragma unroll 1
        for (int o = e - route.experts - 1;; o += route.slots) {
            int window = 0;
            if (later) {
                const int2 f = sk_find_window<NW>(route, o, (int32_t*)lds, list);
                if (f.x < 0) return;
                e = f.x;
                window = f.y;
            }
            const int lo = window << route.shift;
            const int cnt = sk_collect<NW>(route, e, lo, lo + (1 << route.shift), list + NW, list);
            set_rows((int64_t)min(e, route.experts - 1) * p.N);
#pragma unroll 1
            for (int i0 = 0; i0 < cnt; i0 += 16 * TT) {
                const int toks = min(16 * TT, cnt - i0);
                if (e == route.experts) {
                    for (int i = tid; i < toks * rows; i += 64 * NW) {
                        const int64_t y = (int64_t)pairs[i0 + i / rows] * p.ldy + n0 + i % rows;
                        if (p.y_f32)
                            ((float*)p.y)[y] = 0.f;
                        else
                            ((uint16_t*)p.y)[y] = 0;
                    }
                } else {
                    tokens(toks, p.x, ((int64_t)(p.M - 1) * p.ldx + p.K) * 2,
                           [&](int i) { return (int64_t)((uint32_t)pairs[i0 + i] / (uint32_t)route.per_token); },
                           [&](int i) { return (int64_t)pairs[i0 + i]; });
                }
                __syncthreads();  // partial sums and the list are read before they are written again
            }
            if (!later) return;
        }
    }
}

// Token tiles of 16 per workgroup
int token_tiles(int m) { return m <= 16 ? 1 : (m <= 32 ? 2 : 4); }

int64_t workgroups(int64_t n, int m, int rt) {
    const int tt = token_tiles(m);
    return ((n + 16 * rt - 1) / (16 * rt) + 7) / 8 * 8 * (((int64_t)m + 16 * tt - 1) / (16 * tt));
}

// Workgroups of 512 threads, in a grid of less than 2^32 threads
bool grid_ok(int64_t n, int m, int rt) { return workgroups(n, m, rt) < (1 << 23); }

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
    hipLaunchKernelGGL(kern, dim3((unsigned)workgroups(p.N, p.M, RT)), dim3(64 * NW), lds, st, p, (p.M + 16 * TT - 1) / (16 * TT));
    return hipGetLastError();
}

template <int RT, int TT, int S, int SDT, bool ROUTED, int NW>
hipError_t launch_affine(const ProjGemmParams& p, const SkinnyRoute& route, hipStream_t st) {
    constexpr size_t ring = std::max<size_t>((size_t)NW * S * (1024 * RT + 4096 * TT + 512), (size_t)NW * RT * TT * 1024);
    const size_t lds = ring + (ROUTED ? 4 * (NW + std::max(2, 1 << route.shift)) : 0);
    static_assert(ring + 4 * (NW + (1 << SK_WINDOW_MAX_LOG2)) <= 163840, "LDS");
    const auto kern = skinny_affine_kernel<RT, TT, S, SDT, ROUTED, NW>;
    const hipError_t e = set_lds(kern, lds);
    if (e != hipSuccess) return e;
    const int tiles = (p.N + 16 * RT - 1) / (16 * RT), blocks = (p.M + 16 * TT - 1) / (16 * TT);
    const unsigned grid = (unsigned)(ROUTED ? tiles * (route.experts + 1 + route.slots) : workgroups(p.N, p.M, RT));
    hipLaunchKernelGGL(kern, dim3(grid), dim3(64 * NW), lds, st, p, route, blocks);
    return hipGetLastError();
}

template <int RT, int TT, int S, bool ROUTED, int NW>
hipError_t launch_affine_sdt(const ProjGemmParams& p, const SkinnyRoute& route, hipStream_t st) {
    if (p.scale_dtype == 0) return launch_affine<RT, TT, S, 0, ROUTED, NW>(p, route, st);
    if (p.scale_dtype == 1) return launch_affine<RT, TT, S, 1, ROUTED, NW>(p, route, st);
    return launch_affine<RT, TT, S, 2, ROUTED, NW>(p, route, st);
}

bool affine_rows_ok(const ProjGemmParams& p) {
    if (p.bits != 4 || p.group % 64 || p.K % p.group || ((uintptr_t)p.packed & 15)) return false;
    if (((uintptr_t)p.scales | (uintptr_t)p.biases) & 3) return false;
    // 2-byte scales are read by the dword that holds them: every tile's first
    // one and the end of all rows on a dword
    if (p.scale_dtype != 2 && ((int64_t)p.N * (p.K / p.group)) % 2) return false;
    return (int64_t)64 * (p.K / 2) < (1 << 30);
}

}  // namespace

bool skinny_gemm_ok(const ProjGemmParams& p) {
    if (p.M <= 0 || p.N <= 0 || p.K < 32 || p.K % 32 || ((uintptr_t)p.x & 15) || p.ldx % 8 || p.ldx < p.K) return false;
    if ((int64_t)64 * p.ldx * 2 >= (1 << 30)) return false;  // byte offsets of one token block's rows
    if (!grid_ok(p.N, p.M, p.packed ? 2 : 3)) return false;
    if (p.packed) return affine_rows_ok(p);
    return p.w && ((uintptr_t)p.w & 15) == 0 && p.ldw % 8 == 0 && p.ldw >= p.K && (int64_t)64 * p.ldw * 2 < (1 << 30);
}

bool skinny_routed_ok(const ProjGemmParams& p, const SkinnyRoute& route) {
    return p.packed && skinny_gemm_ok(p) && (int64_t)p.M * p.ldx * 2 < (1 << 30) && route.pairs < (1 << 30) &&
           route.experts < SK_MAX_EXPERTS && ((int64_t)p.N / 32 + 1) * (route.experts + 1 + route.pairs / 16) < (1 << 25);
}

namespace {

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
        if (grid_ok(n, m, rt) && dense_cost(n, m, rt, cus) < dense_cost(n, m, best, cus)) best = rt;
    return best;
}

}  // namespace

// Against the large tiles, both in rounds of one workgroup per CU.  Dense
// (gemm.hip): a unit of dense_cost takes 1.65 ns per k (52 us at 12288 x 7168, 64
// tokens), a round of tiles 17.5 ns per k (128 us there).  Over 14 shapes and 64 to
// 512 tokens it never picks a kernel more than 5% slower than the tiles; the
// few-token tiles would still be 5 to 25% faster at some sizes of 129 to 300 tokens
// (12288 x 7168: 129 tokens 91 against 117 us, 192 tokens 105 against 121; 7168 x
// 12288: 300 tokens 162 against 212).  Affine (affine_gemm.hip): a round of 32 rows
// x 64 tokens takes 2.25 ns per k and 3.5 us (7168 x 16384: 128 tokens 81 us, there
// 194; 500 tokens 290, there 209; 24576 x 1536: 64 tokens 24, there 25, 300 tokens
// 104, there 52); over 13 shapes within 5% of the better one, but for 12288 x 7168
// at 129 tokens (100 us, the other 94).
bool skinny_gemm_better(int64_t n, int m, int k, bool affine, int cus) {
    if (m < PROJ_GEMM_MIN_TOKENS) return true;
    if (affine) {
        const int64_t wgs = (int64_t)((n + 31) / 32) * ((m + 63) / 64);
        return (double)((wgs + cus - 1) / cus) * (k * 2.25e-3 + 3.5) < affine_gemm_cost(n, m, k, cus);
    }
    const int64_t tiles = (int64_t)((m + 127) / 128) * ((n + 255) / 256), rounds = (tiles + cus - 1) / cus;
    return dense_cost(n, m, dense_rt(n, m, cus), cus) * 1.65 < 17.5 * rounds;
}

hipError_t launch_skinny_gemm(const ProjGemmParams& p, int cu_count, hipStream_t st) {
    const int tt = token_tiles(p.M);
    if (p.packed) {
        const SkinnyRoute none{};
        if (tt == 1) return launch_affine_sdt<2, 1, 1, false, 8>(p, none, st);
        if (tt == 2) return launch_affine_sdt<2, 2, 1, false, 8>(p, none, st);
        return launch_affine_sdt<2, 4, 1, false, 8>(p, none, st);
    }
    const int rt = dense_rt(p.N, p.M, cu_count);
    if (tt == 1) return rt == 1 ? launch_dense<1, 1, 4, 8>(p, st) : (rt == 2 ? launch_dense<2, 1, 3, 8>(p, st) : launch_dense<3, 1, 2, 8>(p, st));
    if (tt == 2) return rt == 1 ? launch_dense<1, 2, 3, 8>(p, st) : (rt == 2 ? launch_dense<2, 2, 2, 8>(p, st) : launch_dense<3, 2, 2, 8>(p, st));
    return rt == 1 ? launch_dense<1, 4, 2, 8>(p, st) : (rt == 2 ? launch_dense<2, 4, 3, 8>(p, st) : launch_dense<3, 4, 2, 8>(p, st));
}

// Than a GEMV per pair.  Pays once an expert has two tokens (128 experts of 768 x
// 2048, 256 pairs 35 against 31 us, 128 pairs 20 against 27), and once the GEMV,
// about 4.5 us and 14e12 weights a second, takes longer than a workgroup's chain
// of waits, 6 to 13 us by K (8 experts of 1408 x 2048, 32 pairs, 92e6 weights:
// 11.5 against 13.0 us, 40 pairs 17.8 against 13.1; 64 of 512 x 1024, 128 pairs,
// 67e6: 10.4 against 10.6, with half of them to one expert 9.5 against 13.8, 160
// pairs 18.2 against 10.7; 256 of 256 x 512, 512 pairs, 67e6: 13.1 against 13.5,
// with half to one 12.0 against 15.2, 768 pairs 17.7 against 14).
bool skinny_routed_better(int64_t pairs, int64_t experts, int64_t n, int64_t k) {
    return pairs >= 2 * experts && (double)pairs * (double)n * (double)k >= std::max(68e6, 35e6 + 32.4e3 * (double)k);
}

// Windows of 16 pairs (one pass) up to twice the mean of an expert, so that few
// experts have a second one; but where the experts alone do not fill the GPU, four
// workgroups a CU, no more than lets the windows fill it (one expert of 768 x 2048,
// 512 pairs: 16.5 us, 61 by the GEMV).  As many workgroups for the windows that
// follow a first one: half as many took 1.5 times as long at 2048 x 768, 200 tokens
// of 8 slots all on one expert (62 us now, 248 by the GEMV).
hipError_t launch_skinny_routed(const ProjGemmParams& p, const SkinnyRoute& r, int cu_count, hipStream_t st) {
    SkinnyRoute route = r;
    const int tiles = (p.N + 31) / 32;
    route.shift = 4;
    while (route.shift < SK_WINDOW_MAX_LOG2 && ((int64_t)route.experts << route.shift) < 2 * (int64_t)route.pairs &&
           ((int64_t)tiles * route.experts >= 4 * cu_count || ((int64_t)tiles * route.pairs >> (route.shift + 1)) >= 4 * cu_count))
        ++route.shift;
    route.slots = std::min(route.pairs >> route.shift, (4 * cu_count + tiles - 1) / tiles);
    return launch_affine_sdt<2, 1, 1, true, 2>(p, route, st);
}

}  // namespace mr
