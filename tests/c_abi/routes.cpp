// The host rules by which a call takes one kernel or another, behind plain C
// functions for tests/test_routes.py.  Nothing here touches a GPU.
#include "mr_kernels.hpp"

namespace {
// aligned as a device allocation is; never dereferenced
void* at(uintptr_t n) { return reinterpret_cast<void*>(n << 20); }
}  // namespace

extern "C" {

int route_index_run(int tokens, int heads, int dim, int keys, int cus) {
    mr::IndexerParams p{};
    p.q = at(1);
    p.k = at(2);
    p.w = at(3);
    p.out = (float*)at(4);
    p.w_f32 = 1;
    p.q_hs = dim;
    p.q_ss = (int64_t)heads * dim;
    p.k_rs = dim;
    p.w_ss = heads;
    p.out_ss = keys;
    p.S = tokens;
    p.H = heads;
    p.D = dim;
    p.T = keys;
    return mr::indexer_run(p, cus);
}

int route_topk_sorts(int rows, int available, int ratio, int start_pos, int selected, int cus) {
    mr::TopkParams p{};
    p.rows = rows;
    p.cols = p.available = available;
    p.ratio = ratio;
    p.start_pos = start_pos;
    p.selected = selected;
    return mr::topk_sorts_whole(p, cus);
}

// mr::ProjRoute of bf16 tokens through a dense weight (group 0) or a 4-bit affine
// one; tile_rows: token rows of a tile where the route has tiles
int route_projection(int tokens, int out_features, int in_features, int group, int scale_dtype, int x_pad, int y_f32,
                     int cus, int* tile_rows) {
    mr::ProjGemmParams p{};
    p.x = (const uint16_t*)at(1);
    p.ldx = in_features + x_pad;
    if (group) {
        p.packed = at(2);
        p.scales = at(3);
        p.biases = at(4);
        p.scale_dtype = scale_dtype;
        p.group = group;
        p.bits = 4;
    } else {
        p.w = (const uint16_t*)at(2);
        p.ldw = in_features;
    }
    p.y = at(5);
    p.ldy = out_features;
    p.y_f32 = y_f32;
    p.M = tokens;
    p.N = out_features;
    p.K = in_features;
    const mr::ProjRoute r = mr::proj_route(p, cus);
    const int64_t n_tiles = (out_features + 255) / 256;
    *tile_rows = r == mr::PROJ_TILES         ? mr::proj_gemm_rows(n_tiles, tokens, cus)
                 : r == mr::PROJ_GROUP_TILES ? mr::affine_gemm_rows(n_tiles, tokens, in_features, cus)
                                             : 0;
    return r;
}

// whether projections of `rows` weight rows in all, of the same tokens, run as one
// stacked launch of large tiles (the others being takeable by both kinds)
int route_stack(int tokens, int rows, int in_features, int affine, int cus) {
    return tokens >= mr::PROJ_GEMM_MIN_TOKENS && !mr::skinny_gemm_better(rows, tokens, in_features, affine, cus);
}

// -1: a GEMV per pair
int route_gather(int tokens, int experts, int per_token, int out_features, int in_features, int group) {
    mr::ProjGemmParams p{};
    p.x = (const uint16_t*)at(1);
    p.ldx = in_features;
    p.packed = at(2);
    p.scales = at(3);
    p.biases = at(4);
    p.group = group;
    p.bits = 4;
    p.y = at(5);
    p.ldy = out_features;
    p.M = tokens;
    p.N = out_features;
    p.K = in_features;
    const mr::SkinnyRoute r{(const int32_t*)at(6), tokens * per_token, per_token, experts, 0, 0};
    return mr::skinny_routed_better(r.pairs, experts, p.N, p.K) && mr::skinny_routed_ok(p, r) ? mr::PROJ_FEW : -1;
}

}  // extern "C"
