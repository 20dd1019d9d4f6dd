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

}  // extern "C"
