// The Gomoku search kernels on the CPU (hip/hip_runtime.h).  layout.inc is the engine's own choice of a workgroup, as it stands in
// mctsnc_engine.hip.
#include "gomoku_kernels.hpp"
#include "mctsnc_hip.h"
#include "simt.h"
#include <stdlib.h>
#include <algorithm>
#include <memory>
#include <vector>

using namespace mctsnc;
namespace {
#include "layout.inc"
template <bool ACP, int W> void search(const void *args) { gomoku::search_kernel<ACP, W>(*static_cast<const gomoku::SearchArgs *>(args)); }
struct Reset { const gomoku::TreeRef *refs; int n; const uint32_t *bb; const int32_t *turns; };
void reset(const void *args) { const Reset &r = *static_cast<const Reset *>(args); gomoku::reset_kernel(r.refs, r.n, r.bb, r.turns); }
}

extern "C" int64_t simt_gomoku_kernel_lds(int words, int acp) { return (int64_t)gomoku::kernel_lds_bytes(words, acp != 0); }
extern "C" int64_t simt_gomoku_cu_lds() { return (int64_t)gomoku::kLdsBytes; }

// The layout of a search: threads, slots, boards of times, dynamic LDS; and what the kernel puts there, in bytes: the lists, the boards
// of times, a ring of offsets for every 64 slots (counted from playout_shape and the ring's format).
extern "C" void simt_gomoku_layout(int m, int n, int P, int acp, int tree_per_cu, int64_t *out) {
    mctsnc_config c = {};
    c.board_m = m; c.board_n = n; c.max_actions = m * n; c.n_playouts = P;
    const bool wide = gomoku_words(c) > 8;
    const GomokuLayout layout = gomoku_layout(c, acp != 0, tree_per_cu != 0);
    const gomoku::PlayoutShape shape = gomoku::playout_shape(m, n, wide, acp != 0);
    const int64_t cell = wide ? 2 : 1;
    out[0] = layout.threads; out[1] = layout.slots; out[2] = layout.teams; out[3] = (int64_t)layout.lds;
    out[4] = cell * shape.list_rows * layout.slots; out[5] = cell * shape.time_rows * 64 * layout.teams;
    out[6] = (int64_t)(layout.slots / 64) * gomoku::kRingChunks * gomoku::kChunk / 4 * 64 * (int64_t)sizeof(gomoku::u32x2);
}

// One search of `trees` trees of a workgroup count G each, `launches` times nsteps steps.  nodes: per tree S records of
// node_bytes; stats: per tree S times 4 int32; sizes: nodes of each tree; rng_*: states, before and after.  0, or -1: given up.
extern "C" int simt_gomoku(int m, int n, int trees, int P, int acp, int thrifty, int G, int tree_per_cu, int S, int nsteps, int launches, float ucb_c, int prep_levels, int xccs, unsigned seed,
                           const uint32_t *root_bb, int turn, uint64_t *rng_playout, uint64_t *rng_expand, unsigned char *nodes, int32_t *stats, int32_t *sizes, int32_t *layout_out) {
    mctsnc_config c = {};
    c.board_m = m; c.board_n = n; c.max_actions = m * n; c.n_playouts = P;
    const int W = gomoku_words(c), A = m * n;
    const GomokuLayout layout = gomoku_layout(c, acp != 0, tree_per_cu != 0);
    const size_t rec = (size_t)gomoku::node_bytes(W);
    // (every array on its own and of its exact size)
    std::vector<std::unique_ptr<simt::Guarded>> keep;
    auto make = [&](size_t bytes, size_t alignment) -> void * {   // (every array on its own and of its exact size)
        keep.emplace_back(new simt::Guarded(bytes, alignment));
        return keep.back()->get();
    };
    std::vector<gomoku::TreeRef> refs((size_t)trees);
    std::vector<uint32_t> bb; std::vector<int32_t> turns((size_t)trees, turn);
    for (int t = 0; t < trees; t++) {
        gomoku::TreeRef &r = refs[t];
        r.nodes = static_cast<gomoku::Node *>(make(rec * S, 128)); r.stats = static_cast<gomoku::Stat *>(make(sizeof(gomoku::Stat) * S, 16));
        r.hdr = static_cast<gomoku::TreeHdr *>(make(sizeof(gomoku::TreeHdr), 128));
        memset(r.nodes, 0xa5, rec * S); memset(r.stats, 0xa5, sizeof(gomoku::Stat) * S); memset(r.hdr, 0, sizeof(gomoku::TreeHdr));   // (as the engine leaves it)
        const size_t per_tree = (size_t)(acp ? A * P : P) * 2;
        r.rng_playout = rng_playout + per_tree * t; r.rng_expand = acp ? nullptr : rng_expand + 2 * t;
        r.ae = static_cast<int16_t *>(make(2 * (A + 2), 2)); r.root_ae = static_cast<int16_t *>(make(2 * (A + 2), 2));
        r.poc = static_cast<int32_t *>(make(8 * A, 4)); r.path = static_cast<int32_t *>(make(4 * (A + 2), 4));
        memset(r.ae, 0, 2 * (A + 2)); memset(r.poc, 0, 8 * A);
        r.words = W;
        bb.insert(bb.end(), root_bb, root_bb + 2 * W);
    }
    const Reset rs{refs.data(), trees, bb.data(), turns.data()};
    simt::run({(trees + 63) / 64, 64, 0, seed, 1, reset, &rs});
    int32_t abort_flag = 0;
    gomoku::SearchArgs args = {};
    args.refs = refs.data(); args.n_refs = trees; args.m = m; args.n = n; args.P = P; args.G = acp ? G : 1; args.slots = layout.slots; args.teams = layout.teams;
    args.S = S; args.nsteps = nsteps; args.thrifty = thrifty; args.ucb_c = ucb_c; args.prep_levels = prep_levels; args.abort_flag = &abort_flag; args.spin_limit = 1u << 30;
    void (*const kernel)(const void *) = acp ? (W == 8 ? search<true, 8> : W == 12 ? search<true, 12> : search<true, 16>)
                                             : (W == 8 ? search<false, 8> : W == 12 ? search<false, 12> : search<false, 16>);
    for (int l = 0; l < launches; l++) simt::run({args.G * trees, layout.threads, layout.lds, seed + 1 + l, xccs, kernel, &args});
    for (int t = 0; t < trees; t++) {
        sizes[t] = refs[t].hdr->size;
        memcpy(nodes + rec * S * t, refs[t].nodes, rec * (size_t)std::min(S, sizes[t]));
        memcpy(stats + (size_t)4 * S * t, refs[t].stats, sizeof(gomoku::Stat) * (size_t)std::min(S, sizes[t]));
    }
    layout_out[0] = layout.threads; layout_out[1] = layout.slots; layout_out[2] = layout.teams;
    return abort_flag ? -1 : 0;
}
