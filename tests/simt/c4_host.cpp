// The Connect 4 search kernels on the CPU (hip/hip_runtime.h).
#include "c4_kernels.hpp"
#include "simt.h"
#include <algorithm>
#include <memory>
#include <vector>

using namespace mctsnc;
namespace {
template <void (*KERNEL)(c4::SearchArgs)> void search(const void *args) { KERNEL(*static_cast<const c4::SearchArgs *>(args)); }
struct Reset { const c4::TreeRef *refs; int n; const uint64_t *bb; const int32_t *turns; };
void reset(const void *args) { const Reset &r = *static_cast<const Reset *>(args); c4::reset_kernel(r.refs, r.n, r.bb, r.turns); }
enum Form { kPlain, kSplit, kPool, kSolo };
}

// One search of `trees` trees in `launches` times nsteps steps by workgroups of `threads` threads (split: four wavefronts).
// nodes: per tree S records of 128 bytes; sizes: nodes, root visits and root wins of each tree; rng_*: states, before and
// after.  0, or -1: given up.
extern "C" int simt_c4(int m, int n, int trees, int P, int acp, int thrifty, int form, int threads, int S, int nsteps, int launches, float ucb_c, int agent_fences, int xccs, unsigned seed,
                       const uint64_t *root_bb, int turn, uint64_t *rng_playout, uint64_t *rng_expand, unsigned char *nodes, int32_t *sizes) {
    std::vector<std::unique_ptr<simt::Guarded>> keep;
    auto make = [&](size_t bytes, size_t alignment) -> void * {   // (every array on its own and of its exact size)
        keep.emplace_back(new simt::Guarded(bytes, alignment));
        return keep.back()->get();
    };
    std::vector<c4::TreeRef> refs((size_t)trees);
    std::vector<uint64_t> bb; std::vector<int32_t> turns((size_t)trees, turn);
    for (int t = 0; t < trees; t++) {
        c4::TreeRef &r = refs[t];
        r.nodes = static_cast<c4::Node *>(make(sizeof(c4::Node) * S, 128)); r.hdr = static_cast<c4::TreeHdr *>(make(sizeof(c4::TreeHdr), 128));
        memset(r.nodes, 0xa5, sizeof(c4::Node) * S); memset(r.hdr, 0, sizeof(c4::TreeHdr));   // (the header as the engine leaves it)
        r.rng_playout = rng_playout + (size_t)(acp ? n * P : P) * 2 * t; r.rng_expand = acp ? nullptr : rng_expand + 2 * t;
        bb.insert(bb.end(), root_bb, root_bb + 2);
    }
    const Reset rs{refs.data(), trees, bb.data(), turns.data()};
    simt::run({(trees + 63) / 64, 64, 0, seed, 1, reset, &rs});
    int32_t abort_flag = 0;
    const int parts = form == kSplit && acp ? std::max(1, P / 64) : 1;
    c4::SearchArgs args = {};
    args.refs = refs.data(); args.n_refs = trees; args.m = m; args.n = n; args.P = P; args.G = acp && form != kSolo ? n * parts : 1; args.parts = parts;
    args.S = S; args.nsteps = nsteps; args.thrifty = thrifty; args.ucb_c = ucb_c; args.agent_fences = agent_fences; args.abort_flag = &abort_flag; args.spin_limit = 1u << 30;
    if (form == kSplit) threads = c4::kSplitThreads;
    const size_t lds = form == kSolo ? c4::solo_lds_bytes(m, n, P) : form == kPool ? c4::team_pool_lds_bytes(m, n, P) : form == kSplit ? c4::split_lds_bytes(m, n) : c4::search_lds_bytes(m, n);
    void (*const kernel)(const void *) = form == kSolo ? search<c4::search_kernel_solo> : form == kPool ? search<c4::search_kernel_team_pool>
                                         : form == kSplit ? (acp ? search<c4::search_kernel_split<true>> : search<c4::search_kernel_split<false>>)
                                                          : (acp ? search<c4::search_kernel<true>> : search<c4::search_kernel<false>>);
    for (int l = 0; l < launches; l++) simt::run({args.G * 8 * ((trees + 7) / 8), threads, lds, seed + 1 + l, xccs, kernel, &args});
    for (int t = 0; t < trees; t++) {
        sizes[3 * t] = refs[t].hdr->size; sizes[3 * t + 1] = refs[t].hdr->root_ns; sizes[3 * t + 2] = refs[t].hdr->root_wins;
        memcpy(nodes + sizeof(c4::Node) * S * t, refs[t].nodes, sizeof(c4::Node) * (size_t)std::min(S, sizes[3 * t]));
    }
    return abort_flag ? -1 : 0;
}
