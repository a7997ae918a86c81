// Gomoku PUCT search loop with virtual loss behind include/puct_gomoku.h: selection, expansion / evaluation and backup of
// all steps of a search in one launch, one workgroup per tree and one wavefront per traversal, on the loop's own tree
// storage (one 16-byte record per edge, one per node), and the host engine.  A tree belongs to one workgroup for the
// whole launch, so the traversals' claims are taken in a fixed order on registers instead of with atomics in memory,
// which also makes a search reproducible.
#include <chrono>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "puct_device.hpp"
#include "puct_row.h"
#include "puct_synthetic.h"
#include "../../include/puct_gomoku.h"

namespace {
using namespace puct;

constexpr int kEdges = 256;       // edge slots per node (MAX_ACTION of src/puct/puct_gpu_v2.py:72)
constexpr int kBoardWords = 16;   // 8 words per colour

struct Edge {
    int n;          // visits
    float w;        // value sum, for the player who moves along the edge
    float prior;
    uint32_t link;  // child << 8 | claims in flight (virtual loss); child 0 = none (node 0 is the root)
};
static_assert(sizeof(Edge) == 16, "one edge is one 16-byte load");

struct NodeInfo {
    int expanded;    // edge slots with a child, or PUCT_NODE_EXPANDED_TERMINAL
    int tickets;     // expansion tickets in flight
    int legal_turn;  // empty cells of the position (most children the node can have) | 0x10000 if -1 is to move
    float value;     // of the position for its player to move
};
static_assert(sizeof(NodeInfo) == 16, "one node word is one 16-byte load");
constexpr int kTurnBit = 0x10000;

constexpr int kTrav = kMaxWavesPerBlock;   // most traversals per tree: one wavefront each, one workgroup per tree
constexpr int kSlices = kEdges / kWave;    // 64-edge slices of the widest node
constexpr int kRow = 16;                   // lanes of a DPP row
constexpr int kTally = 12;

struct LoopArgs {
    Edge *edges;       // [trees][max_nodes][256]
    NodeInfo *info;    // [trees][max_nodes]
    uint32_t *board;   // [trees][max_nodes][16]
    uint8_t *action;   // [trees][max_nodes][256]: cell of every edge slot
    int *node_count;   // [trees]
    // what the traversals of the last step ended with, [trees][traversals] (paths: [trees][traversals][path_depth])
    int *out_selected, *out_len, *out_claims, *out_path;
    float *out_value;
    unsigned long long *tally;   // [trees][12]: selections by kind (0..4), children created (5), nodes read (6), edges scored (7),
                                 // ticks of the 100 MHz clock that wavefront 0 spent selecting (8), expanding (9), backing up (10)
    float cpuct, c_pw, alpha_pw;
    int m, n, cells, max_nodes, traversals, path_depth, steps;
    uint64_t seed;
    float dirichlet_alpha;
    struct EvalRequests *requests;   // [trees]
    int evaluators;                  // workgroups per tree that work out the priors of new nodes (fused search), 0 = none
    int agent_fences;                // hand-overs between a tree and its evaluators always write the L2 back
};

// What a tree's workgroup hands to its evaluator workgroups, step by step: the non-terminal children the step created.
struct EvalRequests {
    unsigned long long tag;   // posted() once the step's entries are complete; kSearchOver when there are no more
    int done;    // entries the evaluators have worked off since the search began
    int abort;   // a bounded wait gave up: everybody leaves
    int child[kMaxWavesPerBlock];       // node to evaluate, -1 = nothing to do for this entry
    uint64_t hash[kMaxWavesPerBlock];   // its position's hash
    int xcc[1 + 8];                     // XCD that the tree's workgroup [0] and its evaluators [1..] run on, -1 = not known yet
};
constexpr int kMaxEvaluators = 8;
// All that an evaluator needs to know before it can ask for a step's entries, in the word that it waits for: the step, how many
// entries there are (0..16) and the first's node (20 bits; the others follow it).
constexpr unsigned long long kSearchOver = ~0ull;
__device__ __forceinline__ unsigned long long posted(int step, int n, int first) {
    return (uint32_t)(step + 1) | (unsigned long long)n << 32 | (unsigned long long)first << 40;
}
static_assert(sizeof(EvalRequests::xcc) == sizeof(int) * (1 + kMaxEvaluators), "one entry per workgroup of a tree");

__device__ __forceinline__ int my_xcc() { return (int)(__builtin_amdgcn_s_getreg(6164) & 0xfu); }   // HW_REG_XCC_ID, bits 3:0
constexpr unsigned long long kWaitTicks = 300000000ull;   // 3 s of the 100 MHz clock: a partner that is not there

constexpr int kReachedNothing = 0, kReachedValued = 1 /* by s.value */, kReachedPosition = 2, kReachedChild = 3, kReachedWin = 4, kReachedDraw = 5;

// What a step keeps per traversal between its phases.  The paths ([traversals][path_depth] words) follow in dynamic LDS.
struct StepLds {
    int cur[2][kTrav];   // node every traversal stands on, -1 once it has ended; double buffered by level parity
    int sel[kTrav];      // selection word: kind << 28 | slot << 20 | node
    int len[kTrav];      // path length as reported (nodes on the path; 0 for a traversal that reached no node)
    int claims[kTrav];   // edges the traversal holds a claim on = path entries written
    float value[kTrav];  // of the reached node, for the player who moved into it
    int want[kTrav];     // node the traversal expands, -1 if none
    int4 reached[kTrav]; // what the expansion makes of the traversal: kReached..., and of a new child its node, its edge
                         // (parent << 8 | slot) and its NodeInfo::legal_turn
    unsigned long long hash[kTrav];   // of the position on `board`
    int node_count;
    int requests;        // evaluation requests of this step
    int requested;       // ... and of all steps so far
    int gave_up;
    uint32_t board[kTrav][kBoardWords];
    alignas(16) int stage[kTrav][5 * kRow];   // per wavefront: edges on their way from four per lane to one per lane
};

__device__ __forceinline__ int pack_sel(int kind, int node, int slot) {
    return (kind << PUCT_GOMOKU_SEL_KIND_SHIFT) | (slot << PUCT_GOMOKU_SEL_SLOT_SHIFT) | node;
}

__device__ __forceinline__ uint64_t wave_sum64(uint64_t v) {
    auto step = [](uint64_t x, auto ctrl) {
        constexpr int C = decltype(ctrl)::value;
        const uint32_t lo = (uint32_t)dpp<C>((int)(uint32_t)x);
        const uint32_t hi = (uint32_t)dpp<C>((int)(uint32_t)(x >> 32));
        return x + (((uint64_t)hi << 32) | lo);
    };
    v = step(v, std::integral_constant<int, 0xB1>{});
    v = step(v, std::integral_constant<int, 0x4E>{});
    v = step(v, std::integral_constant<int, 0x141>{});
    v = step(v, std::integral_constant<int, 0x140>{});
    return read_lane64(v, 0) + read_lane64(v, 16) + read_lane64(v, 32) + read_lane64(v, 48);
}

// Orders this wavefront's LDS writes before its later LDS reads by other lanes.
__device__ __forceinline__ void wave_lds_fence() { __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup"); }

__device__ __forceinline__ bool stone_at(const uint32_t *colour, int cell) { return (colour[cell >> 5] >> (cell & 31)) & 1u; }

// Does the stone just placed at `cell` complete a row of exactly five (src/mctsnc_game_mechanics.py:181-280: a longer
// row does not win)?  Lane 16 d + 5 + k looks at the cell k steps along direction d; the result is uniform.
__device__ __forceinline__ bool makes_five(const uint32_t *mine, int cell, int m, int n, int lane) {
    const int d = lane >> 4, k = (lane & 15) - 5;
    const int row = (int)(((float)cell + 0.5f) * __builtin_amdgcn_rcpf((float)n));   // (cell < 256: half a cell is far more than the reciprocal's error)
    const int r = row + (d == 0 ? 0 : k), c = cell - row * n + (d == 0 || d == 2 ? k : (d == 1 ? 0 : -k));
    const uint64_t like = __ballot(k <= 5 && r >= 0 && r < m && c >= 0 && c < n && stone_at(mine, r * n + c));
    const uint32_t line = (uint32_t)(like >> (16 * (lane & 3))) & 0x7FFu;   // bit 5: the stone itself
    return __ballot(1 + __builtin_clz(~(line << 27)) + __builtin_ctz(~(line >> 6)) == 5) != 0;
}

// This lane's key and that of lane ^ LANE_XOR, in any order, by vector instructions alone: DPP moves (4: the two directions, each to
// its banks of four lanes), and beyond a row of 16 the swaps of rows and halves, after which one register has the lower partner's
// key on both sides and the other the upper's.
struct KeyPair {
    uint32_t a, b;
};
template <int LANE_XOR>
__device__ __forceinline__ KeyPair with_partner(uint32_t x) {
    if constexpr (LANE_XOR == 1) return {x, (uint32_t)dpp<0xB1>((int)x)};    // quad_perm [1,0,3,2]
    if constexpr (LANE_XOR == 2) return {x, (uint32_t)dpp<0x4E>((int)x)};    // quad_perm [2,3,0,1]
    if constexpr (LANE_XOR == 4) {
        const int up = __builtin_amdgcn_update_dpp((int)x, (int)x, 0x104, 0xF, 0x5, false);            // row_shl:4
        return {x, (uint32_t)__builtin_amdgcn_update_dpp(up, (int)x, 0x114, 0xF, 0xA, false)};         // row_shr:4
    }
    if constexpr (LANE_XOR == 8) return {x, (uint32_t)dpp<0x128>((int)x)};   // row_ror:8
    if constexpr (LANE_XOR == 16) {
        const auto v = __builtin_amdgcn_permlane16_swap(x, x, false, false);
        return {v[0], v[1]};
    }
    const auto v = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    return {v[0], v[1]};
}
__device__ __forceinline__ uint32_t larger_key(KeyPair p) { return p.a > p.b ? p.a : p.b; }
__device__ __forceinline__ uint32_t smaller_key(KeyPair p) { return p.a > p.b ? p.b : p.a; }

// Bitonic sort of the wavefront's 256 keys, largest first: element e = 4 * lane + k lives in v[k] of `lane`.  Partners
// at element distance 1 and 2 are registers of the same lane.
template <int SIZE, int DIST>
__device__ __forceinline__ void bitonic_step(uint32_t (&v)[4], int lane) {
    KeyPair pair[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        if constexpr (DIST < 4) pair[k] = {v[k], v[k ^ DIST]};
        else pair[k] = with_partner<DIST / 4>(v[k]);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int e = 4 * lane + k;
        const bool descending = (e & SIZE) == 0, first = (e & DIST) == 0;   // SIZE == 256: every block descends
        v[k] = (first == descending) ? larger_key(pair[k]) : smaller_key(pair[k]);
    }
}
template <int SIZE, int DIST>
__device__ __forceinline__ void bitonic_merge(uint32_t (&v)[4], int lane) {
    bitonic_step<SIZE, DIST>(v, lane);
    if constexpr (DIST > 1) bitonic_merge<SIZE, DIST / 2>(v, lane);
}
template <int SIZE>
__device__ __forceinline__ void bitonic_sort(uint32_t (&v)[4], int lane) {
    if constexpr (SIZE > 2) bitonic_sort<SIZE / 2>(v, lane);
    bitonic_merge<SIZE, SIZE / 2>(v, lane);
}
__device__ __forceinline__ void sort_keys_descending(uint32_t (&v)[4], int lane) { bitonic_sort<256>(v, lane); }

__device__ __forceinline__ Edge load_edge(const Edge *p) {
    const uint4 v = *reinterpret_cast<const uint4 *>(p);
    return Edge{(int)v.x, __uint_as_float(v.y), __uint_as_float(v.z), v.w};
}
__device__ __forceinline__ void store_edge(Edge *p, int n, float w, float prior, uint32_t link) {
    *reinterpret_cast<uint4 *>(p) = make_uint4((uint32_t)n, __float_as_uint(w), __float_as_uint(prior), link);
}
__device__ __forceinline__ NodeInfo load_info(const NodeInfo *p) {
    const uint4 v = *reinterpret_cast<const uint4 *>(p);
    return NodeInfo{(int)v.x, (int)v.y, (int)v.z, __uint_as_float(v.w)};
}
__device__ __forceinline__ uint64_t lanes_below(int lane) { return (1ull << lane) - 1ull; }

// psyn_gamma_round: two of its three logarithms only say whether the candidate is accepted.  The hardware's, within 6e-6 of them
// together (none is above 17), say so unless the two sides are closer than 2^-15, and then the exact ones do.
__device__ __forceinline__ int gamma_round(float alpha, uint64_t key, int round, float *x) {
    constexpr float kLn2 = 0.693147181f;
    float u2;
    int small;
    psyn_gamma_candidate(alpha, key, round, x, &u2, &small);
    const float bound = small ? -*x : (alpha - 1.0f) * (__builtin_amdgcn_logf(*x) * kLn2);
    const float room = bound - __builtin_amdgcn_logf(u2) * kLn2;
    int accepted = room > 0.0f;
    if (!(fabsf(room) > 0x1p-15f)) accepted = psyn_gamma_accepts(alpha, *x, u2, small);
    return accepted;
}

// Priors of a new node: one Gamma weight per legal cell, prior = weight / sum, edge slots in descending weight order
// (ties: smaller cell first), so that progressive widening opens the most promising moves first.  Writes the whole
// record of every legal slot (no visits, no child, nothing in flight) and the slot's cell.  All 64 lanes must call it
// together.
__device__ void write_priors(const LoopArgs &g, int tree, int node, const uint32_t *board, int lane, uint64_t board_hash,
                             int n_legal) {
    constexpr int kPer = kEdges / kWave;
    uint32_t mine[kPer];
    // Rejection sampling diverges between lanes; every lane walks through its own cells and rounds independently, so
    // the wavefront runs for the largest per-lane total instead of the sum of per-cell maxima.
    int i = 0, round = 0;
#pragma unroll
    for (int k = 0; k < kPer; ++k) mine[k] = 0u;
    auto legal_cell = [&](int k) {
        const int c = lane + k * kWave;
        return c < g.cells && !stone_at(board, c) && !stone_at(board + 8, c);
    };
    while (i < kPer && !legal_cell(i)) ++i;
    uint64_t key = i < kPer ? psyn_cell_key(board_hash, lane + i * kWave) : 0;
    while (__ballot(i < kPer) != 0) {
        float x;
        const int ok = gamma_round(g.dirichlet_alpha, key, round, &x);
        if (i < kPer) {
            if (ok || round == PSYN_GAMMA_ROUNDS - 1) {
                const uint32_t weight = psyn_weight_key(x, lane + i * kWave);
#pragma unroll
                for (int k = 0; k < kPer; ++k)
                    if (k == i) mine[k] = weight;
                ++i;
                round = 0;
                while (i < kPer && !legal_cell(i)) ++i;
                if (i < kPer) key = psyn_cell_key(board_hash, lane + i * kWave);
            } else {
                ++round;
            }
        }
    }
    uint64_t sum = 0;
#pragma unroll
    for (int k = 0; k < kPer; ++k) sum += mine[k] ? psyn_key_weight(mine[k]) : 0;
    sum = wave_sum64(sum);
    // slot of a cell = rank of its key among the node's keys, largest first (0 = not a legal cell: last)
    sort_keys_descending(mine, lane);
    const size_t erow = ((size_t)tree * g.max_nodes + node) * kEdges + (size_t)kPer * lane;
    uint32_t cells_packed = 0;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        cells_packed |= (mine[k] ? 255u - (mine[k] & 0xFFu) : 0u) << (8 * k);
        if (mine[k] != 0u) store_edge(g.edges + erow + k, 0, 0.0f, psyn_prior(psyn_key_weight(mine[k]), sum, n_legal), 0u);
    }
    if (mine[0] != 0u) *reinterpret_cast<uint32_t *>(g.action + erow) = cells_packed;   // keys descend: slot 4 * lane is the lane's first
}

// Order-preserving integer image of a score that can win: the reference starts from (-FLT_MAX, no edge) and accepts
// a score that is greater than or equal to it, so NaN and -inf never win and get 0 (src/puct/puct_gpu_v3_cpp.cu:51-71);
// -0.0f counts as +0.0f because the reference compares floats.  The upper word of candidate_key().
__device__ __forceinline__ uint32_t score_image(float score) {
    if (!(score >= -FLT_MAX)) return 0u;
    const uint32_t b = __float_as_uint(score + 0.0f);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

template <class T>
__device__ __forceinline__ T poll_word(const T *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// ---- selection ---------------------------------------------------------------------------------------------------
// The edges of one node as the deciding traversals see them: up to NS per lane.
template <int NS>
struct EdgeSet {
    float q[NS], cp[NS];   // mean value, cpuct * prior
    int den[NS];           // visits + claims in flight + 1
    uint32_t link[NS], link_loaded[NS];
    int eid[NS];           // edge slot, -1 = none
};

template <int NS>
__device__ __forceinline__ float edge_score(const EdgeSet<NS> &e, int i, float sqrt_parent) {
    return prow_score(e.q[i], e.cp[i], sqrt_parent, e.den[i]);
}

// The traversals `members` decide one after another on the edges in `e` (which must include every edge that can come
// first for any of them); `total` = visits + claims over all expanded edges of the node, `tickets` = expansion tickets out.
template <int NS>
__device__ __forceinline__ void decide_in_turn(const LoopArgs &g, StepLds &s, int *paths, int *next, EdgeSet<NS> &e, int node,
                                               uint64_t members, int depth, int lane, int expanded, int legal, int &total,
                                               int &tickets, bool only_one = false) {
    // sqrt(parent) and the widening limit after 0, 1, 2 ... more claims, worked out side by side in lanes 0..15 (fewer
    // than 64 traversals decide here, and every claim adds one to the node's total)
    const bool widening = expanded != 1 || g.c_pw != 0.0f;
    const int claims_base = total;
    const int eff_lane = widening ? (total + lane > 1 ? total + lane : 1) : 1;
    const float sqrt_lane = widening ? sqrt_of_count(eff_lane) : 1.0f;
    const int allowed_lane = widening ? allowed_children(g.c_pw, g.alpha_pw, eff_lane, legal, sqrt_lane) : 1;
    for (uint64_t rest = members; rest != 0; rest &= rest - 1) {
        const int j = __builtin_ctzll(rest);   // the traversal deciding now
        const int claimed = total - claims_base;
        const float sqrt_parent = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(sqrt_lane), claimed));
        const int allowed = __builtin_amdgcn_readlane(allowed_lane, claimed);
        if (expanded + tickets < allowed) {   // expansion ticket
            if (lane == 0) {
                s.sel[j] = pack_sel(PUCT_SELECT_EXPAND, node, expanded + tickets);
                s.len[j] = depth + 1;
                s.claims[j] = depth;
                next[j] = -1;
            }
            tickets += 1;
            continue;
        }
        // The highest score first: its order-preserving integer image, reduced over the wavefront.  Only if more than
        // one edge attains it does the rotated edge index decide, through the full keys.  (A node's only edge is taken
        // whatever its score, as in the reference.)
        int best_lane = 0, best_slot = 0, hits = 1;
        if (expanded > 1 && !only_one) {
            float score[NS];
            uint32_t image[NS], lane_top = 0;
#pragma unroll
            for (int i = 0; i < NS; ++i) {
                score[i] = edge_score(e, i, sqrt_parent);
                image[i] = e.eid[i] >= 0 ? score_image(score[i]) : 0u;
                lane_top = image[i] > lane_top ? image[i] : lane_top;
            }
            const uint32_t top = wave_max_u32(lane_top);
            hits = 0;
#pragma unroll
            for (int i = 0; i < NS; ++i) {
                const uint64_t at = __ballot(image[i] == top);
                hits += __popcll(at);
                if (at != 0) best_lane = __builtin_ctzll(at), best_slot = i;
            }
            if (top == 0) {
                hits = 0;
            } else if (hits > 1) {
                int tie_offset = j;
                if (tie_offset >= expanded) tie_offset %= expanded;
                uint64_t key = 0;
                int key_slot = 0;
#pragma unroll
                for (int i = 0; i < NS; ++i) {
                    const uint64_t k = image[i] == top ? candidate_key(score[i], e.eid[i], tie_offset, expanded) : 0;
                    if (k > key) key = k, key_slot = i;
                }
                const uint64_t first = wave_max(key);
                best_lane = __builtin_ctzll(__ballot(key == first));
                best_slot = __builtin_amdgcn_readlane(key_slot, best_lane);
            }
        }
        int child = 0, best = 0;
        if (hits > 0) {
#pragma unroll
            for (int i = 0; i < NS; ++i)
                if (best_slot == i) {
                    child = (int)((uint32_t)__builtin_amdgcn_readlane((int)e.link[i], best_lane) >> 8);
                    best = __builtin_amdgcn_readlane(e.eid[i], best_lane);
                }
        }
        if (child <= 0 || child >= g.max_nodes) {   // no edge with a comparable score, or a link that leads nowhere
            if (lane == 0) {
                s.sel[j] = pack_sel(PUCT_SELECT_INVALID, PUCT_GOMOKU_SEL_NODE_MASK, 0);
                s.len[j] = 0;
                s.claims[j] = depth;
                next[j] = -1;
            }
            continue;
        }
#pragma unroll
        for (int i = 0; i < NS; ++i)
            if (best_slot == i && lane == best_lane) {
                e.den[i] += 1;
                e.link[i] += 1u;
            }
        total += 1;
        if (lane == 0) {
            paths[j * g.path_depth + depth] = (node << 8) | best;
            next[j] = child;
        }
    }
}

__device__ __forceinline__ uint32_t row_max_u32(uint32_t v) {   // over the 16 lanes of each row
    auto step = [](uint32_t x, auto ctrl) {
        const uint32_t o = (uint32_t)dpp<decltype(ctrl)::value>((int)x);
        return o > x ? o : x;
    };
    v = step(v, std::integral_constant<int, 0xB1>{});
    v = step(v, std::integral_constant<int, 0x4E>{});
    v = step(v, std::integral_constant<int, 0x141>{});
    return step(v, std::integral_constant<int, 0x140>{});
}

__device__ __forceinline__ float row_max_f32(float v) {   // over the 16 lanes of each row; no NaN
    float top;
    asm("s_nop 1\n\t"
        "v_max_f32_dpp %0, %1, %1 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf bound_ctrl:0\n\ts_nop 1\n\t"
        "v_max_f32_dpp %0, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf bound_ctrl:0\n\ts_nop 1\n\t"
        "v_max_f32_dpp %0, %0, %0 row_half_mirror row_mask:0xf bank_mask:0xf bound_ctrl:0\n\ts_nop 1\n\t"
        "v_max_f32_dpp %0, %0, %0 row_mirror row_mask:0xf bank_mask:0xf bound_ctrl:0"
        : "=&v"(top) : "v"(v));
    return top;
}

// decide_in_turn for at most 16 edges, one per lane from lane 0 on, all of which lead to a node and have a finite score; the n-th
// decision's edge goes to lane n of `mine`.  A decision is a chain on a lone wavefront, eight clocks for every instruction that
// waits for the one before it and more on the way through scalar registers and a branch: 330 clocks by decide_in_turn's way with one
// row (row_decisions).  So where nobody can get a ticket, all decisions are taken by vector instructions alone, without a branch on an
// outcome, by a score of one fused operation on the hardware's reciprocal (70 clocks with up to four edges, 110 with 16).  While the
// maximum is looked for, the reciprocal for an edge that is taken is worked out.  The scores are kept from being negative, so that
// they compare as integers.  An edge is taken if it comes within `apart` of the largest, which is more than both can be off by; if that
// held for more than one edge at any of the decisions, their number says so in the end, and the scores themselves decide them all.
template <int EDGES, int J = 0>
__device__ __forceinline__ void lane_that_took(int takes, int decision, int &lane) {
    lane = (dpp<0x150 + J>(takes) & decision) != 0 ? J : lane;   // row_newbcast:J
    if constexpr (J + 1 < EDGES) lane_that_took<EDGES, J + 1>(takes, decision, lane);
}
struct QuickRow {
    float cp, apart, q, cp_by;   // cp_by: cp over the edge's visits and claims and one
    int den, takes;              // takes: bit n, the n-th decision
};
template <int EDGES, int N = 0>
__device__ __forceinline__ void quick_row_decision(QuickRow &r, int n_members, float sqrt_lane) {
    const float root = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(sqrt_lane), N));
    const float score = prow_quick_score(r.q, r.cp_by, root), near = score + r.apart;
    const float cp_by_if_taken = r.cp * __builtin_amdgcn_rcpf((float)(r.den + 1));
    int top = __float_as_int(score);
    const auto larger = [](int a, int b) { return a > b ? a : b; };
    top = larger(dpp<0xB1>(top), top);
    top = larger(dpp<0x4E>(top), top);
    if constexpr (EDGES > 4) {
        top = larger(dpp<0x141>(top), top);
        top = larger(dpp<0x140>(top), top);
    }
    const bool taken = near >= __int_as_float(top);
    r.cp_by = taken ? cp_by_if_taken : r.cp_by;
    r.den += taken ? 1 : 0;
    r.takes |= taken ? 1 << N : 0;
    if constexpr (N + 1 < kTrav)
        if (N + 1 < n_members) quick_row_decision<EDGES, N + 1>(r, n_members, sqrt_lane);
}
template <int EDGES>
__device__ __forceinline__ bool quick_row_decisions(const EdgeSet<1> &e, int n_members, int lane, float sqrt_lane, int &den, int &mine) {
    const bool edge = e.eid[0] >= 0;
    const float q = prow_q(edge, e.q[0]);
    QuickRow r;
    r.cp = prow_cp(edge, e.cp[0]);
    r.cp_by = r.cp * __builtin_amdgcn_rcpf((float)den);
    r.den = den;
    r.takes = 0;
    const float last_root = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(sqrt_lane), n_members));
    r.apart = prow_quick_apart(row_max_f32(edge ? prow_quick_size(q, r.cp_by, last_root) : 0.0f));
    const float lift = row_max_f32(edge && q < 0.0f ? -q : 0.0f);
    r.q = lane >= EDGES ? __builtin_nanf("") : edge ? q + lift : q;   // (lanes behind the edges are never taken)
    quick_row_decision<EDGES>(r, n_members, sqrt_lane);
    if (wave_sum(__popc((uint32_t)r.takes)) != n_members) return false;
    den = r.den;
    lane_that_took<EDGES>(r.takes, 1 << (lane & (kRow - 1)), mine);
    return true;
}
template <bool TICKETS>
__device__ __forceinline__ void row_decisions(const EdgeSet<1> &e, uint64_t edges, uint32_t members, int n_members, int lane, int expanded, float sqrt_lane,
                                              int allowed_lane, int &tickets, uint32_t &with_ticket, int &den, int &mine) {
    const bool edge = e.eid[0] >= 0;
    const float q = prow_q(edge, e.q[0]), cp = prow_cp(edge, e.cp[0]);
    int claimed = 0;
    uint32_t bit = 1u;
    do {
        if (TICKETS && expanded + tickets < __builtin_amdgcn_readlane(allowed_lane, claimed)) {
            with_ticket |= bit;
            tickets += 1;
        } else {
            const float root = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(sqrt_lane), claimed));
            const float score = prow_row_score(q, cp, root, den, __builtin_amdgcn_rcpf((float)den));
            uint32_t first = (uint32_t)(__builtin_amdgcn_fcmpf(score, row_max_f32(score), 1 /* == */) & edges);
            if (__builtin_popcount(first) > 1) {   // the rotated edge index decides, as in candidate_key
                const uint32_t of_lane = 1u << (lane & (kTrav - 1));   // the deciding traversal: the member with this many before it
                int tie_offset = __builtin_ctzll(__ballot((members & of_lane) != 0 && 1u << __builtin_popcount(members & (of_lane - 1u)) == bit));
                if (tie_offset >= expanded) tie_offset %= expanded;
                const int turned = e.eid[0] - tie_offset + (e.eid[0] < tie_offset ? expanded : 0);
                const uint32_t key = __builtin_amdgcn_inverse_ballot_w64((uint64_t)first) ? 0x10000u - (uint32_t)turned : 0u;
                const uint32_t top_key = row_max_u32(key);
                first &= (uint32_t)__builtin_amdgcn_uicmp(key, top_key, 32);
            }
            den += __builtin_amdgcn_inverse_ballot_w64((uint64_t)first) ? 1 : 0;
            mine = __builtin_amdgcn_inverse_ballot_w64((uint64_t)bit) ? __builtin_ctz(first) : mine;
            claimed += 1;
        }
        bit <<= 1;
    } while (bit != 1u << n_members);
}
__device__ __forceinline__ void decide_in_row(const LoopArgs &g, StepLds &s, int *paths, int *next, Edge *row, const EdgeSet<1> &e, int node,
                                              uint32_t members, int depth, int lane, int expanded, int legal, int total, int &tickets) {
    const bool widening = expanded != 1 || g.c_pw != 0.0f;
    const int eff_lane = widening ? (total + lane > 1 ? total + lane : 1) : 1;
    const float sqrt_lane = widening ? sqrt_of_count(eff_lane) : 1.0f;
    const int allowed_lane = widening ? allowed_children(g.c_pw, g.alpha_pw, eff_lane, legal, sqrt_lane) : 1;
    const int tickets_before = tickets, n_members = __builtin_popcount(members);
    int den = prow_den(e.eid[0] >= 0, e.den[0]), mine = 0;   // mine, in lane n: lane of the edge that the n-th decision takes
    uint32_t with_ticket = 0;                                // bit n: the n-th decision is a ticket
    const uint64_t edges = __ballot(e.eid[0] >= 0);
    // (nobody can get a ticket if none of the limits that the decisions may see leaves one: with a negative alpha_pw the first is the largest)
    // From how many decisions on the quick way is tried matters little: from two, three, four or six on a step of 1 to 16 trees takes as long to
    // within 1 %; without it 1.5 to 2.5 % longer with 16 traversals (8.96 -> 9.17 us, 12.5 -> 12.8).
    if (__ballot(lane < n_members && expanded + tickets < allowed_lane) != 0)
        row_decisions<true>(e, edges, members, n_members, lane, expanded, sqrt_lane, allowed_lane, tickets, with_ticket, den, mine);
    else if (n_members < 4 || !((edges >> 4) == 0 ? quick_row_decisions<4>(e, n_members, lane, sqrt_lane, den, mine)
                                                  : quick_row_decisions<kRow>(e, n_members, lane, sqrt_lane, den, mine)))
        row_decisions<false>(e, edges, members, n_members, lane, expanded, sqrt_lane, allowed_lane, tickets, with_ticket, den, mine);
    const int nth = __builtin_popcount(members & ((1u << (lane & (kTrav - 1))) - 1u));   // which of the decisions is lane's traversal's
    const int from = __builtin_amdgcn_ds_bpermute(nth << 2, mine) << 2;
    const int child = (int)((uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)e.link[0]) >> 8);
    const int eid = __builtin_amdgcn_ds_bpermute(from, e.eid[0]);
    if (lane < kTrav && ((members >> lane) & 1u)) {
        if ((with_ticket >> nth) & 1u) {
            s.sel[lane] = pack_sel(PUCT_SELECT_EXPAND, node, expanded + tickets_before + __builtin_popcount(with_ticket & ((1u << nth) - 1u)));
            s.len[lane] = depth + 1;
            s.claims[lane] = depth;
            next[lane] = -1;
        } else {
            paths[lane * g.path_depth + depth] = (node << 8) | eid;
            next[lane] = child;
        }
    }
    if (e.eid[0] >= 0 && den != e.den[0]) row[e.eid[0]].link = e.link[0] + (uint32_t)(den - e.den[0]);
}

// The traversals of a tree descend in lockstep, one level per round.  The traversals that stand on the same node are
// served by one wavefront (that of the first of them), which loads the node's edges once and lets the traversals decide
// one after another, wid ascending, on registers: every decision is the reference's (progressive widening, expansion
// ticket, score, order on edges with the rotated tie-break: src/puct/puct_gpu_v3_cpp.cu:150-275) on the state that the
// claims of the traversals before it have left.  Taking the claims in turn is one of the interleavings the reference's
// atomics allow, needs no atomics itself, never loses a claim and makes a search reproducible.
__device__ void select_group(const LoopArgs &g, StepLds &s, int *paths, int *next, int tree, int node, uint64_t members,
                             int depth, int wave, int lane, uint32_t &nodes_read, uint32_t &edges_scored) {
    const size_t nrow = (size_t)tree * g.max_nodes + node;
    Edge *row = g.edges + nrow * kEdges;
    // all 256 edge slots are requested together with the node's own word, before anything about the node is known: one
    // round trip per level, whatever the node's width
    const NodeInfo ni = load_info(g.info + nrow);
    Edge loaded[kSlices];
#pragma unroll
    for (int i = 0; i < kSlices; ++i) loaded[i] = load_edge(row + lane + i * kWave);
    const int expanded = ni.expanded, n_members = __popcll(members);
    int tickets = ni.tickets;
    const int legal = ni.legal_turn & 0xFFFF;
    nodes_read += 1;
    if (expanded == PUCT_NODE_EXPANDED_TERMINAL || depth >= g.path_depth) {
        const int kind = expanded == PUCT_NODE_EXPANDED_TERMINAL ? PUCT_SELECT_TERMINAL : PUCT_SELECT_DEPTH_LIMIT;
        if (lane < kTrav && ((members >> lane) & 1ull)) {
            s.sel[lane] = pack_sel(kind, node, 0);
            s.len[lane] = depth + 1;
            s.claims[lane] = depth;
            next[lane] = -1;
        }
        return;
    }
    // The first of these traversals get the tickets that are left under a limit, the others find the node's children being
    // created.
    const auto give_tickets = [&](int allowed) {
        if (lane < kTrav && ((members >> lane) & 1ull)) {
            const int slot = expanded + tickets + __popcll(members & lanes_below(lane));
            const bool with_ticket = slot < allowed;
            s.sel[lane] = with_ticket ? pack_sel(PUCT_SELECT_EXPAND, node, slot) : pack_sel(PUCT_SELECT_BUSY, node, 0);
            s.len[lane] = with_ticket ? depth + 1 : 0;
            s.claims[lane] = depth;
            next[lane] = -1;
        }
        const int left = allowed - expanded - tickets > 0 ? allowed - expanded - tickets : 0;
        if (lane == 0 && left > 0) g.info[nrow].tickets = tickets + (n_members < left ? n_members : left);
    };
    if (expanded == 0) {   // no edge to claim, so the widening limit stays what it is at a count of 1
        give_tickets(allowed_children(g.c_pw, 0.5f, 1, legal, 1.0f));   // (1 to any power is 1)
        return;
    }
    edges_scored += (uint32_t)expanded;

    int total = 0;
#pragma unroll
    for (int i = 0; i < kSlices; ++i) total += lane + i * kWave < expanded ? loaded[i].n + (int)(loaded[i].link & 0xFFu) : 0;
    total = wave_sum(total);
    if (expanded != 1 || g.c_pw != 0.0f) {   // as many tickets as traversals: no edge is claimed, and the limit stays too
        const int allowed = allowed_children(g.c_pw, g.alpha_pw, total > 1 ? total : 1, legal);
        if (expanded + tickets + n_members <= allowed) {
            give_tickets(allowed);
            return;
        }
    }

    // Every one of these traversals takes the same edge: all of them at once, a traversal per lane.
    auto take_all = [&](uint32_t link, int eid) {
        const int child = (int)(link >> 8);
        const bool leads_somewhere = child > 0 && child < g.max_nodes;
        if (lane < kTrav && ((members >> lane) & 1ull)) {
            if (leads_somewhere) {
                paths[lane * g.path_depth + depth] = (node << 8) | eid;
                next[lane] = child;
            } else {
                s.sel[lane] = pack_sel(PUCT_SELECT_INVALID, PUCT_GOMOKU_SEL_NODE_MASK, 0);
                s.len[lane] = 0;
                s.claims[lane] = depth;
                next[lane] = -1;
            }
        }
        if (leads_somewhere && lane == 0) row[eid].link = link + (uint32_t)n_members;
    };
    // No expansion ticket is to be had here however many of these traversals have claimed: none of the widening limits that they may
    // see, one a lane, exceeds the children there are.
    const auto no_ticket_for_anyone = [&] {
        if (expanded >= legal || (expanded == 1 && g.c_pw == 0.0f)) return true;   // (the limit does not exceed the legal moves)
        const int eff_lane = total + lane > 1 ? total + lane : 1;
        return __ballot(lane < n_members && allowed_children(g.c_pw, g.alpha_pw, eff_lane, legal) > expanded) == 0;
    };

    // decide_in_row's terms: every edge leads to a node and has a finite score
    const auto fit_for_row = [&](const EdgeSet<1> &e) {
        const int child = (int)(e.link[0] >> 8);
        return __ballot(e.eid[0] >= 0 && !(child > 0 && child < g.max_nodes && fabsf(e.q[0]) < 1e30f && prow_cp_fits(e.cp[0]) && e.den[0] > 0)) == 0;
    };
    const auto slot_of_edge = [&](EdgeSet<1> &e, int n, float w, float cp, uint32_t link, int eid) {
        e = EdgeSet<1>{{eid >= 0 && n > 0 ? w / (float)n : 0.0f}, {cp}, {n + (int)(link & 0xFFu) + 1}, {link}, {link}, {eid}};
    };
    // Most edges of a wide node cannot come first for any of these traversals.  While they decide, sqrt(parent) only
    // grows (by their own claims) and an edge's claims only grow, and every operation of the score is monotonic, so an
    // edge's score stays below its score at the largest sqrt(parent) and its present claims, and the best edge's score
    // stays above the largest score at the present sqrt(parent) with all of these traversals' claims on it.  Edges whose
    // upper bound is below that lower bound are out, and a decision costs one division instead of one per 64 edges.  The
    // bounds are worked out with the hardware's reciprocals and roots, each right to an ulp: both are moved apart by 2^-18
    // of |q| + u, more than four times what the roundings of the bound and of the score come to (the last steps of
    // subnormal scores: 1e-30).  With the score's own divisions this pass took 2700 clocks a node, more than half of what
    // sixteen decisions do.
    // Returns how many remain if they are in `few` now, 0 if they are not, -1 if all is decided.
    EdgeSet<1> few{{0.0f}, {0.0f}, {1}, {0u}, {0u}, {-1}};
    const auto keep_the_best = [&](auto slices) -> int {
        constexpr int NS = decltype(slices)::value;
        constexpr float kApart = 0x1p-18f;
        const int now = total > 1 ? total : 1, then = total + n_members > 1 ? total + n_members : 1;
        const float sqrt_low = __builtin_amdgcn_sqrtf((float)now) * (1.0f - kApart), sqrt_high = __builtin_amdgcn_sqrtf((float)then) * (1.0f + kApart);
        float low = -FLT_MAX, high[NS];
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            const Edge &e = loaded[i];
            const bool valid = lane + i * kWave < expanded;
            const float q = e.n > 0 ? e.w * __builtin_amdgcn_rcpf((float)e.n) : 0.0f, cp = g.cpuct * e.prior;
            const int den = e.n + (int)(e.link & 0xFFu) + 1;
            const float l = __builtin_fmaf(cp * sqrt_low, __builtin_amdgcn_rcpf((float)(den + n_members)), __builtin_fmaf(-kApart, fabsf(q), q));
            const float h = __builtin_fmaf(cp * sqrt_high, __builtin_amdgcn_rcpf((float)den), __builtin_fmaf(kApart, fabsf(q), q));
            low = valid && l > low ? l : low;   // (a NaN gives no bound)
            high[i] = h;
        }
        const uint32_t low_bits = __float_as_uint(low);   // the largest of the lanes', by its order-preserving image
        const uint32_t top = wave_max_u32(low_bits ^ ((uint32_t)((int32_t)low_bits >> 31) | 0x80000000u));
        low = __uint_as_float((top & 0x80000000u) ? top ^ 0x80000000u : ~top);
        if (!(low > -FLT_MAX)) return 0;
        low -= 1e-30f;
        int kept = 0, place[NS];
        uint64_t in_slice[NS];
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            const uint64_t mask = __ballot(lane + i * kWave < expanded && !(high[i] < low));
            in_slice[i] = mask;
            place[i] = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, (uint32_t)kept));
            kept += __popcll(mask);
        }
        // One edge left and no expansion ticket to be had: every one of these traversals takes that edge.
        if (kept == 1 && no_ticket_for_anyone()) {
#pragma unroll
            for (int i = 0; i < NS; ++i)
                if (in_slice[i] != 0) {
                    const int at = __builtin_ctzll(in_slice[i]);
                    take_all((uint32_t)__builtin_amdgcn_readlane((int)loaded[i].link, at), at + i * kWave);
                }
            return -1;
        }
        int *stage = s.stage[wave];
        if (kept <= kRow) {   // through LDS into the first row, in one go
#pragma unroll
            for (int i = 0; i < NS; ++i)
                if (__builtin_amdgcn_inverse_ballot_w64(in_slice[i])) {
                    *reinterpret_cast<int4 *>(stage + 4 * place[i]) = make_int4(loaded[i].n, __float_as_int(loaded[i].w), __float_as_int(loaded[i].prior), (int)loaded[i].link);
                    stage[4 * kRow + place[i]] = lane + i * kWave;
                }
            wave_lds_fence();
            int4 v = make_int4(0, 0, 0, 0);
            int eid = -1;
            if (lane < kept) v = *reinterpret_cast<const int4 *>(stage + 4 * lane), eid = stage[4 * kRow + lane];
            slot_of_edge(few, v.x, __int_as_float(v.y), g.cpuct * __int_as_float(v.z), (uint32_t)v.w, eid);
            wave_lds_fence();
        } else {
            if (NS == 1 || kept > kWave) return 0;
            int field[5];
#pragma unroll
            for (int f = 0; f < 5; ++f) {
#pragma unroll
                for (int i = 0; i < NS; ++i)
                    if (__builtin_amdgcn_inverse_ballot_w64(in_slice[i]))
                        stage[place[i]] = f == 0 ? loaded[i].n : f == 1 ? __float_as_int(loaded[i].w) : f == 2 ? __float_as_int(loaded[i].prior)
                                        : f == 3 ? (int)loaded[i].link : lane + i * kWave;
                wave_lds_fence();
                field[f] = lane < kept ? stage[lane] : f == 4 ? -1 : 0;
                wave_lds_fence();
            }
            slot_of_edge(few, field[0], __int_as_float(field[1]), g.cpuct * __int_as_float(field[2]), (uint32_t)field[3], field[4]);
        }
        return kept;
    };

    int edges = 0;   // how many there are in `few`, one per lane
    if (expanded > kWave) {
        edges = keep_the_best(std::integral_constant<int, kSlices>{});
    } else if (n_members >= 3) {
        if (expanded > 1) {
            edges = keep_the_best(std::integral_constant<int, 1>{});
        } else if (no_ticket_for_anyone()) {   // a node's only edge is taken whatever its score
            take_all((uint32_t)__builtin_amdgcn_readlane((int)loaded[0].link, 0), 0);
            edges = -1;
        }
    }
    const bool only_one = edges == 1;
    if (edges == 0 && expanded <= kWave) {
        slot_of_edge(few, loaded[0].n, loaded[0].w, g.cpuct * loaded[0].prior, loaded[0].link, lane < expanded ? lane : -1);
        edges = expanded;
    }
    if (edges >= 1 && edges <= kRow && fit_for_row(few)) {
        decide_in_row(g, s, paths, next, row, few, node, (uint32_t)members, depth, lane, expanded, legal, total, tickets);
    } else if (edges > 0) {
        decide_in_turn<1>(g, s, paths, next, few, node, members, depth, lane, expanded, legal, total, tickets, only_one);
        if (few.eid[0] >= 0 && few.link[0] != few.link_loaded[0]) row[few.eid[0]].link = few.link[0];
    } else if (edges == 0) {
        EdgeSet<kSlices> all;
#pragma unroll
        for (int i = 0; i < kSlices; ++i) {
            const Edge &e = loaded[i];
            const bool valid = lane + i * kWave < expanded;
            all.q[i] = valid && e.n > 0 ? e.w / (float)e.n : 0.0f;
            all.cp[i] = g.cpuct * e.prior;
            all.link[i] = all.link_loaded[i] = e.link;
            all.den[i] = e.n + (int)(e.link & 0xFFu) + 1;
            all.eid[i] = valid ? lane + i * kWave : -1;
        }
        decide_in_turn<kSlices>(g, s, paths, next, all, node, members, depth, lane, expanded, legal, total, tickets);
#pragma unroll
        for (int i = 0; i < kSlices; ++i)
            if (all.link[i] != all.link_loaded[i]) row[lane + i * kWave].link = all.link[i];
    }
    if (lane == 0 && tickets != ni.tickets) g.info[nrow].tickets = tickets;
}

// Selection of one step for the traversals of one tree; all wavefronts of the workgroup call it.  Ends behind a
// workgroup barrier with every traversal's result in `s` and its path in `paths`.
// FARM: thread 0 asks for *done, the entries that the evaluators have worked off, with every level and keeps the last answer, so that
// it seldom has to ask, and wait a round trip for it, afterwards.
template <bool FARM>
__device__ void select_phase(const LoopArgs &g, StepLds &s, int *paths, int tree, int wave, int lane, int n_waves,
                             uint32_t &nodes_read, uint32_t &edges_scored, const int *done, int &worked_off) {
    if (threadIdx.x < kTrav) {
        const int t = threadIdx.x;
        s.cur[0][t] = t < n_waves ? 0 : -1;
        s.cur[1][t] = -1;
        s.sel[t] = pack_sel(PUCT_SELECT_INVALID, PUCT_GOMOKU_SEL_NODE_MASK, 0);
        s.len[t] = 0;
        s.claims[t] = 0;
        s.value[t] = 0.0f;
    }
    __syncthreads();
    for (int depth = 0;; ++depth) {
        const int *cur = s.cur[depth & 1];
        int *next = s.cur[(depth & 1) ^ 1];
        const int at = lane < kTrav ? cur[lane] : -1;
        if (__ballot(at >= 0) == 0) break;   // every wavefront reads the same words: all leave together
        if (FARM && threadIdx.x == 0) worked_off = poll_word(done);
        const int mine = __builtin_amdgcn_readlane(at, wave);
        const uint64_t members = __ballot(at >= 0 && at == mine);
        if (mine < 0) {
            if (lane == 0) next[wave] = -1;
        } else if ((members & lanes_below(wave)) == 0) {
            select_group(g, s, paths, next, tree, mine, members, depth, wave, lane, nodes_read, edges_scored);
        }
        __syncthreads();
    }
}

// ---- expansion / evaluation -----------------------------------------------------------------------------------------
// Every wavefront handles the leaf of its own traversal.  Children get consecutive node ids in traversal order and go
// into the node's next free edge slots in traversal order (the expanded edges of a node stay contiguous whatever the
// tickets say); when the tree cannot take all expansions of a step none is committed (those traversals evaluate the
// node they reached instead).
struct Leaf {   // what the selection has brought the wavefront's traversal to, on its way from memory
    NodeInfo info;
    uint32_t board;   // lanes 0..15
};
__device__ __forceinline__ bool reached_a_node(int sel) {
    const int kind = (sel >> PUCT_GOMOKU_SEL_KIND_SHIFT) & 7;
    return kind == PUCT_SELECT_EXPAND || kind == PUCT_SELECT_TERMINAL || kind == PUCT_SELECT_DEPTH_LIMIT;
}
__device__ __forceinline__ Leaf request_leaf(const LoopArgs &g, const StepLds &s, int tree, int wave, int lane) {
    Leaf leaf{{0, 0, 0, 0.0f}, 0u};
    const int sel = __builtin_amdgcn_readfirstlane(s.sel[wave]);
    if (reached_a_node(sel)) {
        const size_t row = (size_t)tree * g.max_nodes + (sel & PUCT_GOMOKU_SEL_NODE_MASK);
        leaf.info = load_info(g.info + row);
        if (lane < kBoardWords) leaf.board = g.board[row * kBoardWords + lane];
    }
    return leaf;
}
template <bool FARM>
__device__ void expand_phase(const LoopArgs &g, StepLds &s, const Leaf &leaf, uint64_t hash_seed, int tree, int wave, int lane, int n_waves, uint32_t &created) {
    const int raw = s.sel[wave];
    const int kind = (raw >> PUCT_GOMOKU_SEL_KIND_SHIFT) & 7;
    const int node = raw & PUCT_GOMOKU_SEL_NODE_MASK, ticket_slot = (raw >> PUCT_GOMOKU_SEL_SLOT_SHIFT) & 0xFF;
    const size_t trow = (size_t)tree * g.max_nodes;
    const bool has_node = reached_a_node(raw);
    uint32_t *board = s.board[wave];
    const NodeInfo ni = leaf.info;
    if (has_node) {
        if (lane < kBoardWords) board[lane] = leaf.board;
        wave_lds_fence();
    }
    const int n_legal = ni.legal_turn & 0xFFFF, turn = (ni.legal_turn & kTurnBit) ? -1 : 1;
    const bool wants = kind == PUCT_SELECT_EXPAND && ticket_slot < n_legal;
    if (lane == 0) s.want[wave] = wants ? node : -1;
    __syncthreads();
    const int other = lane < n_waves ? s.want[lane] : -1;
    const uint64_t all = __ballot(other >= 0), here = __ballot(other >= 0 && other == node);
    const int total = __popcll(all), before = __popcll(all & lanes_below(wave));
    const int rank = __popcll(here & lanes_below(wave)), siblings = __popcll(here);
    const int base = s.node_count;   // (wave 0 counts on behind the next barrier)
    const bool fits = base + total <= g.max_nodes;

    int reached = kReachedNothing, child = 0, child_turn = 0, edge = 0;
    if (wants && fits) {
        const int slot = ni.expanded + rank;
        child = base + before;
        edge = (node << 8) | slot;
        const int action = g.action[(trow + node) * kEdges + slot];
        uint32_t *mine = board + (turn > 0 ? 0 : 8);
        if (lane == 0) mine[action >> 5] |= 1u << (action & 31);
        wave_lds_fence();
        child_turn = (n_legal - 1) | (turn > 0 ? kTurnBit : 0);
        reached = makes_five(mine, action, g.m, g.n, lane) ? kReachedWin : n_legal == 1 ? kReachedDraw : kReachedChild;
        if (lane < kBoardWords) g.board[(trow + child) * kBoardWords + lane] = board[lane];
        if (lane == 0 && rank == 0) g.info[trow + node].expanded = ni.expanded + siblings;
    } else if (kind == PUCT_SELECT_TERMINAL) {
        reached = kReachedValued;
    } else if (has_node) {
        reached = kReachedPosition;
    }
    if (lane == 0) {
        s.reached[wave] = make_int4(reached, child, edge, child_turn);
        s.value[wave] = ni.value;
    }
    __syncthreads();
    // A position's hash is a chain of twenty 64-bit products, at a quarter of the rate whatever the number of lanes: one
    // wavefront works out all of them, a traversal per lane, instead of each its own (four wavefronts on a SIMD: 2 us).
    if (wave == 0) {
        if (lane == 0) {
            if (fits) s.node_count = base + total;
            s.requests = fits ? total : 0;
        }
        if (fits) created += (uint32_t)total;
        if (lane < n_waves) {
            const int4 r = s.reached[lane];
            float u = 0.0f;   // value of the reached node for the player who moved into it
            if (r.x == kReachedValued) u = s.value[lane];
            if (r.x >= kReachedPosition) {
                const uint64_t bh = psyn_board_hash_from(hash_seed, s.board[lane]);
                s.hash[lane] = bh;
                const bool terminal = r.x == kReachedWin || r.x == kReachedDraw;
                const float v = r.x == kReachedWin ? -1.0f : (terminal ? 0.0f : psyn_value(bh));
                u = v;
                if (r.x != kReachedPosition) {
                    *reinterpret_cast<uint4 *>(g.info + trow + r.y) =
                        make_uint4((uint32_t)(terminal ? PUCT_NODE_EXPANDED_TERMINAL : 0), 0u, (uint32_t)r.w, __float_as_uint(v));
                    Edge *e = g.edges + (trow + (r.z >> 8)) * kEdges + (r.z & 0xFF);
                    e->n = 1;
                    e->w = -v;
                    e->link = (uint32_t)r.y << 8;
                    u = -v;
                    if (FARM) {   // the child's priors are an evaluator workgroup's work
                        g.requests[tree].child[r.y - base] = terminal ? -1 : r.y;
                        g.requests[tree].hash[r.y - base] = bh;
                    }
                }
            }
            s.value[lane] = u;
        }
    }
    if (!FARM) {
        __syncthreads();
        if (reached == kReachedChild) write_priors(g, tree, child, board, lane, s.hash[wave], n_legal - 1);
    }
}

// ---- backup ----------------------------------------------------------------------------------------------------------
// Every traversal gives back the claims along its path; one that reached a node (expansion, terminal, depth limit) also
// leaves a visit and the node's value, sign alternating, on every edge of the path (src/puct/puct_gpu_v2.py:847-927
// moved to edge-level virtual loss), and an expansion returns its ticket.  Lane = (traversal, one of four depths): the
// traversals whose paths share an edge at that depth meet inside a row of 16 lanes, and the last of them stores the
// edge after adding the values in traversal order, so the float sums do not depend on timing.  A step's paths are a few
// levels, so this is one pass of one wavefront, as long as its chain of instructions: what the others of a row hold comes by
// DPP broadcasts (by 48 LDS permutes it took 1.2 us longer), and the tickets go back by the last wavefront meanwhile.
template <int J>
__device__ __forceinline__ void meet_in_row(int enc, uint32_t &same) {   // bit j: traversal j of the row stands on this lane's edge
    same |= dpp<0x150 + J>(enc) == enc ? 1u << J : 0u;                     // row_newbcast:J
    if constexpr (J + 1 < kTrav) meet_in_row<J + 1>(enc, same);
}
template <int J>
__device__ __forceinline__ void add_in_order(float val, uint32_t which, float &acc) {
    const float with = acc + __int_as_float(dpp<0x150 + J>(__float_as_int(val)));
    acc = (which >> J) & 1u ? with : acc;
    if constexpr (J + 1 < kTrav) add_in_order<J + 1>(val, which, acc);
}
__device__ void backup_phase(const LoopArgs &g, StepLds &s, const int *paths, int tree, int wave, int lane, int n_waves) {
    const size_t trow = (size_t)tree * g.max_nodes;
    const int t = lane & (kTrav - 1), sub = lane >> 4;
    const int raw = s.sel[t], my_claims = s.claims[t];
    const int kind = (raw >> PUCT_GOMOKU_SEL_KIND_SHIFT) & 7;
    const uint32_t counted = (uint32_t)__ballot(kind == PUCT_SELECT_EXPAND || kind == PUCT_SELECT_TERMINAL || kind == PUCT_SELECT_DEPTH_LIMIT) & 0xFFFFu;
    const float u = s.value[t];
    const int deepest = __builtin_amdgcn_readfirstlane((int)row_max_u32((uint32_t)my_claims));
    for (int d0 = 4 * wave; d0 < deepest; d0 += 4 * n_waves) {
        const int d = d0 + sub;
        const int enc = d < my_claims ? paths[t * g.path_depth + d] : -1;
        const float val = ((my_claims - d) & 1) ? -u : u;   // a counted traversal's path has as many edges as claims
        Edge *e = nullptr;
        Edge old{0, 0.0f, 0.0f, 0u};
        if (enc >= 0) {
            e = g.edges + (trow + (enc >> 8)) * kEdges + (enc & 0xFF);
            old = load_edge(e);
        }
        uint32_t same = 0;
        meet_in_row<0>(enc, same);
        const uint32_t upto = same & ((2u << t) - 1u);   // this traversal and those before it
        float acc = old.w;
        add_in_order<0>(val, upto & counted, acc);
        if (enc >= 0 && upto == same) {   // the last of them
            e->n = old.n + __builtin_popcount(upto & counted);
            e->w = acc;
            e->link = old.link - (uint32_t)__builtin_popcount(upto);
        }
    }
    if (wave == n_waves - 1) {   // expansion tickets back, once per node
        const int sel_l = lane < n_waves ? s.sel[lane] : 0;
        const bool is_exp = lane < n_waves && ((sel_l >> PUCT_GOMOKU_SEL_KIND_SHIFT) & 7) == PUCT_SELECT_EXPAND;
        const int node_l = is_exp ? sel_l & PUCT_GOMOKU_SEL_NODE_MASK : -1;   // (the first row; the others hold none)
        uint32_t same = 0;
        meet_in_row<0>(node_l, same);
        if (is_exp && (same & ((1u << lane) - 1u)) == 0) g.info[trow + node_l].tickets -= __builtin_popcount(same);
    }
}

// Root of every tree: node 0 with the root position and its priors.
__global__ __launch_bounds__(kWave) void init_kernel(const LoopArgs g, const uint32_t *root_board, int root_turn) {
    __shared__ uint32_t board[kBoardWords];
    const int tree = blockIdx.x, lane = threadIdx.x;
    const size_t trow = (size_t)tree * g.max_nodes;
    const uint32_t w = lane < kBoardWords ? root_board[lane] : 0u;
    if (lane < kBoardWords) {
        board[lane] = w;
        g.board[trow * kBoardWords + lane] = w;
    }
    const int n_legal = g.cells - wave_sum(__popc(w));
    wave_lds_fence();
    if (lane < kTally) g.tally[(size_t)tree * kTally + lane] = 0ull;
    if (lane < g.traversals) {
        const size_t out = (size_t)tree * g.traversals + lane;
        g.out_selected[out] = pack_sel(PUCT_SELECT_INVALID, PUCT_GOMOKU_SEL_NODE_MASK, 0);
        g.out_len[out] = 0;
        g.out_claims[out] = 0;
        g.out_value[out] = 0.0f;
    }
    if (lane == 0) {
        *reinterpret_cast<uint4 *>(g.info + trow) =
            make_uint4((uint32_t)(n_legal == 0 ? PUCT_NODE_EXPANDED_TERMINAL : 0), 0u,
                       (uint32_t)(n_legal | (root_turn > 0 ? 0 : kTurnBit)), 0u);
        g.node_count[tree] = 1;
        EvalRequests &rq = g.requests[tree];
        rq.tag = 0;
        rq.done = 0;
        rq.abort = 0;
        for (int &x : rq.xcc) x = -1;
    }
    if (n_legal > 0) write_priors(g, tree, 0, board, lane, psyn_board_hash(psyn_tree_seed(g.seed, tree), board), n_legal);
}

// Makes the stores of a phase visible to the loads of the next one.  All wavefronts of a tree run on one CU and share its
// L1, which takes their loads and stores in order, so among themselves a workgroup barrier is all they need; nothing is
// invalidated.  (An agent-scope acquire in every wavefront here made the CU's next load wait for sixteen invalidations:
// 1.1 us instead of 0.15, twice a step.)  What other workgroups are told of next must also have been acknowledged by the L2
// that they read, which a workgroup-scope release does not wait for.
__device__ __forceinline__ void phase_barrier(bool for_evaluators) {
    if (for_evaluators) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
}

// What the traversals of a step ended with, between the launches of the stepwise mode and for the host to read.
__device__ void state_to_memory(const LoopArgs &g, const StepLds &s, const int *paths, int tree, int n_waves) {
    const size_t out = (size_t)tree * g.traversals;
    for (int i = threadIdx.x; i < n_waves * g.path_depth; i += n_waves * kWave) {   // the workgroup's live threads
        const int t = i / g.path_depth, d = i - t * g.path_depth;
        g.out_path[out * g.path_depth + i] = d < s.claims[t] ? paths[i] : -1;
    }
    if (threadIdx.x < n_waves) {
        const int t = threadIdx.x;
        g.out_selected[out + t] = s.sel[t];
        g.out_len[out + t] = s.len[t];
        g.out_claims[out + t] = s.claims[t];
        g.out_value[out + t] = s.value[t];
    }
    if (threadIdx.x == 0) g.node_count[tree] = s.node_count;
}
__device__ void state_from_memory(const LoopArgs &g, StepLds &s, int *paths, int tree, int n_waves) {
    const size_t out = (size_t)tree * g.traversals;
    for (int i = threadIdx.x; i < n_waves * g.path_depth; i += n_waves * kWave) paths[i] = g.out_path[out * g.path_depth + i];
    if (threadIdx.x < kTrav) {
        const int t = threadIdx.x;
        const bool live = t < n_waves;
        s.sel[t] = live ? g.out_selected[out + t] : pack_sel(PUCT_SELECT_INVALID, PUCT_GOMOKU_SEL_NODE_MASK, 0);
        s.len[t] = live ? g.out_len[out + t] : 0;
        s.claims[t] = live ? g.out_claims[out + t] : 0;
        s.value[t] = live ? g.out_value[out + t] : 0.0f;
    }
    if (threadIdx.x == 0) s.node_count = g.node_count[tree];
    __syncthreads();
}

struct Work {
    uint32_t kinds[5] = {0, 0, 0, 0, 0}, created = 0, nodes_read = 0, edges_scored = 0;
    uint64_t ticks[3] = {0, 0, 0};   // selection, expansion, backup, on wavefront 0
    __device__ void count_kind(const StepLds &s, int wave) {
        const int kind = (s.sel[wave] >> PUCT_GOMOKU_SEL_KIND_SHIFT) & 7;
#pragma unroll
        for (int k = 0; k < 5; ++k) kinds[k] += kind == k ? 1u : 0u;
    }
    __device__ void to_memory(const LoopArgs &g, int tree, int lane) const {
        if (lane != 0) return;
        unsigned long long *row = g.tally + (size_t)tree * kTally;
#pragma unroll
        for (int k = 0; k < 5; ++k)
            if (kinds[k]) atomicAdd(row + k, (unsigned long long)kinds[k]);
        if (created) atomicAdd(row + 5, (unsigned long long)created);
        if (nodes_read) atomicAdd(row + 6, (unsigned long long)nodes_read);
        if (edges_scored) atomicAdd(row + 7, (unsigned long long)edges_scored);
#pragma unroll
        for (int k = 0; k < 3; ++k)
            if (ticks[k]) atomicAdd(row + 8 + k, (unsigned long long)ticks[k]);
    }
};

extern __shared__ int dynamic_lds[];

// ---- evaluator workgroups --------------------------------------------------------------------------------------------
// The priors of a new node are a pure function of its position, and nothing reads them before the next step's
// selection, so they need not be worked out on the compute unit that owns the tree: the tree's workgroup posts the
// step's new nodes, goes on with its backup, and picks the results up before the next step.  An evaluator workgroup
// takes up to four nodes at a time, four wavefronts and one cell per lane each.  A wavefront sorts its 64 keys in registers,
// the node's four lists are merged through LDS, and every wavefront stores 64 consecutive slots.  Same priors, bit for bit, as
// write_priors().  Bound by vector instructions, about 400 a wavefront and node, and by the multiplications of the streams among
// them.  (1200 when every lane compared its key with all 256 and the sampler ran round after round; with a binary search in the
// three other lists for each key's slot, bank conflicts and scattered stores made a step 10.40 us, now 10.04, at 16 trees x 16
// traversals and four evaluators.)
constexpr int kEvalParts = kEdges / kWave;              // wavefronts per node
constexpr int kEvalNodes = kTrav / kEvalParts;          // nodes at a time, at most
struct EvalLds {
    uint32_t keys[2][kEvalNodes][kEvalParts][kWave];   // sorted by 64, by 128
    double weight[kEvalNodes][kEvalParts];
    int legal[kEvalNodes][kEvalParts];
    unsigned long long tag[2];   // by parity of the step
};
__device__ __forceinline__ int eval_nodes_at_once() { return (int)blockDim.x / (kWave * kEvalParts); }   // (2 to 4: 8 to 16 wavefronts)

// psyn_key_weight as a double, which it is exactly, and so are the sums (below 2^48): psyn_prior's quotient without the conversions.
__device__ __forceinline__ double key_weight(uint32_t key) { return trunc((double)__uint_as_float(key & 0x7FFFFF00u) * 4294967296.0); }
__device__ __forceinline__ double wave_sum_f64(double v) {
    const auto step = [](double x, auto ctrl) {
        const uint64_t b = (uint64_t)__double_as_longlong(x);
        const uint32_t lo = (uint32_t)dpp<decltype(ctrl)::value>((int)(uint32_t)b), hi = (uint32_t)dpp<decltype(ctrl)::value>((int)(uint32_t)(b >> 32));
        return x + __longlong_as_double((long long)((uint64_t)hi << 32 | lo));
    };
    v = step(v, std::integral_constant<int, 0xB1>{});
    v = step(v, std::integral_constant<int, 0x4E>{});
    v = step(v, std::integral_constant<int, 0x141>{});
    v = step(v, std::integral_constant<int, 0x140>{});
    const auto row = [&](int lane) { return __longlong_as_double((long long)read_lane64((uint64_t)__double_as_longlong(v), lane)); };
    return (row(0) + row(16)) + (row(32) + row(48));
}

// The wavefront's 64 keys, largest first: a bitonic sort with one key per lane.  SIZE == 64, DIST == 32 alone: a bitonic list.
template <int SIZE, int DIST>
__device__ __forceinline__ void sort64_step(uint32_t &v) {
    constexpr auto takes_larger = [] {
        uint64_t m = 0;
        for (int i = 0; i < kWave; ++i) m |= (uint64_t)(((i & DIST) == 0) == ((i & SIZE) == 0)) << i;
        return m;
    }();
    const KeyPair p = with_partner<DIST>(v);
    v = __builtin_amdgcn_inverse_ballot_w64(takes_larger) ? larger_key(p) : smaller_key(p);
    if constexpr (DIST > 1) sort64_step<SIZE, DIST / 2>(v);
}
template <int SIZE = 2>
__device__ __forceinline__ void sort64_descending(uint32_t &v) {
    sort64_step<SIZE, SIZE / 2>(v);
    if constexpr (SIZE < kWave) sort64_descending<2 * SIZE>(v);
}

// Entry `index` of the step (none if it is not below n), whose node is first_node + index, by four wavefronts, `part` = 0..3; the whole workgroup must call it.
__device__ void evaluate_node(const LoopArgs &g, EvalLds &L, int tree, int index, int n, int first_node, int group, int part, int lane) {
    const EvalRequests &rq = g.requests[tree];
    const size_t trow = (size_t)tree * g.max_nodes;
    int child = -1;
    uint32_t w = 0u;
    uint64_t hash = 0;
    if (index < n) {   // all that there is to know about the entry in one round trip
        child = rq.child[index];
        hash = rq.hash[index];
        if (lane < kBoardWords) w = g.board[(trow + first_node + index) * kBoardWords + lane];
    }
    const bool active = child > 0;
    uint32_t key = 0;
    if (active) {
        const int cell = part * kWave + lane;
        // words of the lane's cell: the same for each half of the wavefront
        uint32_t plus = (uint32_t)__builtin_amdgcn_readlane((int)w, 2 * part), minus = (uint32_t)__builtin_amdgcn_readlane((int)w, 8 + 2 * part);
        const uint32_t plus_hi = (uint32_t)__builtin_amdgcn_readlane((int)w, 2 * part + 1);
        const uint32_t minus_hi = (uint32_t)__builtin_amdgcn_readlane((int)w, 8 + 2 * part + 1);
        if (lane >= 32) plus = plus_hi, minus = minus_hi;
        const bool legal = cell < g.cells && !(((plus | minus) >> (lane & 31)) & 1u);
        const uint64_t stream = psyn_cell_key(hash, cell);
        // One round of the sampler for every cell, then, as the rounds of a cell are independent numbers of its stream, several
        // at once for the cells that are left: 1, 2 or 4 lanes a cell, the first round that accepts counts.  (Round after
        // round the wavefront ran five for its unluckiest lane, 500 of its 700 instructions: 12.8 us a step instead of 11.85 at
        // 16 trees x 16 traversals, four evaluators.)
        float x;
        bool pending = legal && !gamma_round(g.dirichlet_alpha, stream, 0, &x);
        if (legal && !pending) key = psyn_weight_key(x, cell);
        uint64_t left = __ballot(pending);
        for (int round = 1; left != 0;) {
            const int n_left = __popcll(left), shift = n_left <= kWave / 4 ? 2 : n_left <= kWave / 2 ? 1 : 0;
            const int rank = __popcll(left & lanes_below(lane));
            // lane r learns the r-th of these cells' lanes (the lanes behind them learn the others')
            const int nth = __builtin_amdgcn_ds_permute((pending ? rank : n_left + lane - rank) << 2, lane);
            const int owner = __builtin_amdgcn_ds_bpermute((lane >> shift) << 2, nth) << 2;
            const uint32_t lo = (uint32_t)__builtin_amdgcn_ds_bpermute(owner, (int)(uint32_t)stream), hi = (uint32_t)__builtin_amdgcn_ds_bpermute(owner, (int)(uint32_t)(stream >> 32));
            const int mine = round + (lane & ((1 << shift) - 1)), first_lane = (rank << shift) & (kWave - 1);   // (of the cell, if it is left)
            const int ok = gamma_round(g.dirichlet_alpha, ((uint64_t)hi << 32) | lo, mine, &x);
            const uint64_t accepted = __ballot((ok && mine < PSYN_GAMMA_ROUNDS) || mine == PSYN_GAMMA_ROUNDS - 1);
            const uint32_t of_cell = (uint32_t)(accepted >> first_lane) & ((1u << (1 << shift)) - 1u);
            const float gamma = __int_as_float(__builtin_amdgcn_ds_bpermute((first_lane + (of_cell ? __builtin_ctz(of_cell) : 0)) << 2, __float_as_int(x)));
            if (pending && of_cell != 0) {
                key = psyn_weight_key(gamma, cell);
                pending = false;
            }
            left = __ballot(pending);
            round += 1 << shift;
        }
        const double part_sum = wave_sum_f64(key ? key_weight(key) : 0.0);
        const int part_legal = __popcll(__ballot(legal));
        if (lane == 0) {
            L.weight[group][part] = part_sum;
            L.legal[group][part] = part_legal;
        }
        sort64_descending(key);   // (0: not a legal cell, last)
        L.keys[0][group][part][lane] = key;
    }
    __syncthreads();
    double sum = 0.0;
    int n_legal = 0;
    if (active) {   // two lists of 64 to one of 128: the first meets the second from its end, the larger keys stay in front
        sum = L.weight[group][0] + L.weight[group][1] + L.weight[group][2] + L.weight[group][3];
        n_legal = L.legal[group][0] + L.legal[group][1] + L.legal[group][2] + L.legal[group][3];
        const KeyPair p{key, L.keys[0][group][part ^ 1][kWave - 1 - lane]};
        key = (part & 1) == 0 ? larger_key(p) : smaller_key(p);
        sort64_step<kWave, kWave / 2>(key);
        L.keys[1][group][part][lane] = key;
    }
    __syncthreads();
    if (active) {   // two lists of 128 to one of 256, and that step's first one between two wavefronts at once
        const auto &list = L.keys[1][group];
        const KeyPair near{list[0][lane], list[3][kWave - 1 - lane]}, far{list[1][lane], list[2][kWave - 1 - lane]};
        const KeyPair p = part < 2 ? KeyPair{larger_key(near), larger_key(far)} : KeyPair{smaller_key(near), smaller_key(far)};
        key = (part & 1) == 0 ? larger_key(p) : smaller_key(p);
        sort64_step<kWave, kWave / 2>(key);
        const size_t e = (trow + child) * kEdges + part * kWave + lane;
        if (key != 0) {
            store_edge(g.edges + e, 0, 0.0f, sum == 0.0 ? (float)(1.0 / (double)n_legal) : (float)(key_weight(key) / sum), 0u);
            g.action[e] = (uint8_t)(255u - (key & 0xFFu));
        }
    }
    // (the next node's first keys and weights replace what all have read before the second barrier, its second keys come behind
    // its first barrier)
}

__device__ void evaluator_loop(const LoopArgs &g, EvalLds &L, int tree, int helper, int wave, int lane) {
    EvalRequests &rq = g.requests[tree];
    if (threadIdx.x == 0) __hip_atomic_store(&rq.xcc[1 + helper], my_xcc(), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    bool asked = false, same_l2 = false;
    int seen = 0;   // the last step's tag (steps of which this evaluator had nothing to do may pass it by)
    for (int turn = 0;; turn ^= 1) {
        if (threadIdx.x == 0) {
            const uint64_t start = wall_clock64();
            unsigned long long tag;
            while ((int)(uint32_t)(tag = poll_word(&rq.tag)) >= 0 && (int)(uint32_t)tag <= seen) {
                if (poll_word(&rq.abort) != 0 || wall_clock64() - start > kWaitTicks) {
                    __hip_atomic_store(&rq.abort, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    tag = kSearchOver;
                    break;
                }
                __builtin_amdgcn_s_sleep(2);
            }
            L.tag[turn] = tag;
        }
        if (wave == 0) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");   // for all of the workgroup's wavefronts, which share an L1
        __syncthreads();
        const unsigned long long tag = L.tag[turn];
        seen = __builtin_amdgcn_readfirstlane((int)(uint32_t)tag);
        if (seen < 0) return;
        const int n = __builtin_amdgcn_readfirstlane((int)(tag >> 32) & 0xFF), first_node = __builtin_amdgcn_readfirstlane((int)(tag >> 40));
        int worked_off = 0;
        // (the step's nodes are dealt to the evaluators one by one, so that a step with few of them keeps all busy)
        const int at_once = eval_nodes_at_once();
        for (int first = helper; first < n; first += at_once * g.evaluators) {
            const int group = wave / kEvalParts;
            evaluate_node(g, L, tree, first + group * g.evaluators, n, first_node, group, wave & (kEvalParts - 1), lane);
            for (int i = 0; i < at_once; ++i) worked_off += first + i * g.evaluators < n ? 1 : 0;
        }
        // every wavefront's stores have reached the L2 before one of them reports; the release pushes them on
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __syncthreads();
        if (threadIdx.x == 0 && worked_off > 0) {
            // The tree's workgroup wrote its XCD down before it handed out its first step.  On the same XCD the priors
            // are where it reads them, in the L2 that both share; anywhere else the L2 must be written back first.  (Asked
            // once: the answer took a round trip to the L2 of every step that the tree waited for.)
            if (!asked) {
                asked = true;
                same_l2 = !g.agent_fences && poll_word(&rq.xcc[0]) == my_xcc();
            }
            if (!same_l2) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
            __hip_atomic_fetch_add(&rq.done, worked_off, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

// Until the evaluators have worked off everything handed to them so far; gives up after a bounded wait.
__device__ void wait_for_evaluators(EvalRequests &rq, StepLds &s) {
    const uint64_t start = wall_clock64();
    while (poll_word(&rq.done) < s.requested) {
        if (poll_word(&rq.abort) != 0 || wall_clock64() - start > kWaitTicks) {
            __hip_atomic_store(&rq.abort, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            s.gave_up = 1;
            break;
        }
        __builtin_amdgcn_s_sleep(1);
    }
}

// The whole search in one launch.  evaluators == 0: one workgroup per tree (grid = trees).  Otherwise every tree has
// 1 + evaluators workgroups; those of one tree have the same blockIdx.x % 8, which is how workgroups are dealt to the
// eight XCDs, so a tree's requests and results meet in one L2.
// (FARM: with evaluators; two kernels because their code is 60 KB, the instruction cache of two CUs 64.)
template <bool FARM>
__global__ __launch_bounds__(kTrav *kWave) void search_kernel(const LoopArgs g, int trees) {
    __shared__ StepLds s;
    __shared__ EvalLds eval_lds;
    int *paths = dynamic_lds;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), n_waves = g.traversals;
    int tree = blockIdx.x, role = 0;
    if (FARM) {
        const int per_tree = 1 + g.evaluators, nth = blockIdx.x / 8;
        tree = (int)(blockIdx.x % 8) + 8 * (nth / per_tree);
        role = nth % per_tree;
    }
    if (tree >= trees) return;
    if (FARM && role > 0) {
        if (wave >= kEvalParts * eval_nodes_at_once()) return;
        evaluator_loop(g, eval_lds, tree, role - 1, wave, lane);
        return;
    }
    if (wave >= n_waves) return;   // the launch's workgroups are as large as the larger of the two kinds needs
    constexpr bool farm = FARM;
    EvalRequests &rq = g.requests[tree];
    Work work;
    if (threadIdx.x == 0) {
        s.node_count = g.node_count[tree];
        s.requested = 0;
        s.gave_up = 0;
        if (farm) __hip_atomic_store(&rq.xcc[0], my_xcc(), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    const uint64_t hash_seed = psyn_mix64(psyn_tree_seed(g.seed, tree));
    bool same_l2 = false;   // known: every evaluator of the tree runs on this workgroup's XCD
    uint64_t t0 = wave == 0 ? wall_clock64() : 0;
    for (int step = 0; step < g.steps; ++step) {
        int worked_off = 0;
        select_phase<FARM>(g, s, paths, tree, wave, lane, n_waves, work.nodes_read, work.edges_scored, &rq.done, worked_off);
        work.count_kind(s, wave);
        uint64_t t1 = 0, t2 = 0;
        if (wave == 0) t1 = wall_clock64();
        const Leaf leaf = request_leaf(g, s, tree, wave, lane);   // (the tree's own work: on its way while the evaluators are waited for)
        if (farm) {
            // A node created in the step before can be expanded now at the earliest (selection hands out tickets without
            // looking at a node's priors), so this is where its priors must be there, not a step's length earlier.
            // Selection has read rows of such nodes while they were being written: the L1 drops what it holds.  The first
            // wavefront's acquire does that for all of them, which read no evaluator's work before expand_phase's barrier.
            if (threadIdx.x == 0 && worked_off < s.requested) wait_for_evaluators(rq, s);
            if (wave == 0) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        }
        expand_phase<FARM>(g, s, leaf, hash_seed, tree, wave, lane, n_waves, work.created);
        phase_barrier(farm);   // the claims of the selection and the new nodes are in memory
        if (s.gave_up) break;
        if (farm && threadIdx.x == 0) {   // ... and the evaluators may start on this step's nodes
            s.requested += s.requests;
            if (!same_l2 && !g.agent_fences) {
                same_l2 = true;
                for (int h = 1; h <= g.evaluators; ++h) same_l2 = same_l2 && poll_word(&rq.xcc[h]) == my_xcc();
            }
            // The phase barrier above has the step's nodes and requests in the L2.  Evaluators on the same XCD read them
            // there (their acquire drops what their L1 holds); for any other, or one not heard of yet, the L2 is written
            // back first, which is the expensive part of an agent-scope release.
            if (!same_l2) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
            __hip_atomic_store(&rq.tag, posted(step, s.requests, s.node_count - s.requests), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (wave == 0) t2 = wall_clock64();
        backup_phase(g, s, paths, tree, wave, lane, n_waves);
        phase_barrier(false);
        if (wave == 0) {
            const uint64_t t3 = wall_clock64();
            work.ticks[0] += t1 - t0;
            work.ticks[1] += t2 - t1;
            work.ticks[2] += t3 - t2;
            t0 = t3;
        }
    }
    if (farm) {   // the last step's nodes
        if (threadIdx.x == 0) wait_for_evaluators(rq, s);
        __syncthreads();
    }
    if (farm && threadIdx.x == 0) __hip_atomic_store(&rq.tag, kSearchOver, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    state_to_memory(g, s, paths, tree, n_waves);
    work.to_memory(g, tree, lane);
}

__global__ __launch_bounds__(kTrav *kWave) void select_step_kernel(const LoopArgs g) {
    __shared__ StepLds s;
    int *paths = dynamic_lds;
    const int tree = blockIdx.x, lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), n_waves = blockDim.x / kWave;
    Work work;
    if (threadIdx.x == 0) s.node_count = g.node_count[tree];
    int no_evaluators = 0;
    select_phase<false>(g, s, paths, tree, wave, lane, n_waves, work.nodes_read, work.edges_scored, nullptr, no_evaluators);
    work.count_kind(s, wave);
    state_to_memory(g, s, paths, tree, n_waves);
    work.to_memory(g, tree, lane);
}
__global__ __launch_bounds__(kTrav *kWave) void expand_step_kernel(const LoopArgs g) {
    __shared__ StepLds s;
    int *paths = dynamic_lds;
    const int tree = blockIdx.x, lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), n_waves = blockDim.x / kWave;
    Work work;
    state_from_memory(g, s, paths, tree, n_waves);
    expand_phase<false>(g, s, request_leaf(g, s, tree, wave, lane), psyn_mix64(psyn_tree_seed(g.seed, tree)), tree, wave, lane, n_waves, work.created);
    __syncthreads();
    state_to_memory(g, s, paths, tree, n_waves);
    work.to_memory(g, tree, lane);
}
__global__ __launch_bounds__(kTrav *kWave) void backup_step_kernel(const LoopArgs g) {
    __shared__ StepLds s;
    int *paths = dynamic_lds;
    const int tree = blockIdx.x, lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), n_waves = blockDim.x / kWave;
    state_from_memory(g, s, paths, tree, n_waves);
    backup_phase(g, s, paths, tree, wave, lane, n_waves);
}

// ---- the arrays as the host reads them -------------------------------------------------------------------------------
// One element of array `id` (include/puct_gomoku.h) per thread, written in the [trees, nodes, edges] / [trees, nodes]
// shapes of the selection and backup launchers' arrays.
__global__ void unpack_kernel(const LoopArgs g, int trees, int id, void *dst, size_t count) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    switch (id) {
    case PUCT_GOMOKU_ARR_EDGE_CHILD: {
        const int child = (int)(g.edges[i].link >> 8);
        static_cast<int *>(dst)[i] = child > 0 ? child : -1;
        break;
    }
    case PUCT_GOMOKU_ARR_EDGE_PRIOR: static_cast<float *>(dst)[i] = g.edges[i].prior; break;
    case PUCT_GOMOKU_ARR_EDGE_W: static_cast<float *>(dst)[i] = g.edges[i].w; break;
    case PUCT_GOMOKU_ARR_EDGE_N: static_cast<int *>(dst)[i] = g.edges[i].n; break;
    case PUCT_GOMOKU_ARR_EDGE_INFLIGHT: static_cast<int *>(dst)[i] = (int)(g.edges[i].link & 0xFFu); break;
    case PUCT_GOMOKU_ARR_NODE_EXPANDED: static_cast<int *>(dst)[i] = g.info[i].expanded; break;
    case PUCT_GOMOKU_ARR_NODE_EXPAND_INFLIGHT: static_cast<int *>(dst)[i] = g.info[i].tickets; break;
    case PUCT_GOMOKU_ARR_NODE_TURN: static_cast<int8_t *>(dst)[i] = (g.info[i].legal_turn & kTurnBit) ? -1 : 1; break;
    case PUCT_GOMOKU_ARR_NODE_VALUE: static_cast<float *>(dst)[i] = g.info[i].value; break;
    case PUCT_GOMOKU_ARR_NODE_LEGAL: static_cast<int *>(dst)[i] = g.info[i].legal_turn & 0xFFFF; break;
    case PUCT_GOMOKU_ARR_PATH_VALUES: {
        const size_t out = i / g.path_depth;
        const int d = (int)(i - out * g.path_depth), edges_on_path = g.out_len[out] - 1;
        const float u = g.out_value[out];
        static_cast<float *>(dst)[i] = d < edges_on_path ? (((edges_on_path - d) & 1) ? -u : u) : 0.0f;
        break;
    }
    default: break;
    }
}

// ---- host engine -----------------------------------------------------------------------------------------------------
thread_local std::string g_error;

int fail(int code, const char *fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    g_error = buf;
    return code;
}

#define HIP_TRY(expr)                                                                                       \
    do {                                                                                                    \
        hipError_t err_ = (expr);                                                                           \
        if (err_ != hipSuccess) return fail(PUCT_GOMOKU_E_HIP, "%s failed: %s", #expr, hipGetErrorString(err_)); \
    } while (0)

double now_s() { return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count(); }

}  // namespace

struct puct_gomoku_engine {
    puct_gomoku_config cfg;
    LoopArgs args;
    uint32_t *d_root = nullptr;
    std::vector<void *> allocations;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
};

namespace {
template <typename T>
int alloc(puct_gomoku_engine *e, T **out, size_t count) {
    void *p = nullptr;
    HIP_TRY(hipMalloc(&p, sizeof(T) * count));
    e->allocations.push_back(p);
    *out = static_cast<T *>(p);
    return PUCT_GOMOKU_OK;
}

// Element size and count of array `id`, 0 if there is no such array.
size_t array_shape(const puct_gomoku_config &c, int id, size_t *count) {
    const size_t T = c.trees, N = c.max_nodes, W = c.traversals, D = c.path_depth;
    switch (id) {
    case PUCT_GOMOKU_ARR_EDGE_CHILD: case PUCT_GOMOKU_ARR_EDGE_PRIOR: case PUCT_GOMOKU_ARR_EDGE_W:
    case PUCT_GOMOKU_ARR_EDGE_N: case PUCT_GOMOKU_ARR_EDGE_INFLIGHT: *count = T * N * kEdges; return 4;
    case PUCT_GOMOKU_ARR_EDGE_ACTION: *count = T * N * kEdges; return 1;
    case PUCT_GOMOKU_ARR_NODE_EXPANDED: case PUCT_GOMOKU_ARR_NODE_EXPAND_INFLIGHT: case PUCT_GOMOKU_ARR_NODE_VALUE:
    case PUCT_GOMOKU_ARR_NODE_LEGAL: *count = T * N; return 4;
    case PUCT_GOMOKU_ARR_NODE_TURN: *count = T * N; return 1;
    case PUCT_GOMOKU_ARR_NODE_COUNT: *count = T; return 4;
    case PUCT_GOMOKU_ARR_NODE_BOARD: *count = T * N * kBoardWords; return 4;
    case PUCT_GOMOKU_ARR_OUT_SELECTED: case PUCT_GOMOKU_ARR_OUT_LEN: *count = T * W; return 4;
    case PUCT_GOMOKU_ARR_OUT_PATH: case PUCT_GOMOKU_ARR_PATH_VALUES: *count = T * W * D; return 4;
    default: *count = 0; return 0;
    }
}
}  // namespace

extern "C" const char *puct_gomoku_last_error(void) { return g_error.c_str(); }

extern "C" void puct_gomoku_destroy(puct_gomoku_engine *e) {
    if (!e) return;
    (void)hipSetDevice(e->cfg.device);
    for (void *p : e->allocations) (void)hipFree(p);
    if (e->ev0) (void)hipEventDestroy(e->ev0);
    if (e->ev1) (void)hipEventDestroy(e->ev1);
    if (e->stream) (void)hipStreamDestroy(e->stream);
    delete e;
}

extern "C" int puct_gomoku_create(const puct_gomoku_config *c, puct_gomoku_engine **out) {
    if (!c || !out) return fail(PUCT_GOMOKU_E_INVALID, "null argument");
    if (c->board_m < 5 && c->board_n < 5) return fail(PUCT_GOMOKU_E_INVALID, "board %dx%d cannot hold five in a row", c->board_m, c->board_n);
    if (c->board_m < 1 || c->board_n < 1 || c->board_m * c->board_n > kEdges)
        return fail(PUCT_GOMOKU_E_INVALID, "board %dx%d: need 1 <= m * n <= %d", c->board_m, c->board_n, kEdges);
    if (c->trees < 1) return fail(PUCT_GOMOKU_E_INVALID, "trees = %d, need >= 1", c->trees);
    if (c->traversals < 1 || c->traversals > kTrav)
        return fail(PUCT_GOMOKU_E_INVALID, "traversals = %d, need 1..%d", c->traversals, kTrav);
    if (c->max_nodes < 2 || c->max_nodes > PUCT_GOMOKU_MAX_NODES)
        return fail(PUCT_GOMOKU_E_INVALID, "max_nodes = %d, need 2..%d", c->max_nodes, PUCT_GOMOKU_MAX_NODES);
    if (c->path_depth < 1 || c->path_depth > PUCT_GOMOKU_MAX_PATH_DEPTH)
        return fail(PUCT_GOMOKU_E_INVALID, "path_depth = %d, need 1..%d", c->path_depth, PUCT_GOMOKU_MAX_PATH_DEPTH);
    if (!(c->dirichlet_alpha > 0.0f && c->dirichlet_alpha < 1.0f))
        return fail(PUCT_GOMOKU_E_INVALID, "dirichlet_alpha = %g, need 0 < alpha < 1", (double)c->dirichlet_alpha);
    if (!(c->cpuct >= 0.0f) || !(c->c_pw >= 0.0f)) return fail(PUCT_GOMOKU_E_INVALID, "cpuct and c_pw must not be negative");
    if (c->evaluators < 0 || c->evaluators > kMaxEvaluators)
        return fail(PUCT_GOMOKU_E_INVALID, "evaluators = %d, need 0..%d", c->evaluators, kMaxEvaluators);
    HIP_TRY(hipSetDevice(c->device));
    auto *e = new puct_gomoku_engine();
    e->cfg = *c;
    const size_t T = c->trees, N = c->max_nodes, W = c->traversals, D = c->path_depth;
    LoopArgs &g = e->args;
    int rc = 0;
    if ((rc = alloc(e, &g.edges, T * N * kEdges)) || (rc = alloc(e, &g.info, T * N)) || (rc = alloc(e, &g.board, T * N * kBoardWords)) ||
        (rc = alloc(e, &g.action, T * N * kEdges)) || (rc = alloc(e, &g.node_count, T)) || (rc = alloc(e, &g.out_selected, T * W)) ||
        (rc = alloc(e, &g.out_len, T * W)) || (rc = alloc(e, &g.out_claims, T * W)) || (rc = alloc(e, &g.out_path, T * W * D)) ||
        (rc = alloc(e, &g.out_value, T * W)) || (rc = alloc(e, &g.tally, T * kTally)) || (rc = alloc(e, &g.requests, T)) || (rc = alloc(e, &e->d_root, (size_t)kBoardWords))) {
        puct_gomoku_destroy(e);
        return rc;
    }
    g.cpuct = c->cpuct; g.c_pw = c->c_pw; g.alpha_pw = c->alpha_pw;
    g.m = c->board_m; g.n = c->board_n; g.cells = c->board_m * c->board_n; g.max_nodes = c->max_nodes;
    g.traversals = c->traversals; g.path_depth = c->path_depth; g.steps = 0;
    g.seed = c->seed; g.dirichlet_alpha = c->dirichlet_alpha; g.evaluators = c->evaluators;
    g.agent_fences = c->agent_fences != 0;
    hipError_t err = hipStreamCreate(&e->stream);
    if (err == hipSuccess) err = hipEventCreate(&e->ev0);
    if (err == hipSuccess) err = hipEventCreate(&e->ev1);
    if (err == hipSuccess) err = hipMemset(g.out_path, 0xFF, sizeof(int) * T * W * D);
    if (err != hipSuccess) {
        puct_gomoku_destroy(e);
        return fail(PUCT_GOMOKU_E_HIP, "engine set-up failed: %s", hipGetErrorString(err));
    }
    *out = e;
    return PUCT_GOMOKU_OK;
}

extern "C" int puct_gomoku_run(puct_gomoku_engine *e, const int8_t *board, int32_t turn, int32_t steps, int32_t fused,
                               puct_gomoku_result *res) {
    if (!e || !board || !res) return fail(PUCT_GOMOKU_E_INVALID, "null argument");
    if (turn != 1 && turn != -1) return fail(PUCT_GOMOKU_E_ROOT, "turn must be +1 or -1");
    if (steps < 0) return fail(PUCT_GOMOKU_E_INVALID, "steps must not be negative");
    const puct_gomoku_config &c = e->cfg;
    const int cells = c.board_m * c.board_n;
    uint32_t words[kBoardWords] = {0};
    int empty = 0;
    for (int i = 0; i < cells; ++i) {
        if (board[i] == 1) words[i >> 5] |= 1u << (i & 31);
        else if (board[i] == -1) words[8 + (i >> 5)] |= 1u << (i & 31);
        else if (board[i] == 0) ++empty;
        else return fail(PUCT_GOMOKU_E_ROOT, "cell %d holds %d, expected -1, 0 or +1", i, (int)board[i]);
    }
    if (empty == 0) return fail(PUCT_GOMOKU_E_ROOT, "the root position has no empty cell");
    const double t0 = now_s();
    HIP_TRY(hipSetDevice(c.device));
    LoopArgs g = e->args;
    g.steps = steps;
    hipStream_t s = e->stream;
    HIP_TRY(hipMemcpyAsync(e->d_root, words, sizeof words, hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(init_kernel, dim3(c.trees), dim3(kWave), 0, s, g, e->d_root, (int)turn);
    HIP_TRY(hipGetLastError());
    const dim3 grid(c.trees), block(c.traversals * kWave);
    const size_t lds = sizeof(int) * (size_t)c.traversals * c.path_depth;
    HIP_TRY(hipEventRecord(e->ev0, s));
    if (fused) {
        if (steps > 0) {
            // The tree workgroups and their evaluators wait for each other, so every workgroup of the launch must be
            // resident: as many evaluators per tree as the device takes at once, none if it comes to that.
            int waves = c.traversals, per_cu = 0;
            if (g.evaluators > 0 && waves < 8) waves = 8;
            int cus = 0;
            HIP_TRY(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, c.device));
            HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, search_kernel<true>, waves * kWave, lds));
            const long resident = (long)per_cu * cus, groups = 8L * ((c.trees + 7) / 8);
            while (g.evaluators > 0 && groups * (1 + g.evaluators) > resident) g.evaluators -= 1;
            if (g.evaluators > 0)
                hipLaunchKernelGGL(search_kernel<true>, dim3((unsigned)(groups * (1 + g.evaluators))), dim3(waves * kWave), lds, s, g, (int)c.trees);
            else
                hipLaunchKernelGGL(search_kernel<false>, grid, block, lds, s, g, (int)c.trees);
            HIP_TRY(hipGetLastError());
        }
    } else {
        for (int i = 0; i < steps; ++i) {
            hipLaunchKernelGGL(select_step_kernel, grid, block, lds, s, g);
            hipLaunchKernelGGL(expand_step_kernel, grid, block, lds, s, g);
            hipLaunchKernelGGL(backup_step_kernel, grid, block, lds, s, g);
        }
        HIP_TRY(hipGetLastError());
    }
    HIP_TRY(hipEventRecord(e->ev1, s));
    HIP_TRY(hipStreamSynchronize(s));
    float ms = 0.0f;
    HIP_TRY(hipEventElapsedTime(&ms, e->ev0, e->ev1));
    if (fused && g.evaluators > 0 && steps > 0) {
        std::vector<EvalRequests> rq(c.trees);
        HIP_TRY(hipMemcpy(rq.data(), g.requests, sizeof(EvalRequests) * c.trees, hipMemcpyDeviceToHost));
        for (int t = 0; t < c.trees; ++t)
            if (rq[t].abort)
                return fail(PUCT_GOMOKU_E_SYNC, "tree %d: a workgroup waited for more than 3 s for its partners (are all %d workgroups of "
                            "the launch resident?); the search was abandoned", t, (int)(8 * ((c.trees + 7) / 8) * (1 + g.evaluators)));
    }

    // root tables of all trees
    const size_t T = c.trees, N = c.max_nodes;
    std::vector<Edge> root_edges(T * kEdges);
    std::vector<NodeInfo> root_info(T);
    std::vector<uint8_t> a_root(T * kEdges);
    std::vector<int> counts(T);
    std::vector<unsigned long long> tally(T * kTally);
    HIP_TRY(hipMemcpy2D(root_edges.data(), sizeof(Edge) * kEdges, g.edges, sizeof(Edge) * kEdges * N, sizeof(Edge) * kEdges, T, hipMemcpyDeviceToHost));
    HIP_TRY(hipMemcpy2D(root_info.data(), sizeof(NodeInfo), g.info, sizeof(NodeInfo) * N, sizeof(NodeInfo), T, hipMemcpyDeviceToHost));
    HIP_TRY(hipMemcpy2D(a_root.data(), kEdges, g.action, (size_t)kEdges * N, kEdges, T, hipMemcpyDeviceToHost));
    HIP_TRY(hipMemcpy(counts.data(), g.node_count, sizeof(int) * T, hipMemcpyDeviceToHost));
    HIP_TRY(hipMemcpy(tally.data(), g.tally, sizeof(unsigned long long) * T * kTally, hipMemcpyDeviceToHost));
    memset(res, 0, sizeof *res);
    res->steps = steps;
    for (size_t t = 0; t < T; ++t) {
        for (int sl = 0; sl < root_info[t].expanded && sl < kEdges; ++sl) {
            const int a = a_root[t * kEdges + sl];
            res->root_n[a] += root_edges[t * kEdges + sl].n;
            res->root_w[a] += (double)root_edges[t * kEdges + sl].w;
        }
        for (int k = 0; k < 5; ++k) res->selections[k] += (int64_t)tally[t * kTally + k];
        res->expansions_committed += (int64_t)tally[t * kTally + 5];
        res->nodes_read += (int64_t)tally[t * kTally + 6];
        res->edges_scored += (int64_t)tally[t * kTally + 7];
        res->time_select += 1e-8 * (double)tally[t * kTally + 8] / (double)T;
        res->time_expand += 1e-8 * (double)tally[t * kTally + 9] / (double)T;
        res->time_backup += 1e-8 * (double)tally[t * kTally + 10] / (double)T;
        res->nodes_total += counts[t];
        if (counts[t] > res->max_nodes_in_tree) res->max_nodes_in_tree = counts[t];
    }
    res->best_action = -1;
    for (int a = 0; a < cells; ++a)
        if (res->root_n[a] > res->best_n) { res->best_n = res->root_n[a]; res->best_action = a; }
    res->time_device = ms * 1e-3;
    res->time_total = now_s() - t0;
    return PUCT_GOMOKU_OK;
}

extern "C" int64_t puct_gomoku_array_bytes(puct_gomoku_engine *e, int32_t id) {
    size_t count = 0;
    const size_t elem = e ? array_shape(e->cfg, id, &count) : 0;
    if (elem == 0) return fail(PUCT_GOMOKU_E_INVALID, "unknown array id %d", id);
    return (int64_t)(elem * count);
}

extern "C" int puct_gomoku_read(puct_gomoku_engine *e, int32_t id, void *dst, size_t bytes) {
    size_t count = 0;
    const size_t elem = (e && dst) ? array_shape(e->cfg, id, &count) : 0;
    if (elem == 0) return fail(PUCT_GOMOKU_E_INVALID, "unknown array id %d", id);
    if (bytes != elem * count) return fail(PUCT_GOMOKU_E_INVALID, "array %d has %zu bytes, buffer has %zu", id, elem * count, bytes);
    HIP_TRY(hipSetDevice(e->cfg.device));
    const LoopArgs &g = e->args;
    const void *direct = nullptr;   // arrays the engine keeps in the shape the host reads
    switch (id) {
    case PUCT_GOMOKU_ARR_EDGE_ACTION: direct = g.action; break;
    case PUCT_GOMOKU_ARR_NODE_COUNT: direct = g.node_count; break;
    case PUCT_GOMOKU_ARR_NODE_BOARD: direct = g.board; break;
    case PUCT_GOMOKU_ARR_OUT_SELECTED: direct = g.out_selected; break;
    case PUCT_GOMOKU_ARR_OUT_LEN: direct = g.out_len; break;
    case PUCT_GOMOKU_ARR_OUT_PATH: direct = g.out_path; break;
    default: break;
    }
    if (direct) {
        HIP_TRY(hipMemcpy(dst, direct, bytes, hipMemcpyDeviceToHost));
        return PUCT_GOMOKU_OK;
    }
    // the others are fields of the edge and node records: gathered on the device, then copied
    void *staging = nullptr;
    HIP_TRY(hipMalloc(&staging, bytes));
    const unsigned threads = 256;
    hipLaunchKernelGGL(unpack_kernel, dim3((unsigned)((count + threads - 1) / threads)), dim3(threads), 0, e->stream, g, e->cfg.trees,
                       (int)id, staging, count);
    hipError_t err = hipGetLastError();
    if (err == hipSuccess) err = hipStreamSynchronize(e->stream);
    if (err == hipSuccess) err = hipMemcpy(dst, staging, bytes, hipMemcpyDeviceToHost);
    (void)hipFree(staging);
    if (err != hipSuccess) return fail(PUCT_GOMOKU_E_HIP, "reading array %d failed: %s", id, hipGetErrorString(err));
    return PUCT_GOMOKU_OK;
}
