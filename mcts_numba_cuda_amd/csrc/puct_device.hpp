// Device side of PUCT selection and backup with virtual loss for gfx950 (wave64): one 64-lane wavefront per traversal.
//
// Semantics follow src/puct/puct_gpu_v3_cpp.cu:38-448 (selection with edge-level virtual loss),
// src/puct/puct_gpu_v2.py:573-840 (the two selections with node-level virtual loss) and :847-927 (backup); the
// wavefront-level organisation is this library's own:
//   * the first 64 edges of a node (all of them for almost every node under progressive widening) are loaded once,
//     together with the node's own words, before anything about the node is known, so a level costs one round of
//     loads and one claim instead of a chain of dependent loads;
//   * the reference's total order on edges (score descending, rotated edge index ascending) is taken in two steps: the
//     largest score by a max-reduction of 32-bit keys over DPP row operations, the edge among the equal ones from the
//     lane masks of the comparison with it, on the scalar unit;
//   * a level is written once per number of 64-edge slices the node fills, and everything that is the same in all
//     lanes (node, depth, row addresses, branches) is kept on the scalar side: the kernels are bound by instruction
//     issue, not by the memory they read.
#pragma once
#include <hip/hip_runtime.h>
#include <float.h>
#include <stdint.h>

#include <type_traits>

#include "../../include/puct_select.h"

namespace puct {


constexpr int kWave = 64;
constexpr int kMaxWavesPerBlock = 16;
constexpr int kRecalcAttempts = 2;  // MAX_RECALC_RETRY, src/puct/puct_gpu_v3_cpp.cu:36
constexpr int kPasses = (PUCT_PACKED_EDGE_MASK + 1) / kWave;  // 64-edge slices of the widest node
constexpr int kNoEdge = 0x7fffffff;

struct SelectArgs {
    float cpuct, c_pw, alpha_pw;
    int soft_winner;
    const int *edge_child_id;
    const float *edge_prior;
    const float *edge_W;
    const int *edge_N;
    int *edge_inflight;
    int *node_expand_inflight;
    const int *node_expanded;
    const int *tree_nodes;
    int *out_selected_node;
    int *out_path_eids;
    int *out_path_len;
    int trees, nodes, edges, warps, path_depth;
};

// ---- cross-lane reductions -------------------------------------------------------------------------------------
// DPP controls: quad_perm [1,0,3,2], quad_perm [2,3,0,1], row_half_mirror, row_mirror.  After the four steps every
// lane holds the reduction of its 16-lane row; rows 1 and 3 then take the row before (row_bcast:15), row 3 the lower half
// (row_bcast:31), so that the last lane has all of it.
template <int CTRL>
__device__ __forceinline__ int dpp(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, true);
}

template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_rows(int v) {   // 0 in the other rows
    return __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xF, false);
}

__device__ __forceinline__ int wave_sum(int v) {
    v += dpp<0xB1>(v);
    v += dpp<0x4E>(v);
    v += dpp<0x141>(v);
    v += dpp<0x140>(v);
    v += dpp_rows<0x142, 0xA>(v);
    v += dpp_rows<0x143, 0xC>(v);
    return __builtin_amdgcn_readlane(v, 63);
}

template <int CTRL>
__device__ __forceinline__ uint64_t dpp_max64(uint64_t v) {
    const uint32_t lo = (uint32_t)dpp<CTRL>((int)(uint32_t)v);
    const uint32_t hi = (uint32_t)dpp<CTRL>((int)(uint32_t)(v >> 32));
    const uint64_t o = ((uint64_t)hi << 32) | lo;
    return o > v ? o : v;
}

__device__ __forceinline__ uint64_t read_lane64(uint64_t v, int lane) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, lane);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), lane);
    return ((uint64_t)hi << 32) | lo;
}

__device__ __forceinline__ uint64_t wave_max(uint64_t v) {
    v = dpp_max64<0xB1>(v);
    v = dpp_max64<0x4E>(v);
    v = dpp_max64<0x141>(v);
    v = dpp_max64<0x140>(v);
    const uint64_t a = read_lane64(v, 0), b = read_lane64(v, 16), c = read_lane64(v, 32), d = read_lane64(v, 48);
    const uint64_t ab = a > b ? a : b, cd = c > d ? c : d;
    return ab > cd ? ab : cd;
}

__device__ __forceinline__ int load_relaxed(const int *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A field of one edge of a tree: the tree's array (one address per wavefront, kept in scalar registers for the whole
// traversal) plus a 32-bit byte offset per lane.  A tree is at most 2^14 nodes of 256 edges, 16 MB per field, so the
// offset fits, and a load is one instruction with nothing to add to a 64-bit address first.
template <class T>
__device__ __forceinline__ T *at_bytes(T *tree_field, uint32_t byte_offset) {
    typedef std::conditional_t<std::is_const<T>::value, const char, char> Byte;
    return reinterpret_cast<T *>(reinterpret_cast<Byte *>(tree_field) + byte_offset);
}

// ---- selection ---------------------------------------------------------------------------------------------------
__device__ __forceinline__ int pack_selection(int kind, int node, int slot, int reason) {
    return (reason << PUCT_PACKED_REASON_SHIFT) | (kind << PUCT_PACKED_KIND_SHIFT) | (slot << PUCT_PACKED_SLOT_SHIFT) |
           node;
}

// src/puct/puct_gpu_v3_cpp.cu:43-49, in two parts: what the launch says and what the tree does
__device__ __forceinline__ bool valid_select_shape(int path_depth, int nodes, int edges) { return path_depth >= 1 && nodes > 0 && edges > 0 && edges <= PUCT_PACKED_EDGE_MASK + 1; }
__device__ __forceinline__ bool valid_node_count(int node_cnt, int nodes) { return node_cnt > 0 && node_cnt <= nodes && node_cnt <= PUCT_PACKED_NODE_LIMIT; }

// sqrtf((float)n), correctly rounded, for n >= 1: the rounding of the hardware's root is put right as the compiler does it, without
// what it does for arguments that are tiny, infinite or negative.
__device__ __forceinline__ float sqrt_of_count(int n) {
    const float x = (float)n, root = __builtin_amdgcn_sqrtf(x);
    const float below = __uint_as_float(__float_as_uint(root) - 1u), above = __uint_as_float(__float_as_uint(root) + 1u);
    const float rounded = __builtin_fmaf(-below, root, x) <= 0.0f ? below : root;
    return __builtin_fmaf(-above, root, x) > 0.0f ? above : rounded;
}

// Progressive widening, src/puct/puct_gpu_v3_cpp.cu:150-157.
__device__ __forceinline__ int allowed_children(float c_pw, float alpha_pw, int n_node, int edges, float sqrt_n_node) {
    const float val = __builtin_expect(alpha_pw == 0.5f, 1) ? c_pw * sqrt_n_node : c_pw * powf((float)n_node, alpha_pw);
    if (val >= (float)edges) return edges;
    const int allowed = (int)ceilf(val);
    return allowed > 1 ? allowed : 1;
}
__device__ __forceinline__ int allowed_children(float c_pw, float alpha_pw, int n_node, int edges) {
    return allowed_children(c_pw, alpha_pw, n_node, edges, sqrt_of_count(n_node));
}

// The score of an edge (src/puct/puct_gpu_v3_cpp.cu:171-180) is q + u with q = n > 0 ? w / n : 0 and
// u = cpuct * prior * sqrt_parent / (n + inflight + 1), in single precision, operation by operation.  The selections
// below keep q and the numerator of u per edge and divide again when the in-flight counts have been read again.

// One 64-bit key per candidate edge (used by the Gomoku search loop) whose unsigned order is the reference's order "higher score first, then smaller
// rotated edge index" (src/puct/puct_gpu_v3_cpp.cu:51-71).  0 means "not a candidate": the reference starts from
// (-FLT_MAX, no edge) and accepts a score that is greater than or equal to it, so NaN and -inf never win.  -0.0f is
// made +0.0f because the reference compares floats, for which the two are equal.
__device__ __forceinline__ uint64_t candidate_key(float score, int eid, int tie_offset, int span) {
    if (!(score >= -FLT_MAX)) return 0;
    const uint32_t b = __float_as_uint(score + 0.0f);
    const uint32_t ordered = (b & 0x80000000u) ? ~b : (b | 0x80000000u);
    int key = eid - tie_offset;
    if (key < 0) key += span;
    return ((uint64_t)ordered << 32) | ((uint32_t)(0xFFFF - key) << 16) | (uint32_t)eid;
}

// The same order with the score and the edge index kept apart, for the selection kernels of this file: a
// 32-bit key per edge whose unsigned order is the order of the scores (0 = not a candidate, as above), the largest of
// which is found with one `v_max_u32` per DPP step; the edge among the equal ones comes from the lane masks of the
// comparison with that maximum, on the scalar unit.
__device__ __forceinline__ uint32_t score_key(float score) {
    if (!(score >= -FLT_MAX)) return 0;
    const uint32_t b = __float_as_uint(score + 0.0f);
    return b ^ ((uint32_t)((int32_t)b >> 31) | 0x80000000u);
}

__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
    auto larger = [](uint32_t x, int o) { return (uint32_t)o > x ? (uint32_t)o : x; };
    v = larger(v, dpp<0xB1>((int)v));
    v = larger(v, dpp<0x4E>((int)v));
    v = larger(v, dpp<0x141>((int)v));
    v = larger(v, dpp<0x140>((int)v));
    v = larger(v, dpp_rows<0x142, 0xA>((int)v));
    v = larger(v, dpp_rows<0x143, 0xC>((int)v));
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// The edge with the largest key (keys[i] belongs to edge lane + 64 i; `skip` takes no part); among equal keys the one
// whose index rotated by tie_offset is smallest, i.e. the first at or after tie_offset, else the first.  kNoEdge if no
// key is above 0.  Every lane returns the same value.
template <int S>
__device__ __forceinline__ int best_edge(const uint32_t (&keys)[S], int lane, int skip, int tie_offset) {
    uint32_t k[S], m = 0;
#pragma unroll
    for (int i = 0; i < S; ++i) {
        k[i] = lane + i * kWave == skip ? 0u : keys[i];
        m = k[i] > m ? k[i] : m;
    }
    m = wave_max_u32(m);
    if (m == 0) return kNoEdge;
    int at_or_after = kNoEdge, first = kNoEdge;
#pragma unroll
    for (int i = 0; i < S; ++i) {
        const uint64_t equal = __builtin_amdgcn_ballot_w64(k[i] == m);
        const int from = tie_offset - i * kWave;   // lanes of this slice at or after the offset: from `from` on
        const uint64_t late = equal & (from <= 0 ? ~0ull : from >= kWave ? 0ull : ~0ull << from);
        if (first == kNoEdge && equal != 0) first = i * kWave + __builtin_ctzll(equal);
        if (at_or_after == kNoEdge && late != 0) at_or_after = i * kWave + __builtin_ctzll(late);
    }
    return at_or_after != kNoEdge ? at_or_after : first;
}

// The claims in flight on one tree's edges, edge_inflight[tree, :, :].  While a launch runs they are read and changed by
// the traversals of that tree only, so where they are kept depends on how many those are:
//   * OWN: one.  Nobody else changes a claim between its read and the winner's, so the claim is an ordinary store, by the
//     lane that reads that edge, and the row of claims one more load beside the row's other fields.  No LDS, so a CU holds
//     32 such traversals, which is what hides the memory behind a level: each is a chain of dependent levels.
//   * LDS: the wavefronts of one workgroup (up to 16), and the tree is small enough (nodes * edges words).  The workgroup
//     keeps the claims in LDS for the launch: loaded at the start, stored at the end, every read of a node's row and every
//     claim in between an LDS operation instead of an agent-scope load and an atomic performed at the memory side.
//   * SHARED: otherwise, the agent-scope loads and atomics.
typedef __attribute__((address_space(3))) int *LdsInts;
enum class ClaimsIn { SHARED, LDS, OWN };
template <ClaimsIn WHERE>
struct EdgeClaims {
    static constexpr bool LOCAL = WHERE == ClaimsIn::LDS;
    int *in_memory;     // edge_inflight + tree * nodes * edges
    LdsInts in_lds;     // the same counters, the workgroup's copy
    // (at: byte offset of the edge's slot in the tree, (node * edges + edge) * 4)
    __device__ __forceinline__ int peek(uint32_t at) const {
        if (LOCAL) return __hip_atomic_load(in_lds + (at >> 2), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (WHERE == ClaimsIn::OWN) return *at_bytes(in_memory, at);
        return load_relaxed(at_bytes(in_memory, at));
    }
    __device__ __forceinline__ void set(uint32_t at, int v) const { *at_bytes(in_memory, at) = v; }   // OWN: by the lane that peeks there
    __device__ __forceinline__ void add(uint32_t at, int v) const {
        if (LOCAL) __hip_atomic_fetch_add(in_lds + (at >> 2), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        else atomicAdd(at_bytes(in_memory, at), v);
    }
    __device__ __forceinline__ int cas(uint32_t at, int expected, int desired) const {   // returns the value found
        if (LOCAL) {
            __hip_atomic_compare_exchange_strong(in_lds + (at >> 2), &expected, desired, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            return expected;
        }
        return atomicCAS(at_bytes(in_memory, at), expected, desired);
    }
};

// The path of a traversal: lane l holds entry l of the 64 it is in the middle of, and they are stored together when they are
// complete and when the traversal ends (a store by one lane at every level was as many instructions as four levels' tests for an end).
// A traversal that gives way takes its claims back by them, and reads back only what it has stored before, past the L1: all it has to wait
// for is that the stores have reached the L2 (and with them the claims that its atomics take back, where those were stores too).  A
// device-scope fence would write the L2 back: with 1024 trees of 8 traversals, most of which give way to another, 8192 of those
// were five sixths of a launch (122 us, 4097 nodes of 64 edges a tree, paths of two levels).
__device__ __forceinline__ void wait_path_stores() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

struct Path {
    int *entries;
    int mine = 0;   // entry lane + 64 i, where 64 i .. depth - 1 have not been stored yet
    __device__ __forceinline__ void append(int depth, int encoded, int lane) {
        mine = lane == (depth & (kWave - 1)) ? encoded : mine;
        if ((depth & (kWave - 1)) == kWave - 1) entries[depth - (kWave - 1) + lane] = mine;
    }
    __device__ __forceinline__ void finish(int depth, int lane) const {
        if (lane < (depth & (kWave - 1))) entries[(depth & ~(kWave - 1)) + lane] = mine;
    }
};

// Takes back the virtual loss of the first `depth` path entries (src/puct/puct_gpu_v3_cpp.cu:206-217).
template <ClaimsIn WHERE>
__device__ __forceinline__ void rollback_path(const SelectArgs &a, const EdgeClaims<WHERE> &claims, const Path &path, int depth, int lane, int node_cnt) {
    const int stored = depth & ~(kWave - 1);
    if (WHERE == ClaimsIn::OWN || stored > 0) wait_path_stores();
    for (int d = lane; d < depth; d += kWave) {
        const int encoded = d < stored ? load_relaxed(path.entries + d) : path.mine;
        const int parent = encoded >> 8, slot = encoded & 0xFF;
        if (parent >= 0 && parent < node_cnt && slot < a.edges)
            claims.add(((uint32_t)parent * (uint32_t)a.edges + (uint32_t)slot) * 4u, -1);
    }
}

// One traversal (tree, wid) by one wavefront; every lane of the wavefront must call it.  A level is written once per
// number S of 64-edge slices that the node's expanded edges fill (1..4, the same for all lanes): these kernels are bound
// by the wavefronts' instruction issue, vector and scalar together, and a level written for "up to four slices" spends a
// third of it on finding out, slice by slice, that a slice is not there.
template <ClaimsIn WHERE>
__device__ __forceinline__ void select_traversal(const SelectArgs &a, const EdgeClaims<WHERE> &claims, int tree, int wid, int lane) {
    static_assert(kPasses == 4, "the levels below are written for one to four slices");
    const size_t out = (uint64_t)(uint32_t)tree * (uint32_t)a.warps + (uint32_t)wid;
    int *const entries = a.out_path_eids + out * (uint32_t)a.path_depth;
    const int nodes = a.nodes, edges = a.edges;
    int final_packed = pack_selection(PUCT_SELECT_INVALID, PUCT_PACKED_NODE_MASK, 0, PUCT_REASON_INVALID_SHAPE);
    int final_len = 0;

    if (valid_select_shape(a.path_depth, nodes, edges)) {
        const size_t tree_nodes = (uint64_t)(uint32_t)tree * (uint32_t)nodes, tree_edges = tree_nodes * (uint32_t)edges;
        const int *const tree_n = a.edge_N + tree_edges, *const tree_c = a.edge_child_id + tree_edges, *const tree_expanded = a.node_expanded + tree_nodes;
        const float *const tree_p = a.edge_prior + tree_edges, *const tree_w = a.edge_W + tree_edges;
        int *const tree_tickets = a.node_expand_inflight + tree_nodes;
        const int asked_node_cnt = load_relaxed(a.tree_nodes + tree);
        int node = 0, depth = 0, node_cnt = 0;
        uint32_t bound = 0;   // a node's expansion word at or beyond which there is more to ask: the root's always, then an end of a game or no width
        Path path{entries};
        while (true) {
            // (the same in all lanes; said so that the level's addresses and branches are worked out once per wavefront)
            node = __builtin_amdgcn_readfirstlane(node), depth = __builtin_amdgcn_readfirstlane(depth);
            const uint32_t node4 = (uint32_t)node * 4u, row4 = node4 * (uint32_t)edges;   // byte offsets of the node, and of its edges, in the tree's fields

            // Everything a level can need from the first 64 edges, requested in one go, before the node's width is known
            // (lanes beyond the row read its last edge and take no part); the edges of wider nodes follow once it is
            // and stay in registers for the rest of the level.  (Requested at the end of the level before, which moves the claims
            // apart from the rest: deep trees a quarter slower.)
            const uint32_t at0 = row4 + (uint32_t)(lane < edges ? lane : edges - 1) * 4u;
            const int n0 = *at_bytes(tree_n, at0), f0 = claims.peek(at0), c0 = *at_bytes(tree_c, at0);
            const float p0 = *at_bytes(tree_p, at0), w0 = *at_bytes(tree_w, at0);
            const int node_info = *at_bytes(tree_expanded, node4);
            const int tickets = load_relaxed(at_bytes(tree_tickets, node4));

            // A node without an edge, or with one: no score to work out.
            const int cur_expanded = node_info;
            auto try_expand = [&](int allowed) __attribute__((always_inline)) -> int {   // expansion ticket, src/puct/puct_gpu_v3_cpp.cu:219-233; -1: none
                int expand_slot = -1;
                if (cur_expanded + tickets < allowed) {
                    if (lane == 0) {
                        const int slot = cur_expanded + atomicAdd(at_bytes(tree_tickets, node4), 1);
                        if (slot < allowed)
                            expand_slot = slot;
                        else
                            atomicSub(at_bytes(tree_tickets, node4), 1);
                    }
                    expand_slot = __builtin_amdgcn_readfirstlane(expand_slot);
                }
                return expand_slot;
            };
            auto narrow = [&]() __attribute__((always_inline)) -> int {
                int allowed = allowed_children(a.c_pw, 0.5f, 1, edges, 1.0f);   // (no visits: 1 ** alpha_pw is 1, whatever alpha_pw is)
                if (cur_expanded == 1) {
                    const int total = __builtin_amdgcn_readfirstlane(n0 + f0), parent_eff = total > 1 ? total : 1;
                    allowed = a.c_pw != 0.0f ? allowed_children(a.c_pw, a.alpha_pw, parent_eff, edges) : 1;
                }
                if (allowed > cur_expanded) {
                    const int expand_slot = try_expand(allowed);
                    if (expand_slot >= 0) return ~pack_selection(PUCT_SELECT_EXPAND, node, expand_slot, PUCT_REASON_OK_EXPAND);
                    if (cur_expanded == 0) return ~pack_selection(PUCT_SELECT_BUSY, node, 0, PUCT_REASON_BUSY_EXPAND_INFLIGHT);
                }
                const int child = __builtin_amdgcn_readfirstlane(c0);
                if ((uint32_t)child >= (uint32_t)node_cnt) return ~pack_selection(PUCT_SELECT_INVALID, PUCT_PACKED_NODE_MASK, 0, PUCT_REASON_INVALID_CHILD_OOB);
                if (lane == 0) {
                    if (WHERE == ClaimsIn::OWN) claims.set(row4, f0 + 1);
                    else claims.add(row4, 1);
                }
                path.append(depth, node << 8, lane);
                return child;
            };

            // The level proper.
            auto level = [&](auto slices) __attribute__((always_inline)) -> int {
                constexpr int S = decltype(slices)::value;   // (S - 1) * 64 < cur_expanded <= S * 64, two at least
                constexpr int CS = S <= 2 ? S : 1;   // slices whose row of children is requested with the scores' fields (see best_child below)
                int n[S], f[S], c[CS];
                // byte offset of the edge that this lane looks at in slice i (lanes beyond the node's edges: its last edge)
                auto at = [&](int i) {
                    const int eid = lane + i * kWave;
                    return i == 0 ? at0 : row4 + (uint32_t)(i < S - 1 || eid < cur_expanded ? eid : cur_expanded - 1) * 4u;
                };
                float p[S], w[S];
                bool in_node[S];
                n[0] = n0, f[0] = f0, p[0] = p0, w[0] = w0, c[0] = c0;
#pragma unroll
                for (int i = 1; i < S; ++i) {
                    const uint32_t here = at(i);
                    n[i] = *at_bytes(tree_n, here), f[i] = claims.peek(here), p[i] = *at_bytes(tree_p, here), w[i] = *at_bytes(tree_w, here);
                    if (i < CS) c[i] = *at_bytes(tree_c, here);
                }
#pragma unroll
                for (int i = 0; i < S; ++i) in_node[i] = i < S - 1 || lane + i * kWave < cur_expanded;

                int total = 0;
#pragma unroll
                for (int i = 0; i < S; ++i) total += in_node[i] ? n[i] + f[i] : 0;
                total = wave_sum(total);
                const int parent_eff = total > 1 ? total : 1;
                const float sqrt_parent = sqrt_of_count(parent_eff);
                if (a.c_pw != 0.0f) {   // (else there is one child allowed, and there are two)
                    const int allowed = allowed_children(a.c_pw, a.alpha_pw, parent_eff, edges, sqrt_parent);
                    if (allowed > cur_expanded) {
                        const int expand_slot = try_expand(allowed);
                        if (expand_slot >= 0) return ~pack_selection(PUCT_SELECT_EXPAND, node, expand_slot, PUCT_REASON_OK_EXPAND);
                    }
                }

                int tie_offset = WHERE == ClaimsIn::OWN ? 0 : wid;
                if (tie_offset >= cur_expanded) tie_offset %= cur_expanded;

                auto of_edge = [&](const int (&v)[S], int eid) {
                    const int lane_of = eid & (kWave - 1), pass = eid / kWave;
                    int r = __builtin_amdgcn_readlane(v[0], lane_of);
#pragma unroll
                    for (int i = 1; i < S; ++i)
                        if (pass == i) r = __builtin_amdgcn_readlane(v[i], lane_of);
                    return r;
                };

                // Where the winner leads: for nodes of up to 128 edges the row of children came with the scores' fields; of a
                // wider node only its first 64, and beyond them just the winner's word is asked for, on its way while the
                // claim is made (the rest of that row is a sixth of what such a level reads -- and those launches are bound by
                // what they read -- and three registers per lane; at 128 edges waiting for the word cost more than the row).
                int best_eid = kNoEdge, held = 0, best_child = 0;
                // Winner-recalc claim, src/puct/puct_gpu_v3_cpp.cu:235-275: score all edges, try to move the winner's
                // in-flight count from the value the score was computed with to that value plus one, rescore once if
                // another traversal got there first.  The mean value and the numerator of the exploration term do not
                // depend on the in-flight counts, so a second evaluation divides once per edge, and only in the slices
                // whose counts have changed (other traversals' claims sit on a few edges).
                float q[S], num[S];
#pragma unroll
                for (int i = 0; i < S; ++i) {
                    // (of a node of several slices, one none of whose edges has a visit or a value has q = +0 without dividing)
                    q[i] = 0.0f;
                    if (S == 1 || __builtin_amdgcn_ballot_w64(n[i] > 0 && __float_as_uint(w[i]) != 0u) != 0) q[i] = n[i] > 0 ? w[i] / (float)n[i] : 0.0f;
                    num[i] = a.cpuct * p[i] * sqrt_parent;
                }
                uint32_t keys[S];
                auto score_slice = [&](int i, int inflight) {
                    return in_node[i] ? score_key(q[i] + num[i] / (float)(n[i] + inflight + 1)) : 0u;
                };
                for (int attempt = 0; attempt < kRecalcAttempts; ++attempt) {
                    if (attempt == 0) {
#pragma unroll
                        for (int i = 0; i < S; ++i) keys[i] = score_slice(i, f[i]);
                    } else {
#pragma unroll
                        for (int i = 0; i < S; ++i) {
                            const int fi = claims.peek(at(i));
                            if (__builtin_amdgcn_ballot_w64(fi != f[i]) != 0) {
                                f[i] = fi;
                                keys[i] = score_slice(i, fi);
                            }
                        }
                    }
                    best_eid = best_edge<S>(keys, lane, -1, tie_offset);
                    if (best_eid == kNoEdge) break;
                    if (S == CS || best_eid < CS * kWave) {
                        best_child = __builtin_amdgcn_readlane(c[0], best_eid & (kWave - 1));
                        if (CS > 1 && best_eid >= kWave) best_child = __builtin_amdgcn_readlane(c[CS - 1], best_eid & (kWave - 1));
                    } else {
                        best_child = load_relaxed(at_bytes(tree_c, row4 + (uint32_t)best_eid * 4u));   // (every lane the same word)
                    }
                    if (WHERE == ClaimsIn::OWN) {
                        held = 1;
                        break;
                    }
                    const int best_inflight = of_edge(f, best_eid);
                    int got = 0;
                    if (lane == 0) {
                        const int prev = claims.cas(row4 + (uint32_t)best_eid * 4u, best_inflight, best_inflight + 1);
                        got = prev == best_inflight ? 1 : 0;
                    }
                    held = __builtin_amdgcn_readfirstlane(got);
                    if (held) break;
                }
                if (WHERE != ClaimsIn::OWN && a.soft_winner != 0 && held == 0 && best_eid != kNoEdge) {
                    if (lane == 0) claims.add(row4 + (uint32_t)best_eid * 4u, 1);
                    held = 1;
                }

                if (held == 0)
                    return best_eid == kNoEdge ? ~pack_selection(PUCT_SELECT_INVALID, PUCT_PACKED_NODE_MASK, 0, PUCT_REASON_INVALID_NO_VALID_EDGE)
                                               : ~pack_selection(PUCT_SELECT_BUSY, node, 0, PUCT_REASON_BUSY_WINNER_RECALC);

                best_child = __builtin_amdgcn_readfirstlane(best_child);
                if ((uint32_t)best_child >= (uint32_t)node_cnt) {
                    if (WHERE != ClaimsIn::OWN && lane == 0) claims.add(row4 + (uint32_t)best_eid * 4u, -1);
                    return ~pack_selection(PUCT_SELECT_INVALID, PUCT_PACKED_NODE_MASK, 0, PUCT_REASON_INVALID_CHILD_OOB);
                }
                if (WHERE == ClaimsIn::OWN) {   // (the claim, now that the edge is known to lead somewhere)
#pragma unroll
                    for (int i = 0; i < S; ++i)
                        if (lane + i * kWave == best_eid) claims.set(row4 + (uint32_t)best_eid * 4u, f[i] + 1);
                }
                path.append(depth, (node << 8) | best_eid, lane);
                return best_child;
            };

            // Where the traversal goes on, or the complement of its selection word where it ends.
            int next = 0;
            if (__builtin_expect((uint32_t)node_info >= bound, 0)) {
                if (bound == 0) {   // (how many nodes the tree has is not waited for before the root's row is on its way)
                    int count = asked_node_cnt;
                    asm volatile("" : "+v"(count));
                    node_cnt = __builtin_amdgcn_readfirstlane(count);
                    bound = (uint32_t)edges + 1u;
                    if (!valid_node_count(node_cnt, nodes)) next = ~pack_selection(PUCT_SELECT_INVALID, PUCT_PACKED_NODE_MASK, 0, PUCT_REASON_INVALID_SHAPE);
                }
                if (next == 0 && node_info == PUCT_NODE_EXPANDED_TERMINAL) next = ~pack_selection(PUCT_SELECT_TERMINAL, node, 0, PUCT_REASON_OK_TERMINAL);
                else if (next == 0 && (uint32_t)node_info >= bound) next = ~pack_selection(PUCT_SELECT_INVALID, PUCT_PACKED_NODE_MASK, 0, PUCT_REASON_INVALID_NODE_INFO);
            }
            if (next == 0) {
                if (depth >= a.path_depth) next = ~pack_selection(PUCT_SELECT_DEPTH_LIMIT, node, 0, PUCT_REASON_OK_DEPTH_LIMIT);
                else if (cur_expanded <= 1) next = narrow();
                else if (cur_expanded <= kWave) next = level(std::integral_constant<int, 1>{});
                else if (cur_expanded <= 2 * kWave) next = level(std::integral_constant<int, 2>{});
                else if (cur_expanded <= 3 * kWave) next = level(std::integral_constant<int, 3>{});
                else next = level(std::integral_constant<int, 4>{});
            }
            if (next < 0) {
                final_packed = ~next;
                break;
            }
            node = next;
            depth += 1;
        }
        const int kind = (final_packed >> PUCT_PACKED_KIND_SHIFT) & PUCT_PACKED_KIND_MASK;
        if (kind == PUCT_SELECT_INVALID || kind == PUCT_SELECT_BUSY) rollback_path(a, claims, path, depth, lane, node_cnt);
        else final_len = depth + 1;
        path.finish(depth, lane);
    }

    if (lane == 0) {
        a.out_selected_node[out] = final_packed;
        a.out_path_len[out] = final_len;
    }
}

// ---- selection with node-level virtual loss ------------------------------------------------------------------------
// The two selection kernels of src/puct/puct_gpu_v2.py, whose virtual loss lives in node_inflight[tree, child] and is
// what backup_traversal<true> below takes back: _select_kernel_native (:573-697; every candidate child is claimed
// before it is scored and the losers are released afterwards) and _select_kernel_winner_recalc (:700-840; scores from
// the counters as read, a counter compare-and-swap on the winner only, one re-evaluation without the first winner
// when that child already carried claims).  Their selection word has no reason field and no BUSY kind: a traversal
// that cannot get an expansion ticket, or finds no edge, gives its claims back and reports PACKED_INVALID with length 0.
struct NodeSelectArgs {
    float cpuct, c_pw, alpha_pw;
    const int *edge_child_id;
    const float *edge_prior;
    const float *edge_W;
    const int *edge_N;
    int *node_inflight;
    int *node_expand_inflight;
    const int *node_expanded;
    const int *node_count;
    int *out_selected_node;
    int *out_path_eids;
    int *out_path_len;
    int trees, nodes, edges, warps, path_depth;
};

constexpr int kPackedInvalidV2 = (PUCT_SELECT_INVALID << PUCT_PACKED_KIND_SHIFT) | PUCT_PACKED_NODE_MASK;

__device__ __forceinline__ int pack_selection_v2(int kind, int node, int slot) {
    return (kind << PUCT_PACKED_KIND_SHIFT) | (slot << PUCT_PACKED_SLOT_SHIFT) | node;
}

// The virtual visits of one tree's nodes, node_inflight[tree, :].  While a launch runs they are read and changed by
// the traversals of that tree only; when those are the wavefronts of one workgroup (up to 16 traversals per tree) and the
// tree's counters fit, the workgroup keeps them in LDS for the launch (LOCAL): loaded at the start, stored at the end, and
// every claim in between is an LDS atomic instead of one performed at the memory side (the preclaim kernel makes two per
// edge and level; in device memory they were what bounded it).
template <bool LOCAL>
struct NodeVisits {
    int *in_memory;     // node_inflight + tree * nodes
    LdsInts in_lds;     // the same counters, workgroup's copy
    __device__ __forceinline__ int peek(int node) const {
        if (LOCAL) return __hip_atomic_load(in_lds + node, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        return load_relaxed(in_memory + node);
    }
    __device__ __forceinline__ int add(int node, int v) const {   // returns the count found
        if (LOCAL) return __hip_atomic_fetch_add(in_lds + node, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        return atomicAdd(in_memory + node, v);
    }
    __device__ __forceinline__ void sub(int node, int v) const {
        if (LOCAL) __hip_atomic_fetch_sub(in_lds + node, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        else atomicSub(in_memory + node, v);
    }
};

// src/puct/puct_gpu_v2.py:291-310: the claims of the first `depth` path entries live on the child each entry leads to.
template <bool LOCAL>
__device__ __forceinline__ void rollback_node_path(const NodeSelectArgs &a, const NodeVisits<LOCAL> &visits_of, const Path &path, int tree, int depth, int lane,
                                                   int node_limit) {
    const int stored = depth & ~(kWave - 1);
    if (stored > 0) wait_path_stores();
    for (int d = lane; d < depth; d += kWave) {
        const int encoded = d < stored ? load_relaxed(path.entries + d) : path.mine;
        if (encoded < 0) continue;
        const int parent = encoded >> 8, slot = encoded & 0xFF;
        if (parent < node_limit && slot < a.edges) {
            const int child = a.edge_child_id[((size_t)tree * a.nodes + parent) * a.edges + slot];
            if (child >= 0 && child < node_limit) visits_of.sub(child, 1);
        }
    }
}

// The claim of the winner-recalc kernel (src/puct/puct_gpu_v2.py:313-349) is one more virtual visit on the child's
// counter; "conflict" = the counter already held visits when the claim went in.  The reference moves the counter from the
// value it read to that value plus one with compare-and-swap, reads again when the exchange is lost, and after
// MAX_SELECT_RETRY lost exchanges adds one atomically instead: a counter, not a lock, so every claim goes in and all it
// learns is the value it found.  That is a fetch-and-add, which is what node_select_traversal does, without the lost
// exchanges (the traversals of a tree that reach a node together all claim the same child, and compare-and-swap then
// costs a round trip per traversal ahead).

// One traversal (tree, wid) by one wavefront; every lane of the wavefront must call it.  A level is written once per
// number S of 64-edge slices that the node's expanded edges fill (1..4, the same for all lanes): what bounds these
// kernels is the wavefronts' instruction issue, vector and scalar together, and a level written for "up to four slices"
// spends a third of it on finding out, slice by slice, that a slice is not there.
// before_claims is called once, before the counters are looked at, where the launch has a valid shape.
template <bool PRECLAIM, bool LOCAL, class BeforeClaims>
__device__ __forceinline__ void node_select_traversal(const NodeSelectArgs &a, const NodeVisits<LOCAL> &visits_of, int tree, int wid, int lane, BeforeClaims before_claims) {
    static_assert(kPasses == 4, "the levels below are written for one to four slices");
    // Preclaims in memory: the traversals of a tree (more than 16, where it matters) are bound by their atomics on the same few lines, and the sooner
    // each comes to them the more they are in each other's way.  A widening limit that nobody needs is worked out between the reads and the
    // claims, and beyond 64 edges the depth is asked for apart from the other ends.  us a selection and its backup of 64 trees, before levels asked
    // for ends once / with neither / the first / both: 129 x 128, 32 traversals, 256 levels 3223 / 3649 / 3390 / 3129, 24 traversals, 128 levels
    // 1483 / 1732 / 1570 / 1444; 65 x 64, 32 traversals, 256 levels 1968 / 2009 / 1981 / 2000, 64 traversals, 128 levels 1571 / 1515 / 1521 / 1549 (2518
    // with the depth apart at 64 edges too); 256 of 257 x 256, 32 traversals, 256 levels 10600 / 10700 / 9890 / 9850.
    constexpr bool CONTENDED = PRECLAIM && !LOCAL;
    const size_t out = (uint64_t)(uint32_t)tree * (uint32_t)a.warps + (uint32_t)wid;
    int *const entries = a.out_path_eids + out * (uint32_t)a.path_depth;
    const int nodes = a.nodes, edges = a.edges;

    int final_packed = kPackedInvalidV2, final_len = 0;
    if (valid_select_shape(a.path_depth, nodes, edges)) {   // src/puct/puct_gpu_v2.py:357-366
        const size_t tree_nodes = (uint64_t)(uint32_t)tree * (uint32_t)nodes, tree_edges = tree_nodes * (uint32_t)edges;
        const int *const tree_c = a.edge_child_id + tree_edges, *const tree_n = a.edge_N + tree_edges, *const tree_expanded = a.node_expanded + tree_nodes;
        const float *const tree_p = a.edge_prior + tree_edges, *const tree_w = a.edge_W + tree_edges;
        int *const tree_tickets = a.node_expand_inflight + tree_nodes;
        // the first 64 edges are requested together with the node's own words, before the node's width is known (lanes beyond the row
        // read its last edge and take no part), when the level before has chosen the node
        struct Row { int n, c, info, tickets; float p, w; };
        const uint32_t lane4 = (uint32_t)(lane < edges ? lane : edges - 1) * 4u;
        auto request = [=](int node) __attribute__((always_inline)) -> Row {
            const uint32_t node4 = (uint32_t)node * 4u, at0 = node4 * (uint32_t)edges + lane4;
            Row r;
            r.c = *at_bytes(tree_c, at0), r.n = *at_bytes(tree_n, at0), r.p = *at_bytes(tree_p, at0), r.w = *at_bytes(tree_w, at0);
            r.info = *at_bytes(tree_expanded, node4), r.tickets = load_relaxed(at_bytes(tree_tickets, node4));
            return r;
        };
        int node = 0, depth = 0;
        Row row = request(0);
        const int node_limit = a.node_count[tree];
        before_claims();
        Path path{entries};
        while (valid_node_count(node_limit, nodes)) {
            // (the same in all lanes; said so that the level's addresses and branches are worked out once per wavefront)
            node = __builtin_amdgcn_readfirstlane(node), depth = __builtin_amdgcn_readfirstlane(depth);
            const uint32_t node4 = (uint32_t)node * 4u, row4 = node4 * (uint32_t)edges;   // byte offsets of the node, and of its edges, in the tree's fields
            const int n0 = row.n, c0 = row.c, node_info = row.info, tickets = row.tickets;
            const float p0 = row.p, w0 = row.w;
            const int cur_expanded = node_info;
            // Expansion ticket, :389-403.  Tickets are only given back by the backup, and a ticket beyond the quota is
            // returned at once, so a counter that already shows the quota used up stays that way for this launch.
            auto expand = [&](int allowed) __attribute__((always_inline)) -> int {
                int expand_slot = -1;
                if (cur_expanded + tickets < allowed) {
                    if (lane == 0) {
                        const int slot = cur_expanded + atomicAdd(at_bytes(tree_tickets, node4), 1);
                        if (slot < allowed)
                            expand_slot = slot;
                        else
                            atomicSub(at_bytes(tree_tickets, node4), 1);
                    }
                    expand_slot = __builtin_amdgcn_readfirstlane(expand_slot);
                }
                return ~(expand_slot >= 0 ? pack_selection_v2(PUCT_SELECT_EXPAND, node, expand_slot) : kPackedInvalidV2);
            };

            // The level proper.
            auto level = [&](auto slices) __attribute__((always_inline)) -> int {
                constexpr int S = decltype(slices)::value;   // (S - 1) * 64 < cur_expanded <= S * 64, one at least
                int n[S], f[S], c[S];
                float p[S], w[S];
                bool cand[S];
                c[0] = c0, n[0] = n0, p[0] = p0, w[0] = w0;
#pragma unroll
                for (int i = 1; i < S; ++i) {
                    const int eid = lane + i * kWave;
                    const uint32_t at = row4 + (uint32_t)(i < S - 1 || eid < cur_expanded ? eid : cur_expanded - 1) * 4u;
                    c[i] = *at_bytes(tree_c, at), n[i] = *at_bytes(tree_n, at), p[i] = *at_bytes(tree_p, at), w[i] = *at_bytes(tree_w, at);
                }
                // an edge takes part when it is expanded and leads to a node of the tree; its virtual visits are its
                // child's (the other lanes read the root's counter and drop it)
                int total = 0;
#pragma unroll
                for (int i = 0; i < S; ++i) {
                    cand[i] = (i < S - 1 || lane + i * kWave < cur_expanded) && (uint32_t)c[i] < (uint32_t)node_limit;
                    const int visits = visits_of.peek(cand[i] ? c[i] : 0);
                    f[i] = cand[i] ? visits : 0;
                }
#pragma unroll
                for (int i = 0; i < S; ++i) total += cand[i] ? n[i] + f[i] : 0;
                total = wave_sum(total);
                const int parent_eff = total > 1 ? total : 1;   // :407-416
                const float sqrt_parent = sqrt_of_count(parent_eff);
                if (CONTENDED || a.c_pw != 0.0f) {   // (else there is one child allowed, and there is one)
                    const int allowed = allowed_children(a.c_pw, a.alpha_pw, parent_eff, edges, sqrt_parent);
                    if (allowed > cur_expanded) return expand(allowed);
                }

                // puct_score in two parts: the mean value and the numerator of the exploration term do not depend on the
                // virtual visits, so an evaluation on counters read again divides once per edge, not twice
                float q[S], num[S];
#pragma unroll
                for (int i = 0; i < S; ++i) {
                    // (a slice none of whose edges has a visit or a value has q = +0 without dividing)
                    q[i] = 0.0f;
                    if (__builtin_amdgcn_ballot_w64(n[i] > 0 && __float_as_uint(w[i]) != 0u) != 0) q[i] = n[i] > 0 ? w[i] / (float)n[i] : 0.0f;
                    num[i] = a.cpuct * p[i] * sqrt_parent;
                }
                uint32_t keys[S];
                auto score_slice = [&](int i, int visits) {
                    return cand[i] ? score_key(q[i] + num[i] / (float)(n[i] + visits + 1)) : 0u;
                };
                auto of_edge = [&](const int (&v)[S], int eid) {
                    const int at = eid & (kWave - 1), pass = eid / kWave;
                    int r = __builtin_amdgcn_readlane(v[0], at);
#pragma unroll
                    for (int i = 1; i < S; ++i)
                        if (pass == i) r = __builtin_amdgcn_readlane(v[i], at);
                    return r;
                };
                int best_eid = kNoEdge, held = 0;
                if (PRECLAIM) {
                    // :448-483: claim every candidate, score it with the count found, keep the winner's claim
                    int tie_offset = wid;
                    if (tie_offset >= cur_expanded) tie_offset %= cur_expanded;
#pragma unroll
                    for (int i = 0; i < S; ++i) {
                        int before = 0;
                        if (cand[i]) before = visits_of.add(c[i], 1);
                        keys[i] = score_slice(i, before);
                    }
                    best_eid = best_edge<S>(keys, lane, -1, tie_offset);
#pragma unroll
                    for (int i = 0; i < S; ++i)
                        if (cand[i] && lane + i * kWave != best_eid) visits_of.sub(c[i], 1);
                    held = best_eid != kNoEdge ? 1 : 0;
                } else {
                    // :520-560 with MAX_RECALC_RETRY = 2 written out: the best edge by the counters as read; its child is
                    // claimed; if that child already carried claims and the node has other edges, the claim is given back and
                    // the best of the other edges is claimed and kept whatever it carries (none: the first winner again).
                    // The counters for the second evaluation are requested together with the first claim (just ahead of it, so
                    // that the wait for the claim's result covers them), before it is known whether they will be needed: the
                    // reference reads them after its release, but nothing orders those loads after its relaxed atomics on
                    // other counters, and the first winner's own counter is not among the ones the second evaluation looks at.
                    // one more visit on `child`'s counter, kept unless the counter was negative or full (:329-331): the value found
                    auto claim = [&](int child, int &found) {
                        int v = 0;
                        if (lane == 0) v = visits_of.add(child, 1);
                        found = __builtin_amdgcn_readfirstlane(v);
                        if (found < 0 || found >= INT32_MAX) {
                            if (lane == 0) visits_of.sub(child, 1);
                            return 0;
                        }
                        return 1;
                    };
#pragma unroll
                    for (int i = 0; i < S; ++i) keys[i] = score_slice(i, f[i]);
                    best_eid = best_edge<S>(keys, lane, -1, 0);
                    if (best_eid != kNoEdge) {
                        const int first_child = of_edge(c, best_eid), first_eid = best_eid;
                        const int seen = of_edge(f, first_eid);
                        bool second_round = false;
                        if (seen > 0 && seen < INT32_MAX && cur_expanded > 1) {
                            // The winner's counter already held visits when it was read.  In the execution in which no other
                            // traversal acts between that read and this traversal's claim, the claim finds the same value: a
                            // conflict, upon which the claim is given back and the other edges are evaluated on counters
                            // that are still the ones read (so the scores stand).  That execution is the one taken: nothing is
                            // added to the first winner's counter and nothing taken back.  (A claim that is added and taken back
                            // differs from it only in what other traversals may see in passing, and costs two of the three
                            // atomics and two of the five round trips of a level.)
                            second_round = true;
                        } else {
                            int again[S];
#pragma unroll
                            for (int i = 0; i < S; ++i) {
                                const int visits = visits_of.peek(cand[i] ? c[i] : 0);
                                again[i] = cand[i] ? visits : 0;
                            }
                            int found;
                            if (claim(first_child, found) == 0) {
                                // (the counter cannot be claimed: nothing is held)
                            } else if (found == 0 || cur_expanded <= 1) {
                                held = 1;
                            } else {
                                if (lane == 0) visits_of.sub(first_child, 1);
                                second_round = true;
                                // on the counters read again; other traversals' claims sit on a few edges, so most slices of a
                                // wide node read what they read before and keep their scores
#pragma unroll
                                for (int i = 0; i < S; ++i)
                                    if (S == 1 || __builtin_amdgcn_ballot_w64(again[i] != f[i]) != 0) keys[i] = score_slice(i, again[i]);
                            }
                        }
                        if (second_round) {
                            const int second = best_edge<S>(keys, lane, first_eid, 0);
                            if (second != kNoEdge) best_eid = second;
                            int found2;
                            held = claim(of_edge(c, best_eid), found2);
                        }
                    }
                }
                if (held == 0) return ~kPackedInvalidV2;   // no edge leads anywhere (or the winner's counter cannot be claimed)
                // (only edges that lead to a node of the tree were candidates, so the child is one)
                path.append(depth, (node << 8) | best_eid, lane);
                return of_edge(c, best_eid);
            };

            // Where the traversal goes on, or the complement of its selection word where it ends.
            int next;
            if (__builtin_expect((uint32_t)node_info > (uint32_t)edges, 0)) next = ~(node_info == PUCT_NODE_EXPANDED_TERMINAL ? pack_selection_v2(PUCT_SELECT_TERMINAL, node, 0) : kPackedInvalidV2);
            else if (cur_expanded == 0) next = expand(PRECLAIM ? 1 : allowed_children(a.c_pw, 0.5f, 1, edges, 1.0f));   // (no visits: 1 ** alpha_pw is 1, whatever alpha_pw is)
            else if (cur_expanded <= kWave) next = level(std::integral_constant<int, 1>{});
            else if (cur_expanded <= 2 * kWave) next = level(std::integral_constant<int, 2>{});
            else if (cur_expanded <= 3 * kWave) next = level(std::integral_constant<int, 3>{});
            else next = level(std::integral_constant<int, 4>{});
            // the path buffer is full: stop before reading or claiming anything there
            const bool apart = CONTENDED && cur_expanded > kWave;
            if (!apart && next >= 0 && ++depth >= a.path_depth) next = ~pack_selection_v2(PUCT_SELECT_DEPTH_LIMIT, next, 0);
            if (next < 0) {
                final_packed = ~next;
                break;
            }
            node = next;
            if (apart && ++depth >= a.path_depth) {
                final_packed = pack_selection_v2(PUCT_SELECT_DEPTH_LIMIT, node, 0);
                break;
            }
            row = request(__builtin_amdgcn_readfirstlane(node));
        }
        if (final_packed >> PUCT_PACKED_KIND_SHIFT == PUCT_SELECT_INVALID) rollback_node_path(a, visits_of, path, tree, depth, lane, node_limit);
        else final_len = depth + 1;
        path.finish(depth, lane);
    }
    if (lane == 0) {
        a.out_selected_node[out] = final_packed;
        a.out_path_len[out] = final_len;
    }
}

// ---- backup --------------------------------------------------------------------------------------------------------
struct BackupArgs {
    int virtual_loss;
    const int *edge_child_id;
    float *edge_W;
    int *edge_N;
    int *edge_inflight;
    int *node_inflight;
    int *node_expand_inflight;
    const int *node_count;
    const int *out_selected_node;
    const int *out_path_eids;
    const int *out_path_len;
    const float *path_edge_values;
    int trees, nodes, edges, warps, path_depth;
};

// NODE_LEVEL = true: src/puct/puct_gpu_v2.py:847-927 as written (virtual loss lives in node_inflight[child], the
// selection word has no reason field).  NODE_LEVEL = false: the same conversion of virtual visits into real ones for
// the edge-level virtual loss of select_kernel; BUSY selections hold nothing and are skipped, as in
// src/puct/test_puct_gpu_v3.py:297-302.
// All that a path of up to 64 levels needs is requested at once: a launch of few traversals is as long as its chain of loads,
// which was four long, each asked for when the one before was known to matter (16 trees x 8 traversals 3.5 -> 2.7 us, 1024 x 8
// 4.1 -> 3.8).
struct BackupRequest {
    const int *path;
    const float *values;
    int node_limit, raw, plen, encoded;
    float value;
};
__device__ __forceinline__ BackupRequest request_backup(const BackupArgs &a, int tree, int wid, int lane) {
    const size_t out = (uint64_t)(uint32_t)tree * (uint32_t)a.warps + (uint32_t)wid, first = out * (uint32_t)a.path_depth;
    BackupRequest r;
    r.path = a.out_path_eids + first;
    r.values = a.path_edge_values == nullptr ? nullptr : a.path_edge_values + first;
    r.node_limit = a.node_count[tree], r.raw = a.out_selected_node[out], r.plen = a.out_path_len[out];
    r.encoded = lane < a.path_depth ? r.path[lane] : -1;
    r.value = r.values != nullptr && lane < a.path_depth ? r.values[lane] : 0.0f;
    asm volatile("" ::: "memory");
    return r;
}
template <bool NODE_LEVEL, bool COUNTED = false>
__device__ __forceinline__ void backup_traversal(const BackupArgs &a, LdsInts counted, int tree, int lane, const BackupRequest &request) {
    const int *const path = request.path;
    const float *const values = request.values;
    const int node_limit = request.node_limit, raw = request.raw, plen = request.plen;
    int encoded = request.encoded;
    float value = request.value;
    if (node_limit <= 0 || node_limit > a.nodes || node_limit > PUCT_PACKED_NODE_LIMIT) return;
    if (raw < 0) return;
    const int kind = NODE_LEVEL ? raw >> PUCT_PACKED_KIND_SHIFT : (raw >> PUCT_PACKED_KIND_SHIFT) & PUCT_PACKED_KIND_MASK;
    if (kind == PUCT_SELECT_INVALID) return;
    if (!NODE_LEVEL && kind == PUCT_SELECT_BUSY) return;
    if (plen <= 0) return;

    int edge_count = plen - 1;
    if (edge_count > a.path_depth) edge_count = a.path_depth;
    for (int d = lane; d < edge_count; d += kWave) {
        const int here = encoded;
        const float v = value;
        if (d + kWave < edge_count) {   // (the next 64 levels, on their way meanwhile)
            encoded = path[d + kWave];
            if (values != nullptr) value = values[d + kWave];
        }
        if (here < 0) continue;
        const int parent = here >> 8, slot = here & 0xFF;
        if (parent >= node_limit || slot >= a.edges) continue;
        const size_t e = ((size_t)tree * a.nodes + parent) * a.edges + slot;
        if (COUNTED) {
            __hip_atomic_fetch_add(counted + (parent * a.edges + slot), 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        } else if (NODE_LEVEL) {
            const int child = a.edge_child_id[e];
            if (child >= 0 && child < node_limit)
                atomicSub(&a.node_inflight[(size_t)tree * a.nodes + child], a.virtual_loss);
        } else {
            atomicSub(&a.edge_inflight[e], a.virtual_loss);
        }
        if (values != nullptr) {
            if (!COUNTED) atomicAdd(&a.edge_N[e], 1);
            unsafeAtomicAdd(&a.edge_W[e], v);
        }
    }

    if (lane == 0 && kind == PUCT_SELECT_EXPAND) {
        const int leaf = raw & PUCT_PACKED_NODE_MASK;
        if (leaf < node_limit) atomicSub(&a.node_expand_inflight[(size_t)tree * a.nodes + leaf], 1);
    }
}


}  // namespace puct
