// Kernels and C ABI of PUCT selection and backup with virtual loss (device code: puct_device.hpp).
#include "puct_device.hpp"

namespace {
using namespace puct;

// Trees of a workgroup of counted_backup_kernel (up to kMaxWavesPerBlock traversals each), a traversal for each of its wavefronts where there are
// many trees.  Where paths are short they share what it costs to start a workgroup with its LDS; where they are long they are counted
// one after the other, which costs more the fewer workgroups there are.
constexpr int kMostCountedTrees = 8;
inline int trees_of_counting_block(int trees, int warps, int threads) {
    const int waves = threads / kWave / warps, spread = trees / 2048, most = waves < kMostCountedTrees ? waves : kMostCountedTrees;
    return spread < 1 || most < 1 ? 1 : spread < most ? spread : most;
}
inline __host__ __device__ int traversals_of_block(int warps) { return warps < kMaxWavesPerBlock ? warps : kMaxWavesPerBlock; }

// Has a launch's arguments read at once: the compiler asks for them where they are used, three waits one after the other (16 trees of
// 257 x 64 edges, 8 traversals, a selection and its backup: 9.7 us, 8.8 with this and with the traversal's own scalar work below).
__device__ __forceinline__ void fetch_arguments(const SelectArgs &a) {
    asm volatile("" ::"s"(a.edge_child_id), "s"(a.edge_prior), "s"(a.edge_W), "s"(a.edge_N), "s"(a.edge_inflight), "s"(a.node_expand_inflight), "s"(a.node_expanded),
                 "s"(a.tree_nodes), "s"(a.out_selected_node), "s"(a.out_path_eids), "s"(a.out_path_len), "s"(a.nodes), "s"(a.edges), "s"(a.warps), "s"(a.path_depth),
                 "s"(a.cpuct), "s"(a.c_pw), "s"(a.alpha_pw), "s"(a.soft_winner));
}
__device__ __forceinline__ void fetch_arguments(const NodeSelectArgs &a) {
    asm volatile("" ::"s"(a.edge_child_id), "s"(a.edge_prior), "s"(a.edge_W), "s"(a.edge_N), "s"(a.node_inflight), "s"(a.node_expand_inflight), "s"(a.node_expanded),
                 "s"(a.node_count), "s"(a.out_selected_node), "s"(a.out_path_eids), "s"(a.out_path_len), "s"(a.nodes), "s"(a.edges), "s"(a.warps), "s"(a.path_depth),
                 "s"(a.cpuct), "s"(a.c_pw), "s"(a.alpha_pw));
}
__device__ __forceinline__ void fetch_arguments(const BackupArgs &a) {
    asm volatile("" ::"s"(a.edge_child_id), "s"(a.edge_W), "s"(a.edge_N), "s"(a.edge_inflight), "s"(a.node_inflight), "s"(a.node_expand_inflight), "s"(a.node_count),
                 "s"(a.out_selected_node), "s"(a.out_path_eids), "s"(a.out_path_len), "s"(a.path_edge_values), "s"(a.virtual_loss), "s"(a.nodes), "s"(a.edges), "s"(a.warps),
                 "s"(a.path_depth));
}

// `words` words by the whole workgroup, eight reads of a lane in flight where there are as many.
__device__ __forceinline__ void copy_words(int *to, const int *from, int words) {
    constexpr int kBatch = 8;
    const int threads = blockDim.x;
    int i = threadIdx.x;
    for (; i + (kBatch - 1) * threads < words; i += kBatch * threads) {
        int v[kBatch];
#pragma unroll
        for (int k = 0; k < kBatch; ++k) v[k] = from[i + k * threads];
#pragma unroll
        for (int k = 0; k < kBatch; ++k) to[i + k * threads] = v[k];
    }
#pragma unroll 1
    for (; i < words; i += threads) to[i] = from[i];
}

// LDS: the tree's traversals are this workgroup's wavefronts (grid.y == 1) and the claims on its edges are kept in
// the workgroup's dynamic LDS for the launch (a.nodes * a.edges words).  OWN: the tree has one traversal.
template <ClaimsIn WHERE>
__global__ __launch_bounds__(kMaxWavesPerBlock *kWave) __attribute__((amdgpu_waves_per_eu(8, 8))) void select_kernel(const SelectArgs a) {
    fetch_arguments(a);
    extern __shared__ int tree_claims[];
    const int wid = __builtin_amdgcn_readfirstlane(blockIdx.y * traversals_of_block(a.warps) + threadIdx.x / kWave);   // the same in all lanes
    constexpr bool LOCAL = WHERE == ClaimsIn::LDS;
    const int words = a.nodes * a.edges;
    int *const in_memory = a.edge_inflight + (uint64_t)blockIdx.x * (uint32_t)a.nodes * (uint32_t)a.edges;
    const EdgeClaims<WHERE> claims{in_memory, (LdsInts)tree_claims};
    if (LOCAL) {
        copy_words(tree_claims, in_memory, words);
        __syncthreads();
    }
    if (LOCAL || wid < a.warps) select_traversal<WHERE>(a, claims, blockIdx.x, wid, threadIdx.x & (kWave - 1));
    if (LOCAL) {
        __syncthreads();
        copy_words(in_memory, tree_claims, words);
    }
}

// LOCAL: the tree's traversals are this workgroup's wavefronts (grid.y == 1) and its virtual-visit counters are kept
// in the workgroup's dynamic LDS for the launch (a.nodes words).
template <bool PRECLAIM, bool LOCAL>
__global__ __launch_bounds__(kMaxWavesPerBlock *kWave) __attribute__((amdgpu_waves_per_eu(8, 8))) void node_select_kernel(const NodeSelectArgs a) {
    fetch_arguments(a);
    extern __shared__ int tree_visits[];
    const int wid = __builtin_amdgcn_readfirstlane(blockIdx.y * traversals_of_block(a.warps) + threadIdx.x / kWave);   // the same in all lanes
    int *const in_memory = a.node_inflight + (uint64_t)blockIdx.x * (uint32_t)a.nodes;
    const NodeVisits<LOCAL> visits_of{in_memory, (LdsInts)tree_visits};
    auto take_visits = [=]() {   // (while the root's row is on its way)
        if (!LOCAL) return;
        copy_words(tree_visits, in_memory, a.nodes);
        __syncthreads();
    };
    if (LOCAL || wid < a.warps) node_select_traversal<PRECLAIM, LOCAL>(a, visits_of, blockIdx.x, wid, threadIdx.x & (kWave - 1), take_visits);
    if (LOCAL && valid_select_shape(a.path_depth, a.nodes, a.edges)) {
        __syncthreads();
        copy_words(in_memory, tree_visits, a.nodes);
    }
}

template <bool NODE_LEVEL>
__global__ __launch_bounds__(kMaxWavesPerBlock *kWave) void backup_kernel(const BackupArgs a) {
    fetch_arguments(a);
    const int wid = __builtin_amdgcn_readfirstlane(blockIdx.y * traversals_of_block(a.warps) + threadIdx.x / kWave);   // the same in all lanes
    if (wid >= a.warps) return;
    const int lane = threadIdx.x & (kWave - 1);
    backup_traversal<NODE_LEVEL>(a, nullptr, blockIdx.x, lane, request_backup(a, blockIdx.x, wid, lane));
}

// Whether a tree's backup is counted (see below): by the levels that its paths have together, which only the device knows.  Both forms take as long at
// some 40 + slots / 85 levels where paths wander evenly over all edges (us a release of 16384 trees, atomics / counted: 65 x 64 with
// paths of 64 levels 37 / 42, of 128 72 / 68; 10 x 9 with 32 9.2 / 11, with 64 15 / 11), and at some 15 + slots / 300 where they keep
// coming back to the same ones, which is what selections do (65 x 64 with 55 levels on average 47 / 23; 10 x 9 with 33 21 / 11).
inline __host__ __device__ bool counting_pays(long long levels, long long slots) { return levels >= 24 + slots / 128; }

// The backup of small trees whose paths may be long, a few trees a workgroup, so that each of its wavefronts has a traversal (grid.y == 1).
// Where a tree's paths are short, its traversals are backed up as by backup_kernel.  Otherwise how often each edge is passed
// is counted in LDS (a.nodes * a.edges words, and at node level a.nodes more), and the edges that were passed, and the nodes that they
// lead to, are then updated in one sweep by the whole workgroup, an atomic each and lanes side by side, instead of one a level wherever the
// path leads.  (Values are added one by one, in the order in which they come, as before.)  Loads and stores in the sweep
// instead of atomics would be faster with values and slower without, but then two launches on the same trees would no longer add up.
template <bool NODE_LEVEL>
__global__ __launch_bounds__(kMaxWavesPerBlock *kWave) void counted_backup_kernel(const BackupArgs a, int at_once) {
    fetch_arguments(a);
    extern __shared__ int times_passed[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x & (kWave - 1);
    const int words = a.nodes * a.edges, threads = blockDim.x;
    const auto tree_at = [&](int k) { return (int)(blockIdx.x + (uint32_t)k * gridDim.x); };   // the workgroup's k-th (neighbours go to neighbours)
    const auto nth_tree = [&](int traversal) {   // (by divisions, and with sums over lanes where a tree has one traversal, a launch on short paths took 8.3 us, not 7.0)
        int n = 0;
#pragma unroll
        for (int k = 1; k <= kMostCountedTrees; ++k) n += traversal >= k * a.warps ? 1 : 0;
        return n;
    };
    const int tree_of_lane = nth_tree(lane), tree_of_wave = nth_tree(wave);
    const bool has_traversal = tree_of_wave < at_once && tree_at(tree_of_wave) < a.trees;
    BackupRequest mine{};
    if (has_traversal) mine = request_backup(a, tree_at(tree_of_wave), wave - tree_of_wave * a.warps, lane);
    int levels = 0;   // of traversal `lane` of the workgroup's
    if (tree_of_lane < at_once && tree_at(tree_of_lane) < a.trees) {
        const int len = a.out_path_len[(uint64_t)(uint32_t)tree_at(tree_of_lane) * (uint32_t)a.warps + (uint32_t)(lane - tree_of_lane * a.warps)];
        const int most = a.path_depth < 1 << 20 ? a.path_depth : 1 << 20;
        levels = len <= 1 ? 0 : len - 1 < most ? len - 1 : most;
    }
    uint32_t counted = 0;   // bit k: the workgroup's k-th tree
    if (a.warps == 1) counted = (uint32_t)__ballot(counting_pays(levels, words));
    else
        for (int k = 0; k < at_once; ++k) counted |= counting_pays(wave_sum(tree_of_lane == k ? levels : 0), words) ? 1u << k : 0u;
    if (has_traversal && !((counted >> tree_of_wave) & 1u)) backup_traversal<NODE_LEVEL>(a, nullptr, tree_at(tree_of_wave), lane, mine);

    int *const times_reached = times_passed + words;
    for (uint32_t rest = counted; rest != 0; rest &= rest - 1) {   // (the same in all wavefronts)
        const int kth = __builtin_ctz(rest), tree = tree_at(kth), node_limit = a.node_count[tree];
        __syncthreads();   // (nobody reads the tree before any more)
        for (int i = threadIdx.x; i < words + (NODE_LEVEL ? a.nodes : 0); i += threads) times_passed[i] = 0;
        __syncthreads();
        if (tree_of_wave == kth) backup_traversal<NODE_LEVEL, true>(a, (LdsInts)times_passed, tree, lane, mine);
        __syncthreads();
        const uint64_t first_node = (uint64_t)(uint32_t)tree * (uint32_t)a.nodes, first = first_node * (uint32_t)a.edges;
        for (int i = threadIdx.x; i < words; i += threads) {
            const int passed = times_passed[i];
            if (passed == 0) continue;
            if (!NODE_LEVEL) {
                atomicAdd(&a.edge_inflight[first + i], (int)(0u - (uint32_t)passed * (uint32_t)a.virtual_loss));
            } else {
                const int child = a.edge_child_id[first + i];
                if (child >= 0 && child < node_limit) __hip_atomic_fetch_add((LdsInts)times_reached + child, passed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
            if (a.path_edge_values != nullptr) atomicAdd(&a.edge_N[first + i], passed);
        }
        if (NODE_LEVEL) {
            __syncthreads();
            for (int c = threadIdx.x; c < a.nodes; c += threads) {
                const int reached = times_reached[c];
                if (reached != 0) atomicAdd(&a.node_inflight[first_node + c], (int)(0u - (uint32_t)reached * (uint32_t)a.virtual_loss));
            }
        }
    }
}

constexpr int kLocalVisitNodes = 16384;   // (what a selection word can name; 64 KB of LDS, two workgroups per CU: still ahead of counters in memory)
constexpr int kLocalClaimSlots = 8192;

// One wavefront per traversal; a tree with more than 16 traversals is spread over several workgroups.
inline void launch_shape(int trees, int warps, dim3 &grid, dim3 &block) {
    const int per_block = warps < kMaxWavesPerBlock ? warps : kMaxWavesPerBlock;
    block = dim3(per_block > 0 ? per_block * kWave : 0);
    grid = dim3(trees > 0 ? trees : 0, per_block > 0 ? (warps + per_block - 1) / per_block : 0);
}

}  // namespace

extern "C" int puct_select_winner_recalc_launch(float cpuct, float c_pw, float alpha_pw, int soft_winner,
                                                const int *edge_child_id, const float *edge_prior, const float *edge_W,
                                                const int *edge_N, int *edge_inflight, int *node_expand_inflight,
                                                const int *node_expanded, const int *tree_nodes,
                                                int *out_selected_node, int *out_path_eids, int *out_path_len, int trees,
                                                int nodes, int edges, int warps, int path_depth, void *stream) {
    SelectArgs a{cpuct,        c_pw,          alpha_pw,        soft_winner,          edge_child_id,
                 edge_prior,   edge_W,        edge_N,          edge_inflight,        node_expand_inflight,
                 node_expanded, tree_nodes,   out_selected_node, out_path_eids,      out_path_len,
                 trees,        nodes,         edges,           warps,                path_depth};
    dim3 grid, block;
    launch_shape(trees, warps, grid, block);
    // A single traversal's claims are plain stores, whatever the size of the tree (plain stores / atomics, us a selection and its backup:
    // 512 trees of 4097 x 64, two levels, 8.9 / 10.4; 64 trees of 1500 x 200 8.6 / 9.5; 512 levels, 16384 trees of 129 x 64 2630 / 3047,
    // 2048 trees of 257 x 256 1790 / 1990).  The claims of a tree with more of them in LDS: up to 8192 edge slots, so that a CU still holds
    // four workgroups.  (In rows of LDS given to the nodes as they are visited, trees of any size: no faster.  16 trees of 257 x 64
    // with 8 traversals 9.9 against 9.5, 1024 of 4097 x 64 18.9 against 17.1: what the claims gain, clearing the rows and adding
    // them up afterwards costs.)  Larger trees go by atomics.
    const long long slots = (long long)nodes * edges;
    const bool small = grid.y == 1 && slots > 0 && slots <= kLocalClaimSlots;
    if (warps == 1)
        hipLaunchKernelGGL(select_kernel<ClaimsIn::OWN>, grid, block, 0, reinterpret_cast<hipStream_t>(stream), a);
    else if (small)
        hipLaunchKernelGGL(select_kernel<ClaimsIn::LDS>, grid, block, sizeof(int) * (size_t)slots, reinterpret_cast<hipStream_t>(stream), a);
    else
        hipLaunchKernelGGL(select_kernel<ClaimsIn::SHARED>, grid, block, 0, reinterpret_cast<hipStream_t>(stream), a);
    return static_cast<int>(hipGetLastError());
}

namespace {
template <bool PRECLAIM>
int launch_node_select(float cpuct, float c_pw, float alpha_pw, const int *edge_child_id, const float *edge_prior,
                       const float *edge_W, const int *edge_N, int *node_inflight, int *node_expand_inflight,
                       const int *node_expanded, const int *node_count, int *out_selected_node, int *out_path_eids,
                       int *out_path_len, int trees, int nodes, int edges, int warps, int path_depth, void *stream) {
    NodeSelectArgs a{cpuct,         c_pw,         alpha_pw,          edge_child_id, edge_prior,   edge_W, edge_N,
                     node_inflight, node_expand_inflight, node_expanded, node_count,    out_selected_node,
                     out_path_eids, out_path_len, trees,             nodes,         edges,        warps,  path_depth};
    dim3 grid, block;
    launch_shape(trees, warps, grid, block);
    // The counters of a tree in LDS: up to 16384 nodes, and a single traversal's where copying them costs little beside reading them in memory at every
    // level that its path may have.  The copy costs by the nodes, a level in memory by its edges, and how long the paths really are the
    // launch does not know: beyond the line, paths of a few levels are two to five times as fast with the counters in memory, and those that
    // fill path_depth up to 1.5 times as slow (before the copy was made eight words at a time they were no slower either).
    // In memory / in LDS, us a preclaim selection and its backup, 64 trees: 700 nodes of 16 edges, 3 levels 8.2 / 9.0, 50 levels 71 / 38;
    // 2000 of 64, 8 levels 14.6 / 13.1, 20 levels 31 / 21; 5000 of 64, 20 levels 31 / 23; 12000 of 64, 50 levels 73 / 49; 5000
    // of 256, 8 levels 31 / 24.  1024 trees: 2000 of 64, 8 levels 16.5 / 15.7, 20 levels 35 / 26; 5000 of 64, 20 levels 35 / 31.
    const long long slices = (edges + kWave - 1) / kWave;
    if (grid.y == 1 && nodes > 0 && nodes <= kLocalVisitNodes && (warps > 1 || nodes <= 200 * slices * path_depth))
        hipLaunchKernelGGL((node_select_kernel<PRECLAIM, true>), grid, block, sizeof(int) * (size_t)nodes, reinterpret_cast<hipStream_t>(stream), a);
    else
        hipLaunchKernelGGL((node_select_kernel<PRECLAIM, false>), grid, block, 0, reinterpret_cast<hipStream_t>(stream), a);
    return static_cast<int>(hipGetLastError());
}
}  // namespace

extern "C" int puct_node_select_preclaim_launch(float cpuct, float c_pw, float alpha_pw, const int *edge_child_id,
                                                const float *edge_prior, const float *edge_W, const int *edge_N,
                                                int *node_inflight, int *node_expand_inflight, const int *node_expanded,
                                                const int *node_count, int *out_selected_node, int *out_path_eids,
                                                int *out_path_len, int trees, int nodes, int edges, int warps,
                                                int path_depth, void *stream) {
    return launch_node_select<true>(cpuct, c_pw, alpha_pw, edge_child_id, edge_prior, edge_W, edge_N, node_inflight,
                                    node_expand_inflight, node_expanded, node_count, out_selected_node, out_path_eids,
                                    out_path_len, trees, nodes, edges, warps, path_depth, stream);
}

extern "C" int puct_node_select_winner_recalc_launch(float cpuct, float c_pw, float alpha_pw, const int *edge_child_id,
                                                     const float *edge_prior, const float *edge_W, const int *edge_N,
                                                     int *node_inflight, int *node_expand_inflight,
                                                     const int *node_expanded, const int *node_count,
                                                     int *out_selected_node, int *out_path_eids, int *out_path_len,
                                                     int trees, int nodes, int edges, int warps, int path_depth,
                                                     void *stream) {
    return launch_node_select<false>(cpuct, c_pw, alpha_pw, edge_child_id, edge_prior, edge_W, edge_N, node_inflight,
                                     node_expand_inflight, node_expanded, node_count, out_selected_node, out_path_eids,
                                     out_path_len, trees, nodes, edges, warps, path_depth, stream);
}

namespace {
template <bool NODE_LEVEL>
int launch_backup(const BackupArgs &a, hipStream_t stream) {
    dim3 grid, block;
    launch_shape(a.trees, a.warps, grid, block);
    // Counted in LDS where paths may be so long that they can only come back to nodes, so that they pass a good part of a small tree's edges, and
    // where there are many of them; whether they are that long the kernel sees for each tree.  Atomics on scattered words go at 25 G a second,
    // whatever the occupancy, one for a release and three with values.  us, atomics / counted, release and with values, paths as
    // selections of recurrent trees leave them: 16384 trees of 65 x 64, paths of 512 368 / 65 and 1140 / 581, of 128 88 / 31 and
    // 281 / 166; of 91 x 90 (512 threads), 512, 364 / 106 and 1183 / 671; of 21 x 20, 64, 47 / 13 and 146 / 76; 2048
    // trees of 65 x 64 with 8 traversals of up to 512 111 / 13 and 347 / 152.  Paths of two levels in the same room: 5.2 / 7.0 with one traversal a
    // tree, whatever the tree, 4.0 / 6.6 with 8 or 16 (when they were counted too, 26 with 65 x 64, 48 with 91 x 90).  Few trees, which
    // take a few us, have nothing to gain: 1030 of 65 x 64 with one path of 64 4.1 / 5.5, of 512 20 / 14.  (Threads, us a release of
    // 16384 x 512 by loads and stores with 64 / 128 / 256 / 512: 65 x 64 179 / 124 / 98 / 116, 91 x 90 627 / 415 / 291 / 213.)
    const long long slots = (long long)a.nodes * a.edges, walked = (long long)a.warps * a.path_depth;
    if (grid.y == 1 && slots > 0 && slots <= kLocalClaimSlots && a.path_depth >= a.nodes && walked * 40 >= slots && counting_pays(walked, slots) && a.trees * walked >= 1 << 19) {
        const unsigned least = slots <= 4608 ? 256 : 512, threads = block.x < least ? least : block.x;
        const int at_once = trees_of_counting_block(a.trees, a.warps, (int)threads);
        hipLaunchKernelGGL(counted_backup_kernel<NODE_LEVEL>, dim3((unsigned)((a.trees - 1) / at_once + 1)), dim3(threads),
                           sizeof(int) * (size_t)(slots + (NODE_LEVEL ? a.nodes : 0)), stream, a, at_once);
    } else {
        hipLaunchKernelGGL(backup_kernel<NODE_LEVEL>, grid, block, 0, stream, a);
    }
    return static_cast<int>(hipGetLastError());
}
}  // namespace

extern "C" const char *puct_cpp_cuda_error_string(int code) { return hipGetErrorString(static_cast<hipError_t>(code)); }

extern "C" int puct_edge_backup_launch(int virtual_loss, float *edge_W, int *edge_N, int *edge_inflight,
                                       int *node_expand_inflight, const int *node_count, const int *out_selected_node,
                                       const int *out_path_eids, const int *out_path_len, const float *path_edge_values,
                                       int trees, int nodes, int edges, int warps, int path_depth, void *stream) {
    BackupArgs a{virtual_loss, nullptr,    edge_W,           edge_N,        edge_inflight, nullptr,
                 node_expand_inflight, node_count, out_selected_node, out_path_eids, out_path_len, path_edge_values,
                 trees,        nodes,      edges,            warps,         path_depth};
    return launch_backup<false>(a, reinterpret_cast<hipStream_t>(stream));
}

extern "C" int puct_node_backup_launch(int virtual_loss, const int *edge_child_id, float *edge_W, int *edge_N,
                                       int *node_inflight, int *node_expand_inflight, const int *node_count,
                                       const int *out_selected_node, const int *out_path_eids, const int *out_path_len,
                                       const float *path_edge_values, int trees, int nodes, int edges, int warps,
                                       int path_depth, void *stream) {
    BackupArgs a{virtual_loss, edge_child_id, edge_W,        edge_N,        nullptr,       node_inflight,
                 node_expand_inflight, node_count, out_selected_node, out_path_eids, out_path_len, path_edge_values,
                 trees,        nodes,         edges,         warps,         path_depth};
    return launch_backup<true>(a, reinterpret_cast<hipStream_t>(stream));
}
