// Kernels and C ABI of PUCT selection and backup with virtual loss (device code: puct_device.hpp).
#include "puct_device.hpp"

namespace {
using namespace puct;

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
    backup_traversal<NODE_LEVEL>(a, nullptr, blockIdx.x, wid, threadIdx.x & (kWave - 1));
}

// The backup of small trees with long paths, whose traversals are wavefronts of this workgroup (grid.y == 1): how often each edge is passed
// is counted in LDS (a.nodes * a.edges words, and at node level a.nodes more), and the edges that were passed, and the nodes that they
// lead to, are then updated in one sweep, an atomic each and lanes side by side, instead of one a level wherever the path leads.  (Values
// are added one by one, in the order in which they come, as before.)  Bound by the lines that the sweep updates: 16384 trees of 65 x 64
// edges with one path of 512 levels, some 0.55 GB in 86 us, where 8.4 M scattered atomics took 324.  Loads and stores in the sweep
// instead of atomics: 100 us, with values 463 instead of 580, but then two launches on the same trees would no longer add up.
template <bool NODE_LEVEL>
__global__ __launch_bounds__(kMaxWavesPerBlock *kWave) void counted_backup_kernel(const BackupArgs a) {
    fetch_arguments(a);
    extern __shared__ int times_passed[];
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), words = a.nodes * a.edges, threads = blockDim.x;
    int *const times_reached = times_passed + words;
    const int node_limit = a.node_count[blockIdx.x];
    for (int i = threadIdx.x; i < words + (NODE_LEVEL ? a.nodes : 0); i += threads) times_passed[i] = 0;
    __syncthreads();
    if (wid < a.warps) backup_traversal<NODE_LEVEL, true>(a, (LdsInts)times_passed, blockIdx.x, wid, threadIdx.x & (kWave - 1));
    __syncthreads();
    const uint64_t first_node = (uint64_t)blockIdx.x * (uint32_t)a.nodes, first = first_node * (uint32_t)a.edges;
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
    // The counters of a tree in LDS: up to 16384 nodes, and a single traversal's only where its path may be long (in memory / in LDS, us a
    // selection and its backup: 256 trees of 2000 x 128, three levels, 8.9 / 13.2; 4096 of 65 x 64, 512 levels, 1329 / 996).
    if (grid.y == 1 && nodes > 0 && nodes <= kLocalVisitNodes && (warps > 1 || nodes <= 16 * (long long)path_depth))
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
    // Counted in LDS where paths can only be that long by coming back to nodes, so that they pass a good part of a small tree's edges, and
    // where there are many of them.  Atomics on scattered words go at 25 G a second, whatever the occupancy, one for a release and
    // three with values.  us, atomics / counted, release and with values: 16384 trees of 65 x 64, paths of 512 324 / 86 and 1043 / 580, of
    // 128 81 / 50 and 255 / 187; of 91 x 90 (512 threads) 316 / 131 and 1038 / 649; of 21 x 20, paths of 64, 39 / 18 and 122 / 71; 2048
    // trees of 65 x 64 with 8 traversals of up to 512 98 / 15 and 309 / 144.  Few trees, which take a few us: 64 of 65 x 64 with one path
    // of 128 4.3 / 6.4, with 8 traversals 4.6 / 5.1.  (Threads, us a release of 16384 x 512 by loads and stores with 64 / 128 / 256 / 512:
    // 65 x 64 179 / 124 / 98 / 116, 91 x 90 627 / 415 / 291 / 213.)
    const long long slots = (long long)a.nodes * a.edges, walked = (long long)a.warps * a.path_depth;
    if (grid.y == 1 && slots > 0 && slots <= kLocalClaimSlots && a.path_depth >= a.nodes && walked * 40 >= slots && a.trees * walked >= 1 << 19) {
        const unsigned threads = slots <= 4608 ? 256 : 512;
        hipLaunchKernelGGL(counted_backup_kernel<NODE_LEVEL>, grid, dim3(block.x < threads ? threads : block.x),
                           sizeof(int) * (size_t)(slots + (NODE_LEVEL ? a.nodes : 0)), stream, a);
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
