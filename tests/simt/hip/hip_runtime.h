// What the search kernels use of HIP, on the CPU: each lane of a workgroup runs on a stack of its own and the lanes of a
// wavefront meet at every operation that crosses lanes (simt.cpp).  For tests: the kernels' sources run unchanged, except for
// what tests/simt_build.py rewrites (LDS variables, inline assembly).
#pragma once
#define __HIPCC__ 1
#include <math.h>
#include <stddef.h>
#include <stdint.h>
#include <string.h>
#include <type_traits>

#define __host__
#define __device__
#define __global__
#define __forceinline__ inline
#define __launch_bounds__(...)

namespace simt {
struct Dim3 { int x, y, z; };
struct Where { Dim3 thread, block, block_dim; int lane; };   // of the lane that runs
extern thread_local Where where;
enum Kind { kSync = 1, kBallot, kLane, kShuffle, kDpp, kBarrier, kBarrierAnd };
// All lanes of the wavefront bring a value; returns the 64 of them.
const uint64_t *together(Kind kind, uint64_t mine);
bool barrier(Kind kind, bool mine);     // of the workgroup; whether all brought true
void pause();                           // lets others run
void *dynamic_lds();
int xcc();
inline void together_only() { together(kSync, 0); }
template <class T> inline uint64_t as_bits(T v) { static_assert(sizeof(T) <= 8); uint64_t u = 0; memcpy(&u, &v, sizeof v); return u; }
template <class T> inline T of_bits(uint64_t u) { T v; memcpy(&v, &u, sizeof v); return v; }
template <class T> inline T from(Kind kind, T v, int lane) { return of_bits<T>(together(kind, as_bits(v))[lane & 63]); }
inline uint32_t alignbit(uint32_t hi, uint32_t lo, uint32_t s) { return (uint32_t)((((uint64_t)hi << 32) | lo) >> (s & 31)); }
inline uint32_t bitop3(uint32_t a, uint32_t b, uint32_t c, uint32_t table) {
    uint32_t r = 0;
    for (int i = 0; i < 8; i++) if (table >> i & 1) r |= (i & 4 ? a : ~a) & (i & 2 ? b : ~b) & (i & 1 ? c : ~c);
    return r;
}
inline uint32_t perm(uint32_t s0, uint32_t s1, uint32_t sel) {
    const uint64_t both = ((uint64_t)s0 << 32) | s1;
    uint32_t r = 0;
    for (int i = 0; i < 4; i++) { const uint32_t k = sel >> (8 * i) & 0xff; r |= (k < 8 ? (uint32_t)(both >> (8 * k)) & 0xffu : 0u) << (8 * i); }   // (0x0c: zero)
    return r;
}
inline int dpp(int v, int control) {
    const int l = where.lane, n = control & 15;
    if (control > 0x110 && control < 0x120) { const int o = from(kDpp, v, l >= n ? l - n : l); return (l & 15) >= n ? o : 0; }   // (row_shr)
    return from(kDpp, v, control == 0xB1 ? l ^ 1 : control == 0x4E ? l ^ 2 : (l & ~7) | (7 - (l & 7)));
}
inline uint64_t ballot(bool v) {
    const uint64_t *const all = together(kBallot, v);
    uint64_t r = 0;
    for (int i = 0; i < 64; i++) r |= all[i] << i;
    return r;
}
inline void fence(const char *scope) { if (strcmp(scope, "agent") != 0) together_only(); }
template <class T> inline T load(const T *p, int scope) { if (scope == 2) pause(); return __atomic_load_n(p, __ATOMIC_ACQUIRE); }
template <class T> inline T atomic_max(T *p, T v) { T o = __atomic_load_n(p, __ATOMIC_RELAXED); while (o < v && !__atomic_compare_exchange_n(p, &o, v, false, __ATOMIC_RELAXED, __ATOMIC_RELAXED)); return o; }
template <class T> inline T atomic_min(T *p, T v) { T o = __atomic_load_n(p, __ATOMIC_RELAXED); while (o > v && !__atomic_compare_exchange_n(p, &o, v, false, __ATOMIC_RELAXED, __ATOMIC_RELAXED)); return o; }
inline uint32_t mad24(uint32_t a, uint32_t b, uint32_t c) { return (a & 0xffffffu) * (b & 0xffffffu) + c; }
}  // namespace simt

#define threadIdx simt::where.thread
#define blockIdx simt::where.block
#define blockDim simt::where.block_dim
template <class A, class B> inline std::common_type_t<A, B> min(A a, B b) { using T = std::common_type_t<A, B>; return (T)a < (T)b ? (T)a : (T)b; }
template <class A, class B> inline std::common_type_t<A, B> max(A a, B b) { using T = std::common_type_t<A, B>; return (T)a > (T)b ? (T)a : (T)b; }
inline int __popc(uint32_t v) { return __builtin_popcount(v); }
inline int __popcll(unsigned long long v) { return __builtin_popcountll(v); }
inline int __ffs(int v) { return __builtin_ffs(v); }
inline int __ffsll(long long v) { return __builtin_ffsll(v); }
inline int __clz(int v) { return v ? __builtin_clz((uint32_t)v) : 32; }
inline uint32_t __brev(uint32_t v) { return __builtin_bitreverse32(v); }
inline uint32_t __float_as_uint(float f) { return simt::of_bits<uint32_t>(simt::as_bits(f)); }
inline double __dsqrt_rn(double x) { return sqrt(x); }
inline unsigned long long wall_clock64() { return 0; }
inline unsigned long long __ballot(int v) { return simt::ballot(v != 0); }
template <class T> inline T __shfl(T v, int lane) { return simt::from(simt::kShuffle, v, lane); }
template <class T> inline T __shfl_xor(T v, int x) { return simt::from(simt::kShuffle, v, simt::where.lane ^ x); }
template <class T> inline T __shfl_down(T v, int d) { return simt::from(simt::kShuffle, v, simt::where.lane + d < 64 ? simt::where.lane + d : simt::where.lane); }
inline void __syncthreads() { simt::barrier(simt::kBarrier, true); }
inline int __syncthreads_and(int v) { return simt::barrier(simt::kBarrierAnd, v != 0); }
inline void __threadfence_block() {}
template <class T, class V> inline T atomicAdd(T *p, V v) { return __atomic_fetch_add(p, (T)v, __ATOMIC_RELAXED); }
template <class T, class V> inline T atomicOr(T *p, V v) { return __atomic_fetch_or(p, (T)v, __ATOMIC_RELAXED); }
template <class T, class V> inline T atomicMax(T *p, V v) { return simt::atomic_max(p, (T)v); }
template <class T, class V> inline T atomicMin(T *p, V v) { return simt::atomic_min(p, (T)v); }
template <class T, class V> inline T atomicExch(T *p, V v) { return __atomic_exchange_n(p, (T)v, __ATOMIC_ACQ_REL); }
template <class T, class V> inline T atomicCAS(T *p, V o, V n) { T old = (T)o; __atomic_compare_exchange_n(p, &old, (T)n, false, __ATOMIC_ACQ_REL, __ATOMIC_ACQUIRE); return old; }

// (LDS operations of a wavefront keep their order, and every agent-scope access of these kernels that others wait on comes with
// its fence or wait: all are acquire and release here)
#define __HIP_MEMORY_SCOPE_WORKGROUP 2
#define __HIP_MEMORY_SCOPE_AGENT 3
#define __hip_atomic_load(p, order, scope) simt::load(p, scope)
#define __hip_atomic_store(p, v, order, scope) __atomic_store_n(p, (std::remove_reference_t<decltype(*(p))>)(v), __ATOMIC_RELEASE)
#define __hip_atomic_fetch_add(p, v, order, scope) __atomic_fetch_add(p, v, __ATOMIC_ACQ_REL)
#define __builtin_amdgcn_alignbit(hi, lo, s) simt::alignbit(hi, lo, s)
#define __builtin_amdgcn_bitop3_b32(a, b, c, t) simt::bitop3(a, b, c, t)
#define __builtin_amdgcn_perm(a, b, s) simt::perm(a, b, s)
#define __builtin_amdgcn_ubfe(v, offset, width) (((uint32_t)(v) >> ((offset) & 31u)) & ((1u << ((width) & 31u)) - 1u))
#define __builtin_amdgcn_mbcnt_lo(mask, base) ((base) + (uint32_t)__builtin_popcountll((uint64_t)(uint32_t)(mask) & ((1ull << simt::where.lane) - 1ull)))
#define __builtin_amdgcn_mbcnt_hi(mask, base) ((base) + (uint32_t)__builtin_popcountll(((uint64_t)(uint32_t)(mask) << 32) & ((1ull << simt::where.lane) - 1ull)))
#define __builtin_amdgcn_readfirstlane(v) simt::from(simt::kLane, (int)(v), 0)
#define __builtin_amdgcn_readlane(v, l) simt::from(simt::kLane, (int)(v), l)
#define __builtin_amdgcn_update_dpp(old, v, control, rows, banks, bound) simt::dpp(v, control)
#define __builtin_amdgcn_inverse_ballot_w64(mask) (((mask) >> simt::where.lane & 1ull) != 0)
#define __builtin_amdgcn_fence(order, scope) simt::fence(scope)
#define __builtin_amdgcn_s_getreg(which) ((uint32_t)simt::xcc())
#define __builtin_amdgcn_s_sleep(n) simt::pause()
#define __builtin_amdgcn_s_setprio(n) ((void)0)
#define __builtin_amdgcn_sched_barrier(n) ((void)0)
