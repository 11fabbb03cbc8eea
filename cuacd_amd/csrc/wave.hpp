// wave.hpp - wave64 primitives for gfx950 (CDNA4).
//
// Every kernel in this library is written for 64-lane wavefronts: ballots are
// 64-bit masks, reductions and scans are 6 DPP steps, and a single-wave workgroup
// uses the LDS as wave-private memory with __syncthreads() as its fence.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace cuacd {

template <int AS, class T> using asptr = __attribute__((address_space(AS))) T*;
constexpr int AS_GLOBAL = 1;
constexpr int AS_LDS = 3;

// A generic pointer whose memory is known, so that its accesses compile to
// global or ds instructions: a flat access counts as outstanding in both
// memories, and a wait for one of them waits for everything in flight. (A cut
// of 24k triangles 894 us with its 1,800 flat accesses, 825 us without; a
// 64-mesh decomposition 459 and 425 ms.)
// (Through an integer: a pair of pointer casts would cancel.)
template <class T> __device__ __forceinline__ T* in_hbm(T* p) { return (T*)(asptr<AS_GLOBAL, T>)(uintptr_t)p; }
template <class T> __device__ __forceinline__ T* in_lds(T* p) {
    return (T*)(asptr<AS_LDS, T>)(uint32_t)(uintptr_t)(p);  // the low half of a generic LDS address is the offset
}

constexpr int WAVE = 64;

__device__ __forceinline__ int lane_id() { return __lane_id(); }

// Number of set bits of `mask` below this lane (exclusive prefix of a ballot).
__device__ __forceinline__ int mask_rank(uint64_t mask) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                     __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0));
}

__device__ __forceinline__ uint64_t ballot(bool p) { return __ballot(p); }

template <class T> __device__ __forceinline__ T uniform(T v) {
    return __builtin_amdgcn_readfirstlane(v);
}

__device__ __forceinline__ int read_lane(int v, int l) { return __builtin_amdgcn_readlane(v, l); }
__device__ __forceinline__ double read_lane_d(double v, int l) {
    return __hiloint2double(read_lane(__double2hiint(v), l), read_lane(__double2loint(v), l));
}
__device__ __forceinline__ float read_lane(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// Wave-wide reductions and scans on DPP: four row_shr steps inside the rows of
// 16 lanes, then row_bcast 15 and 31 across them, so lane 63 ends with the
// whole wave's value. Each step is one VALU operation; the same butterfly on
// __shfl_xor goes through the LDS crossbar (ds_bpermute, about 130 cycles a
// step: 64-bit keys cost 12 of them, 0.8k cycles of a hull insertion's 1.2k
// selection). All 64 lanes have to be active. Lanes without a source keep
// `old`. FP64 and FP32 sums stay on the butterfly: their bits depend on the
// order of the additions.
template <int CTRL, int ROWS> __device__ __forceinline__ int dpp_i(int old, int v) {
    return __builtin_amdgcn_update_dpp(old, v, CTRL, ROWS, 0xf, false);
}
constexpr int DPP_SHR1 = 0x111, DPP_SHR2 = 0x112, DPP_SHR4 = 0x114, DPP_SHR8 = 0x118, DPP_BC15 = 0x142, DPP_BC31 = 0x143;

// idempotent operations: a lane without a source combines with itself
template <class Op> __device__ __forceinline__ int wave_reduce_idem(int v, Op op) {
    v = op(v, dpp_i<DPP_SHR1, 0xf>(v, v));
    v = op(v, dpp_i<DPP_SHR2, 0xf>(v, v));
    v = op(v, dpp_i<DPP_SHR4, 0xf>(v, v));
    v = op(v, dpp_i<DPP_SHR8, 0xf>(v, v));
    v = op(v, dpp_i<DPP_BC15, 0xa>(v, v));
    v = op(v, dpp_i<DPP_BC31, 0xc>(v, v));
    return read_lane(v, 63);
}
// 0 is the identity, so each step folds into one v_max_u32 with DPP operand
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
    v = max(v, (uint32_t)dpp_i<DPP_SHR1, 0xf>(0, (int)v));
    v = max(v, (uint32_t)dpp_i<DPP_SHR2, 0xf>(0, (int)v));
    v = max(v, (uint32_t)dpp_i<DPP_SHR4, 0xf>(0, (int)v));
    v = max(v, (uint32_t)dpp_i<DPP_SHR8, 0xf>(0, (int)v));
    v = max(v, (uint32_t)dpp_i<DPP_BC15, 0xa>(0, (int)v));
    v = max(v, (uint32_t)dpp_i<DPP_BC31, 0xc>(0, (int)v));
    return (uint32_t)read_lane((int)v, 63);
}
__device__ __forceinline__ uint32_t wave_min_u32(uint32_t v) {
    return (uint32_t)wave_reduce_idem((int)v, [](int a, int b) { return (int)min((uint32_t)a, (uint32_t)b); });
}
// 64-bit: the high words, then the low words of the lanes that hold the best one
__device__ __forceinline__ uint64_t wave_max_u64(uint64_t v) {
    const uint32_t hi = wave_max_u32((uint32_t)(v >> 32));
    const uint32_t lo = wave_max_u32((uint32_t)(v >> 32) == hi ? (uint32_t)v : 0u);
    return ((uint64_t)hi << 32) | lo;
}
__device__ __forceinline__ uint64_t wave_min_u64(uint64_t v) {
    const uint32_t hi = wave_min_u32((uint32_t)(v >> 32));
    const uint32_t lo = wave_min_u32((uint32_t)(v >> 32) == hi ? (uint32_t)v : ~0u);
    return ((uint64_t)hi << 32) | lo;
}
__device__ __forceinline__ float wave_min_f(float v) {
    return __int_as_float(wave_reduce_idem(
        __float_as_int(v), [](int a, int b) { return __float_as_int(fminf(__int_as_float(a), __int_as_float(b))); }));
}
__device__ __forceinline__ float wave_max_f(float v) {
    return __int_as_float(wave_reduce_idem(
        __float_as_int(v), [](int a, int b) { return __float_as_int(fmaxf(__int_as_float(a), __int_as_float(b))); }));
}
// Inclusive prefix sum across the wave.
__device__ __forceinline__ int wave_incl_scan(int v) {
    v += dpp_i<DPP_SHR1, 0xf>(0, v);
    v += dpp_i<DPP_SHR2, 0xf>(0, v);
    v += dpp_i<DPP_SHR4, 0xf>(0, v);
    v += dpp_i<DPP_SHR8, 0xf>(0, v);
    v += dpp_i<DPP_BC15, 0xa>(0, v);
    v += dpp_i<DPP_BC31, 0xc>(0, v);
    return v;
}
__device__ __forceinline__ int wave_sum_i(int v) { return read_lane(wave_incl_scan(v), 63); }
__device__ __forceinline__ double wave_sum_d(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}
__device__ __forceinline__ float wave_sum_f(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

// Order-preserving float <-> uint mapping (total order incl. negatives).
__device__ __forceinline__ uint32_t fkey(float f) {
    uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// Device-scope atomics used by the heap and the work queues.
template <class T> __device__ __forceinline__ T ld_acquire(T* p) {
    return __hip_atomic_load(p, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T> __device__ __forceinline__ bool cas_acq_rel(T* p, T& expected, T desired) {
    return __hip_atomic_compare_exchange_strong(p, &expected, desired, __ATOMIC_ACQ_REL,
                                                __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T> __device__ __forceinline__ T fetch_add_relaxed(T* p, T v) {
    return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// XCD-aware workgroup order. The dispatcher hands consecutive workgroups of a
// launch to the 8 XCDs in turn; this renumbers workgroup b of nb so that each
// XCD runs groups of G consecutive task slots (groups still go round the XCDs,
// keeping the load spread). Tasks that read the same data (the candidate
// planes of one part) then share one XCD's L2 instead of fetching the data
// into several. A bijection of [0, nb); the last nb mod 8G workgroups keep
// their own index.
__device__ __forceinline__ unsigned xcd_group_slot(unsigned b, unsigned nb, unsigned G) {
    const unsigned span = 8u * G;
    const unsigned full = nb / span * span;
    if (b >= full) return b;
    const unsigned x = b % 8u, j = b / 8u;
    return ((j / G) * 8u + x) * G + (j % G);
}

// err == nullptr: the caller handles the failure itself (nothing recorded)
__device__ __forceinline__ void err_or(int* err, int bits) {
    if (bits && err) __hip_atomic_fetch_or(err, bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace cuacd
