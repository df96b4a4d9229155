// common.hpp -- shared device helpers: wave64 reductions, scoped fences and
// atomics, workspace carving, host error plumbing.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "devmath.hpp"

namespace obvh {

constexpr int kWave = 64;

// Agent-scope relaxed accesses: they go past the XCDs' L2 caches, so what one
// workgroup stores (and waits for, `drain`) before it counts itself done is
// what a workgroup that saw the count loads, without writing back or
// invalidating an L2.
template <class T>
__device__ __forceinline__ T ld_agent(const T* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ void st_agent(T* p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Waits for this wave's stores.
__device__ __forceinline__ void drain() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

__device__ __forceinline__ int lane_id() { return (int)(threadIdx.x & (kWave - 1)); }
__device__ __forceinline__ int wave_id() { return (int)(threadIdx.x / kWave); }

// Butterfly reductions over the 64 lanes (every lane gets the result).
__device__ __forceinline__ float wave_min(float v) {
#pragma unroll
    for (int m = 1; m < kWave; m <<= 1) v = fminf(v, __shfl_xor(v, m, kWave));
    return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int m = 1; m < kWave; m <<= 1) v = fmaxf(v, __shfl_xor(v, m, kWave));
    return v;
}

// Integer min / max over the 64 lanes, result uniform (in every lane).  Four
// DPP steps leave each 16-lane row's result in all of its lanes (xor 1, xor 2,
// half-row mirror, row mirror); the four rows are combined on the scalar
// unit.  Every lane of the wave must be active.
// (mov_dpp with every lane enabled: the compiler folds it into the min / max,
// where update_dpp with an old value cost a move and two wait states more)
template <int kCtrl>
__device__ __forceinline__ int32_t dpp_mov(int32_t v) {
    return __builtin_amdgcn_mov_dpp(v, kCtrl, 0xF, 0xF, true);
}
__device__ __forceinline__ int32_t wave_min_i32(int32_t v) {
    v = min(v, dpp_mov<0xB1>(v));   // quad_perm [1,0,3,2]
    v = min(v, dpp_mov<0x4E>(v));   // quad_perm [2,3,0,1]
    v = min(v, dpp_mov<0x141>(v));  // row_half_mirror
    v = min(v, dpp_mov<0x140>(v));  // row_mirror
    const int32_t a = __builtin_amdgcn_readlane(v, 0), b = __builtin_amdgcn_readlane(v, 16);
    const int32_t c = __builtin_amdgcn_readlane(v, 32), d = __builtin_amdgcn_readlane(v, 48);
    return min(min(a, b), min(c, d));
}
__device__ __forceinline__ int32_t wave_max_i32(int32_t v) {
    v = max(v, dpp_mov<0xB1>(v));
    v = max(v, dpp_mov<0x4E>(v));
    v = max(v, dpp_mov<0x141>(v));
    v = max(v, dpp_mov<0x140>(v));
    const int32_t a = __builtin_amdgcn_readlane(v, 0), b = __builtin_amdgcn_readlane(v, 16);
    const int32_t c = __builtin_amdgcn_readlane(v, 32), d = __builtin_amdgcn_readlane(v, 48);
    return max(max(a, b), max(c, d));
}

// (value, key) lexicographic reductions: smaller value wins (MIN) or larger
// value wins (MAX); equal values (== compare, so -0 == +0) keep the smaller
// key.  Associative and commutative, so the result does not depend on the
// reduction order.
template <bool MIN>
__device__ __forceinline__ bool pair_better(float v, uint32_t k, float ov, uint32_t ok) {
    if (MIN) return (ov < v) || (ov == v && ok < k);
    return (ov > v) || (ov == v && ok < k);
}
// Bump allocator over a caller-provided workspace (256 B aligned pieces).
struct Carver {
    char* base;
    size_t used;
    size_t cap;
    template <class T>
    T* take(size_t count) {
        size_t off = (used + 255) & ~(size_t)255;
        used = off + count * sizeof(T);
        return base ? reinterpret_cast<T*>(base + off) : nullptr;
    }
    bool ok() const { return used <= cap; }
};

}  // namespace obvh

// Host-side error helpers (defined in abi.hip).
void obvh_set_error(const char* msg);
const char* obvh_hip_error(hipError_t e, const char* where);

#define OBVH_HIP_TRY(expr)                                           \
    do {                                                             \
        hipError_t e__ = (expr);                                     \
        if (e__ != hipSuccess) return obvh_hip_error(e__, #expr);    \
    } while (0)
