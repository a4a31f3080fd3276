// cs_wave.hpp -- device helpers shared by the search kernels: accesses to
// wave-private workspace, wave-wide reductions, ordering.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

// 64-bit wave reductions of the device library (declared by HIP only under an
// opt-in macro).
extern "C" __device__ uint32_t __ockl_wfscan_add_u32(uint32_t, bool);
extern "C" __device__ __attribute__((const)) unsigned long long __ockl_wfred_add_u64(unsigned long long);
extern "C" __device__ __attribute__((const)) double __ockl_wfred_add_f64(double);

namespace cs {
namespace {

constexpr uint32_t kXcd = 8;   // XCDs; workgroups are dealt to them round-robin

// Wave-private workspace: only the owning wave reads or writes it, so
// workgroup scope (coherent in the CU's L1 and the XCD's L2) is sufficient.
__device__ __forceinline__ uint64_t ld64(const uint64_t *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ uint32_t ld32(const uint32_t *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ double ldd(const double *p) {
  return __longlong_as_double((long long)ld64(reinterpret_cast<const uint64_t *>(p)));
}
__device__ __forceinline__ void st32(uint32_t *p, uint32_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void st64(uint64_t *p, uint64_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void std_(double *p, double v) {
  st64(reinterpret_cast<uint64_t *>(p), (uint64_t)__double_as_longlong(v));
}
__device__ __forceinline__ uint64_t wmax64(uint64_t *p, uint64_t v) {
  return __hip_atomic_fetch_max(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void wadd_f64(double *p, double v) {
  __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// LDS ring counters (one wave's private row).
__device__ __forceinline__ uint32_t lds_ld(const uint32_t *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void lds_st(uint32_t *p, uint32_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ uint32_t lds_add(uint32_t *p, uint32_t v) {
  return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ uint32_t lds_min(uint32_t *p, uint32_t v) {
  return __hip_atomic_fetch_min(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void lds_or(uint32_t *p, uint32_t v) {
  (void)__hip_atomic_fetch_or(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ uint32_t lds_ld8(const uint8_t *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void lds_st8(uint8_t *p, uint8_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// Results shared by all waves (accumulators): device scope.
__device__ __forceinline__ void gadd_f64(double *p, double v) { unsafeAtomicAdd(p, v); }
// Orders this wave's earlier memory operations before its later ones (all lanes).
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}
__device__ __forceinline__ uint32_t lane_id() { return __lane_id(); }
__device__ __forceinline__ uint32_t rank_below(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}
// Wave-wide reductions over the active lanes (the device library's DPP
// sequences: no LDS round trips), result in every lane.
__device__ __forceinline__ uint32_t wave_sum(uint32_t v) { return __ockl_wfred_add_u32(v); }
__device__ __forceinline__ unsigned long long wave_sum(unsigned long long v) { return __ockl_wfred_add_u64(v); }
__device__ __forceinline__ double wave_sum(double v) { return __ockl_wfred_add_f64(v); }
__device__ __forceinline__ uint32_t uniform(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ uint32_t wave_or(uint32_t v) { return __ockl_wfred_or_u32(v); }

// More forms of the same workspace accesses.
__device__ __forceinline__ float ld_f(const float *p) { return __uint_as_float(ld32(reinterpret_cast<const uint32_t *>(p))); }
__device__ __forceinline__ void st_f(float *p, float v) { st32(reinterpret_cast<uint32_t *>(p), __float_as_uint(v)); }
__device__ __forceinline__ float2 ld_f2(const float2 *p) {
  const uint64_t v = ld64(reinterpret_cast<const uint64_t *>(p));
  return make_float2(__uint_as_float((uint32_t)v), __uint_as_float((uint32_t)(v >> 32)));
}
__device__ __forceinline__ void st_f2(float2 *p, float2 v) {
  st64(reinterpret_cast<uint64_t *>(p), ((uint64_t)__float_as_uint(v.y) << 32) | __float_as_uint(v.x));
}
__device__ __forceinline__ uint32_t ld_u16(const uint16_t *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void st_u16(uint16_t *p, uint16_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

}  // namespace
}  // namespace cs
