// buffer_access.hpp - range-checked 32-bit addressing of a field plane.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace g4 {

// A pass addresses a plane through a buffer resource of the plane's size:
// an access at an offset beyond it reads zero and writes nothing.  Lanes off
// the grid, edge lanes without a neighbour line and cells outside the source
// rectangle take the offset kOut, so the chunk loops carry no divergent
// branches and the loads of the next chunk stay in flight (counted exactly by
// the wait before their use) while the current chunk's recurrence runs.  The
// offsets are 32-bit: a pass that loads and stores the same cells keeps one
// register per address at most, not two.
using Rsrc = __amdgpu_buffer_rsrc_t;
constexpr uint32_t kOut = 0x80000000u;  // past any plane; offset + 16 B does not wrap
constexpr int kRsrcWord3 = 0x00020000;  // gfx9 raw buffer, no format conversion
constexpr int kNT = 2;                  // cache policy: nontemporal

__device__ __forceinline__ Rsrc range_rsrc(const void* p, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, kRsrcWord3);
}
__device__ __forceinline__ Rsrc plane_rsrc(const void* p, int G, int elem_bytes) {
  const uint32_t n = p ? static_cast<uint32_t>(G) * static_cast<uint32_t>(G) * elem_bytes : 0u;
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, static_cast<int>(n), kRsrcWord3);
}
// byte offset of cell (row, col), or kOut when `ok` is false
__device__ __forceinline__ uint32_t cell_off(bool ok, int row, int col, int G, int elem_bytes) {
  return ok ? (static_cast<uint32_t>(row) * G + static_cast<uint32_t>(col)) * elem_bytes : kOut;
}

template <int AUX>
__device__ __forceinline__ float2 bload(Rsrc r, uint32_t off, float2*) {
  const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, AUX);
  float2 o;
  __builtin_memcpy(&o, &v, sizeof(o));
  return o;
}
template <int AUX>
__device__ __forceinline__ double2 bload(Rsrc r, uint32_t off, double2*) {
  const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, AUX);
  double2 o;
  __builtin_memcpy(&o, &v, sizeof(o));
  return o;
}
template <int AUX, class T2>
__device__ __forceinline__ T2 bload(Rsrc r, uint32_t off) {
  return bload<AUX>(r, off, static_cast<T2*>(nullptr));
}
template <int AUX>
__device__ __forceinline__ void bstore(Rsrc r, uint32_t off, float2 v) {
  __attribute__((ext_vector_type(2))) int d;
  __builtin_memcpy(&d, &v, sizeof(d));
  __builtin_amdgcn_raw_buffer_store_b64(d, r, off, 0, AUX);
}
template <int AUX>
__device__ __forceinline__ void bstore(Rsrc r, uint32_t off, double2 v) {
  __attribute__((ext_vector_type(4))) int d;
  __builtin_memcpy(&d, &v, sizeof(d));
  __builtin_amdgcn_raw_buffer_store_b128(d, r, off, 0, AUX);
}

}  // namespace g4
