// V consecutive fp32 entries of a row at a time: one 16-byte access (V = 4, aligned) or one element (V = 1, any layout).
#pragma once
#include "common.h"

namespace dlia {

template <int V> struct Unit { float v[V]; };
template <int V> __device__ __forceinline__ Unit<V> ldu(const float* p) {
  Unit<V> u;
  if constexpr (V == 4) {
    const f32x4 t = *reinterpret_cast<const f32x4*>(p);
    u.v[0] = t.x; u.v[1] = t.y; u.v[2] = t.z; u.v[3] = t.w;
  } else {
    u.v[0] = p[0];
  }
  return u;
}
template <int V> __device__ __forceinline__ void stu(float* p, const Unit<V>& u) {
  if constexpr (V == 4) *reinterpret_cast<f32x4*>(p) = f32x4{u.v[0], u.v[1], u.v[2], u.v[3]};
  else p[0] = u.v[0];
}
template <int V> __device__ __forceinline__ void stu(bf16* p, const Unit<V>& u) {
  if constexpr (V == 4) *reinterpret_cast<u32x2*>(p) = u32x2{pack_bf16(u.v[0], u.v[1]), pack_bf16(u.v[2], u.v[3])};
  else p[0] = (bf16)u.v[0];
}

// four entries of a table row (8 or 16 bytes) as fp32
__device__ __forceinline__ Unit<4> ldu4(const float* p) { return ldu<4>(p); }
__device__ __forceinline__ Unit<4> ldu4(const bf16* p) {
  const u32x2 t = *reinterpret_cast<const u32x2*>(p);
  Unit<4> u;
  u.v[0] = bf16_lo(t.x); u.v[1] = bf16_hi(t.x); u.v[2] = bf16_lo(t.y); u.v[3] = bf16_hi(t.y);
  return u;
}

// A row of up to 16384 fp32 entries in the registers of ONE workgroup, 16 bytes (a unit) at a time: thread i holds units i, i + nt,
// ... (NR of them). Rows go through memory once in each direction; a walk of single floats that re-reads what it wrote is three
// serial passes of 16 (width 4096, 256 threads) dependent accesses each, and with a workgroup per row of a decode step that chain,
// not the bytes, is the kernel's time. Steps of few rows take as many threads as there are units (one unit each, one memory
// latency per pass); with many rows (more than `per_cu` threads a CU) the chip is full anyway and 4 units per thread keep the reductions short.
struct RowShape { int threads, nr; };
inline RowShape row_shape(int rows, int H, int per_cu = 1024) {
  const int units = H / 4;
  int threads = 64;
  while (threads < units && threads < 1024) threads <<= 1;
  if (rows > 512 && (long)rows * threads > 256 * per_cu)
    for (threads = 64; threads * 4 < units && threads < 1024;) threads <<= 1;
  return {threads, (units + threads - 1) / threads <= 1 ? 1 : 4};
}
inline bool row_fits(int H) { return H % 4 == 0 && H <= 16384; }
inline bool al16_(const void* p) { return (uintptr_t)p % 16 == 0; }
// (units beyond the row repeat the last one: nothing is masked but what is added up or stored)
template <int NR, typename F>
__device__ __forceinline__ void row_units(int units, F f) {
#pragma unroll
  for (int k = 0; k < NR; ++k) {
    const int u = threadIdx.x + k * blockDim.x;
    f(k, u < units, min(u, units - 1) * 4);
  }
}

}  // namespace dlia
