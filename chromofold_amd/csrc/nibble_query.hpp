// nibble_query.hpp — what the VALU and the MFMA nibble attention kernels share about an item's queries: reading rows of
// any dtype and stride, and which key positions a query sees.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "nibble_kv.hpp"

namespace cfnib {

// Eight elements from byte offsets off[j] + e * es of `base` for every j, all loads in flight before any conversion:
// a test of the type around each load makes the compiler wait for one before the next (32 serial memory latencies in
// the attention prologue, half of that kernel's 19 us on short tails). `packed` (wave-uniform): base and strides are
// multiples of 16 bytes, so contiguous elements can be read 16 bytes at a time.
template <int G>
__device__ inline void load_rows8(float (&x)[G][8], const void *base, uint32_t type, const uint64_t (&off)[G], uint64_t es,
                                  bool packed) {
  const char *p = static_cast<const char *>(base);
  if (type == CF_DEVICE_F32) {
    if (packed && es == 4u) {
#pragma unroll
      for (int j = 0; j < G; ++j) {
        const float4 a = *reinterpret_cast<const float4 *>(p + off[j]), b = *reinterpret_cast<const float4 *>(p + off[j] + 16);
        x[j][0] = a.x; x[j][1] = a.y; x[j][2] = a.z; x[j][3] = a.w;
        x[j][4] = b.x; x[j][5] = b.y; x[j][6] = b.z; x[j][7] = b.w;
      }
      return;
    }
#pragma unroll
    for (int j = 0; j < G; ++j)
#pragma unroll
      for (int e = 0; e < 8; ++e) x[j][e] = *reinterpret_cast<const float *>(p + off[j] + e * es);
    return;
  }
  uint16_t r[G][8];
  if (packed && es == 2u) {
#pragma unroll
    for (int j = 0; j < G; ++j) {
      const uint4 a = *reinterpret_cast<const uint4 *>(p + off[j]);
      const uint32_t w[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
      for (int e = 0; e < 8; ++e) r[j][e] = static_cast<uint16_t>(w[e / 2] >> (16 * (e & 1)));
    }
  } else {
#pragma unroll
    for (int j = 0; j < G; ++j)
#pragma unroll
      for (int e = 0; e < 8; ++e) r[j][e] = *reinterpret_cast<const uint16_t *>(p + off[j] + e * es);
  }
#pragma unroll
  for (int j = 0; j < G; ++j)
#pragma unroll
    for (int e = 0; e < 8; ++e)
      x[j][e] = type == CF_DEVICE_F16 ? static_cast<float>(__builtin_bit_cast(_Float16, r[j][e]))
                                      : __uint_as_float(uint32_t(r[j][e]) << 16);
}

// Visible positions [lo, hi] of query position qpos: p <= q and, with a window, p + window > q; with kOpenWindow
// every p except those with window > 0 and p + window < q.
struct Visible {
  uint32_t lo, hi;
  __device__ bool operator()(uint32_t pos) const { return pos >= lo && pos <= hi; }
};
__device__ inline Visible visible_range(uint32_t qpos, uint32_t window, uint32_t flags) {
  if (flags & kOpenWindow) return {window != 0u && qpos >= window ? qpos - window : 0u, 0xFFFFFFFFu};
  return {window != 0u && qpos >= window ? qpos - window + 1u : 0u, qpos};
}

}  // namespace cfnib
