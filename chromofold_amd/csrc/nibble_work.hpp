// nibble_work.hpp — which workgroup of a one-dimensional launch serves which item of a batch (nibble_kv.hip,
// nibble_mfma.hip).
//
// The items of a batch differ in query tokens and context splits by orders of magnitude (a decode item of one token
// beside a prefill chunk, contexts of 500 and 12,000 tokens). A three-dimensional grid of (most splits) x (most
// tokens) x items launches mostly workgroups that find nothing to do: a batch of 24 decode items and two 16-token
// chunks came to 83,000 workgroups of which 5 % had work. Each launch therefore covers exactly the workgroups its
// items need: item i owns workgroups [first[i], first[i + 1]), and a workgroup finds its item by bisection over the
// prefix sums (scalar loads that hit the scalar cache).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace cfnib {

// Grid of `blocks` workgroups (at most 2^31) of up to 256 threads: a dimension of a launch holds 2^32 work-items, so
// larger grids go on in y, kGridX (a multiple of the 8 XCDs, which take consecutive workgroups in turn) to a row.
constexpr uint32_t kGridX = 1u << 22;
inline dim3 work_grid(uint64_t blocks) {
  if (blocks <= kGridX) return dim3(static_cast<uint32_t>(blocks));
  return dim3(kGridX, static_cast<uint32_t>((blocks + kGridX - 1u) / kGridX));
}
__device__ __forceinline__ uint32_t work_block() { return blockIdx.y * kGridX + blockIdx.x; }  // may be past the last

// The item that owns unit `u` (u < first[items]): the last i with first[i] <= u, which skips items without units.
__device__ __forceinline__ uint32_t work_item(const uint32_t *__restrict__ first, uint32_t items, uint32_t u) {
  uint32_t lo = 0, hi = items;  // first[lo] <= u < first[hi]
  while (hi - lo > 1u) {
    const uint32_t mid = (lo + hi) >> 1;
    if (first[mid] <= u) lo = mid;
    else hi = mid;
  }
  return lo;
}

}  // namespace cfnib
