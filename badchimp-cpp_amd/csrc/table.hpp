// Viscosity-table lookup shared by the FP64 and reduced-precision kernels.
#pragma once
#include <hip/hip_runtime.h>

namespace lbamd {

// std::upper_bound over the inner rows sr[1 .. n-2] of a table with its
// constant extension rows 0 and n-1 (libstdc++'s loop), returned as the
// index i with sr[i] <= v < sr[i+1] (LBrheology.h:459-460).
template <typename P, typename T>
__device__ __forceinline__ int table_index(P sr, int n, T v) {
  int first = 1, len = n - 2;
  while (len > 0) {
    const int half = len >> 1, mid = first + half;
    if (v < sr[mid]) {
      len = half;
    } else {
      first = mid + 1;
      len = len - half - 1;
    }
  }
  return first - 1;
}

// Rows of a viscosity table (with its extension) that a step keeps in LDS,
// 4 KB in FP64.  The search is a chain of dependent reads, one per halving, then
// the rows found.  Against the same kernel with the table in global memory
// (40 rows): FP64 200^3 194 us per step for 217, 101x96x90 22.8 for 23.7, FP32S
// 13.0 for 13.4.  Larger tables are read from global memory.
constexpr int kTableLds = 256;

// a table in LDS, as an LDS pointer (a generic one would make its reads flat)
template <typename T>
using LdsPtr = const __attribute__((address_space(3))) T*;
template <typename T>
__device__ __forceinline__ LdsPtr<T> lds_ptr(const T* p) { return (LdsPtr<T>)p; }

// Copies a table of n <= kTableLds rows to LDS (the whole workgroup).
template <typename T>
__device__ __forceinline__ void table_to_lds(const T* __restrict__ sr, const T* __restrict__ nu, int n, T* lds) {
  for (int k = threadIdx.x; k < n; k += blockDim.x) {
    lds[k] = sr[k];
    lds[kTableLds + k] = nu[k];
  }
  __syncthreads();
}

}  // namespace lbamd
