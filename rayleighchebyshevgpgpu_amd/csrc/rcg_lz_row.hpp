// rcg_lz_row.hpp -- one row of the Lanczos kernels' CSR product.  Compiles for
// the host too (its tests run there).
#pragma once

#include <cmath>
#include <cstdint>

#ifdef __HIPCC__
#define RCG_LZ_FN __host__ __device__ __forceinline__
#else
#define RCG_LZ_FN inline
#endif

namespace rcg {

// (A (x scale))_i, the nonzeros in order.  Eight at a time: their columns and
// values are loaded together, then the gathers, then the FMAs (one at a time, each
// of a row's nonzeros is a trip to memory of its own: n = 17576, 7 nonzeros, with
// a row per thread instead of two, 11.3 -> 8.2 us).  Indices are 64-bit: eight past
// the last nonzeros of an operator of nearly 2^31 would wrap in 32.
template <bool SCALE>
RCG_LZ_FN double lz_row(const int* __restrict__ rowptr, const int* __restrict__ col,
                        const double* __restrict__ val, const double* __restrict__ x, int64_t i,
                        double scale) {
  const int64_t p1 = rowptr[i + 1];
  double a = 0.0;
  for (int64_t p = rowptr[i]; p < p1; p += 8) {
    int j[8];
    double v[8], u[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      j[e] = p + e < p1 ? col[p + e] : 0;
      v[e] = p + e < p1 ? val[p + e] : 0.0;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) u[e] = p + e < p1 ? x[j[e]] : 0.0;
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (p + e < p1) a = fma(v[e], SCALE ? u[e] * scale : u[e], a);
  }
  return a;
}

}  // namespace rcg
