// rcg_small.hip -- the whole Chebyshev filter of a small CSR operator in one
// launch.  A translation unit of its own, so that its register-heavy kernels
// cannot change the code generated for the others.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "rcg_internal.hpp"

namespace rcg {
namespace {

// One workgroup owns one column of the block (a complex column: its re and im)
// and runs every step of the recurrence on it; columns never meet in a filter,
// so nothing is exchanged between workgroups.  The column of X_{j-1} lives in
// LDS (double-buffered: one barrier per step), the row's own entries of
// X_{j-1} and X_{j-2} in registers, and so does the operator: thread t holds
// the first NZ nonzeros of rows t, t + NT, .. (kSmallRows of them), so a step
// reads no memory but LDS.  Longer rows read their remaining nonzeros from
// global memory in every step.
//
// What bounds a step is the LDS gather (nnz entries of the column) and the
// barrier, below 1 us, against 4.5 us and a launch for a step of the general
// kernel, which cannot be shorter than a trip to memory.
//
// Nonzeros are summed in the row's order with the arithmetic of csr_rows, and
// absent ones are skipped (not multiplied by zero), so the result is the general
// kernel's bit for bit, infinities and NaN included.
constexpr int kSmallRows = 4;

template <typename T, bool CX, bool SRC, int NT, int NZ>
__global__ __launch_bounds__(NT) void cheb_small_kernel(SmallFilter<T> a) {
  constexpr int R = kSmallRows;
  constexpr int CW = CX ? 2 : 1;
  __shared__ T xs[2][NT * R * CW];
  const int t = threadIdx.x;
  const int n = a.n;
  const int64_t c = (int64_t)blockIdx.x * CW;  // first real column of this workgroup's
  const int64_t ld = a.ld;

  unsigned lens = 0;  // row lengths, a byte each (255: look it up)
  unsigned jp[R][(NZ + 1) / 2];  // column indices, two to a register (n <= 4096)
  T av[R][NZ], ai[CX ? R : 1][NZ];
  // a row's own X_{j-1} and X_{j-2}: in registers too where they fit (2 of the
  // 8 LDS accesses per row of 5 nonzeros), else read back from LDS
  constexpr bool FITS = NT <= 512 || NZ <= 5;
  constexpr bool KEEP = std::is_same<T, float>::value ? FITS || !CX : FITS && !CX;
  T xo[KEEP ? R : 1][CW], zo[KEEP ? R : 1][CW];
  T rs[SRC ? R : 1][CW];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = t + r * NT;
    const int beg = i < n ? a.rowptr[i] : 0;
    const int len = i < n ? a.rowptr[i + 1] - beg : 0;
    lens |= (unsigned)min(len, 255) << (8 * r);
#pragma unroll
    for (int e = 0; e < (NZ + 1) / 2; ++e) jp[r][e] = 0u;
#pragma unroll
    for (int e = 0; e < NZ; ++e) {
      const bool live = e < len;
      const int64_t p = live ? beg + e : 0;
      const unsigned j = live ? (unsigned)a.col[p] : 0u;
      jp[r][e / 2] |= (e & 1) ? j << 16 : j;
      if constexpr (CX) {
        av[r][e] = live ? a.val[2 * p] : T(0);
        ai[r][e] = live ? a.val[2 * p + 1] : T(0);
      } else {
        av[r][e] = live ? a.val[p] : T(0);
      }
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = t + r * NT;
    if (i < n) {
#pragma unroll
      for (int w = 0; w < CW; ++w) {
        const int64_t o = i * ld + c + w;
        if constexpr (SRC) {
          xs[0][i * CW + w] = a.e1[o];
          xs[1][i * CW + w] = a.e0[o];
          rs[r][w] = a.r[o];
        } else {
          xs[0][i * CW + w] = a.x[o];
        }
        if constexpr (KEEP) {
          xo[r][w] = xs[0][i * CW + w];
          zo[r][w] = SRC ? xs[1][i * CW + w] : T(0);
        }
      }
    }
  }
  const T g1 = a.g1, g2 = a.g2;
  const int m = a.m;
  int cur = 0;
  // the correction steps' coefficients, one step ahead of their use
  T kv[CW];
  if constexpr (SRC) {
#pragma unroll
    for (int w = 0; w < CW; ++w) kv[w] = a.kap[2 * ld + c + w];
  }
  __syncthreads();
  for (int j = SRC ? 2 : 1; j <= m; ++j) {
    T kn[CW];
    if constexpr (SRC) {
#pragma unroll
      for (int w = 0; w < CW; ++w) kn[w] = j < m ? a.kap[(int64_t)(j + 1) * ld + c + w] : T(0);
    }
    const T sc = SRC ? T(1) : (m == 1 ? T(0.5) : (j == m ? a.s_end : T(1)));
    const T* __restrict__ x = xs[cur];
    T* y = xs[1 - cur];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int i = t + r * NT;
      if (i >= n) continue;
      const int len = (int)((lens >> (8 * r)) & 255u);
      T acc[CW];
#pragma unroll
      for (int w = 0; w < CW; ++w) acc[w] = T(0);
      T u[NZ][CW];
#pragma unroll
      for (int e = 0; e < NZ; ++e) {
        const unsigned jj = (e & 1) ? jp[r][e / 2] >> 16 : jp[r][e / 2] & 0xffffu;
#pragma unroll
        for (int w = 0; w < CW; ++w) u[e][w] = x[jj * CW + w];
      }
#pragma unroll
      for (int e = 0; e < NZ; ++e) {
        const bool live = e < len;
        if constexpr (CX) {
          T re = fma(av[r][e], u[e][0], acc[0]);
          re = fma(-ai[r][e], u[e][1], re);
          T im = fma(av[r][e], u[e][1], acc[1]);
          im = fma(ai[r][e], u[e][0], im);
          acc[0] = live ? re : acc[0];
          acc[1] = live ? im : acc[1];
        } else {
          const T v = fma(av[r][e], u[e][0], acc[0]);
          acc[0] = live ? v : acc[0];
        }
      }
      if (len > NZ) {
        const int64_t end = a.rowptr[i + 1];
        for (int64_t p = a.rowptr[i] + NZ; p < end; ++p) {
          const int jj = a.col[p];
          if constexpr (CX) {
            const T vr = a.val[2 * p], vi = a.val[2 * p + 1];
            const T ur = x[2 * jj], ui = x[2 * jj + 1];
            acc[0] = fma(vr, ur, acc[0]);
            acc[0] = fma(-vi, ui, acc[0]);
            acc[1] = fma(vr, ui, acc[1]);
            acc[1] = fma(vi, ur, acc[1]);
          } else {
            acc[0] = fma(a.val[p], x[jj], acc[0]);
          }
        }
      }
#pragma unroll
      for (int w = 0; w < CW; ++w) {
        T xi, zi = T(0), o;
        if constexpr (KEEP) {
          xi = xo[r][w];
          zi = zo[r][w];
        } else {
          xi = x[i * CW + w];
          if (SRC || j > 1) zi = y[i * CW + w];
        }
        if constexpr (SRC)
          o = sc * fma(kv[w], rs[r][w], fma(g2, fma(g1, acc[w], xi), -zi));
        else if (j == 1)
          o = sc * (g2 * fma(g1, acc[w], xi));
        else
          o = sc * fma(g2, fma(g1, acc[w], xi), -zi);
        if constexpr (KEEP) {
          zo[r][w] = xi;
          xo[r][w] = o;
        }
        y[i * CW + w] = o;
      }
    }
    cur = 1 - cur;
    if constexpr (SRC) {
#pragma unroll
      for (int w = 0; w < CW; ++w) kv[w] = kn[w];
    }
    __syncthreads();
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = t + r * NT;
    if (i >= n) continue;
#pragma unroll
    for (int w = 0; w < CW; ++w) {
      const int64_t o = i * ld + c + w;
      const T x = xs[cur][i * CW + w];
      if constexpr (SRC) a.v[o] = a.vs_end * fma(a.um[c + w], a.v[o], double(x));
      else a.x[o] = x;
    }
  }
}

template <typename T, bool CX, bool SRC, int NZ>
void small_launch(const SmallFilter<T>& a, int cols, hipStream_t st) {
  // the fewest waves that hold every row: the step's barrier is cheaper
  if (a.n <= 256 * kSmallRows)
    hipLaunchKernelGGL((cheb_small_kernel<T, CX, SRC, 256, NZ>), dim3(cols), dim3(256), 0, st, a);
  else if (a.n <= 512 * kSmallRows)
    hipLaunchKernelGGL((cheb_small_kernel<T, CX, SRC, 512, NZ>), dim3(cols), dim3(512), 0, st, a);
  else if constexpr (!(CX && std::is_same<T, double>::value))
    hipLaunchKernelGGL((cheb_small_kernel<T, CX, SRC, 1024, NZ>), dim3(cols), dim3(1024), 0, st, a);
  else
    throw Error(1, "operator too large for the one-launch filter");
  RCG_HIP(hipGetLastError());
}

}  // namespace

// The rule: every row of the column in one workgroup's LDS and registers
// (n <= 4096; complex128 values take twice the registers: n <= 2048), rows of
// at most 7 nonzeros on average (the registers hold 7; the rest of a longer row
// costs a trip to memory per step) and no row so long that its thread holds up
// the step, at most two rounds of columns over the 256 compute units, and enough
// steps to pay for loading the operator: measured fixed cost above the general
// kernel's and time per step, 12-48 columns, FP64 (us, one launch against
// general): n = 1056 +7 and 0.5 against 5; n = 3904 +15 and 1.2 against 5; 16^3
// +18 and 1.6 against 5.
//
// The mixed filter's correction steps begin one step later, after a launch that the
// FP64 filter does not have, and the general kernel's FP32 steps are the shorter, so
// they need more steps, most of all where two workgroups share a compute unit.  The
// whole call, one launch over general, 96-256 and 272-512 columns: n = 1000 m = 2
// 1.00-1.11 and 1.10-1.17, m = 4 0.70-0.79 and 0.86-0.91; n = 2025 m = 3 1.00 and
// 1.21-1.23, m = 6 0.77-0.80 and 0.92-0.96; n = 3904 m = 5 1.03-1.08 and 1.29-1.35,
// m = 6 0.96-1.00 and 1.22-1.27, m = 17 0.57-0.62 and 0.79-0.83; 4096 rows of 1 to 12
// nonzeros m = 6 0.95-0.98 and 1.24-1.31, m = 17 0.65-0.70 and 0.95-1.03; complex, 64-256
// columns, n = 1600 m = 3 0.95-1.08, m = 5 0.81-0.94; n = 3136 m = 5 1.05-1.13, m = 8
// 0.85-0.93.
bool small_filter_fits(int64_t n, int64_t nnz, int64_t max_row, int64_t cols, int64_t m, bool cx,
                       bool fp32) {
  int64_t least = 2 + n / 1024;
  if (fp32) {
    if (cx) least = 3 + n / 700;
    else if (cols <= 256) least = 3 + n / 1200;
    else least = n <= 2048 ? 3 + n / 650 : 4 + n / 250;
  }
  return n <= (cx && !fp32 ? kSmallFilterRows / 2 : kSmallFilterRows) && m >= least &&
         nnz <= 7 * n && max_row <= 12 && cols <= 512;
}

template <typename T>
void launch_small_filter(const SmallFilter<T>& a, int cols, int64_t max_row, bool cx, hipStream_t st) {
  if (a.n <= 0 || cols <= 0) return;
  static_assert(kSmallFilterRows == 1024 * kSmallRows, "rows one workgroup holds");
  if (a.n > kSmallFilterRows) throw Error(1, "operator too large for the one-launch filter");
  constexpr bool SRC = std::is_same<T, float>::value;
  if (a.m < (SRC ? 2 : 1)) throw Error(1, "one-launch filter: degree too small");
  if (cx) {
    if (max_row <= 5) small_launch<T, true, SRC, 5>(a, cols, st);
    else small_launch<T, true, SRC, 7>(a, cols, st);
  } else {
    if (max_row <= 5) small_launch<T, false, SRC, 5>(a, cols, st);
    else small_launch<T, false, SRC, 7>(a, cols, st);
  }
}
template void launch_small_filter<double>(const SmallFilter<double>&, int, int64_t, bool, hipStream_t);
template void launch_small_filter<float>(const SmallFilter<float>&, int, int64_t, bool, hipStream_t);

}  // namespace rcg
