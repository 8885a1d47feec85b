// rcg_kernels.hip -- CDNA4 (gfx950, wave64) kernels of the Rayleigh-Chebyshev solve.
//
// Replaces LanczosCpolyOperatorLMCuda::apply (CPO-LMC:194-265: copy + SpMM +
// subtract per degree), the cuda_kernels.cu ops (scale, substract, normalize,
// residuals; CK:9-382), the cuBLAS projections (LMC:2139-2161, 2200-2222) and
// cuSOLVER QR (LMC:1979-2107) with kernels written for this chip:
//  * csr_block_kernel: one fused three-term Chebyshev step per degree.  A row
//    of the block (ld elements, 16-byte vectors) is owned by G lanes, so each
//    CSR gather is a single contiguous read of that row; launches are remapped
//    so that each XCD's L2 streams a contiguous range of rows.
//  * gram_partial_kernel / tall_gemm_kernel: LDS-tiled tall-skinny products
//    with 4x4 register tiles per thread; partial sums are reduced in a fixed
//    order so results do not depend on scheduling.
//  * column reductions (norms, residuals) and the Lanczos vector kernels.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "rcg_csr_rows.hpp"
#include "rcg_lz_row.hpp"

namespace rcg {
namespace {

template <typename T, int G, int NV, int MODE, int RPI, bool CX>
__global__ __launch_bounds__(kThreads) void csr_block_kernel(
    int64_t n, const int* __restrict__ rowptr, const int* __restrict__ col,
    const T* __restrict__ val, const T* __restrict__ X, const T* Z, T* out, int ld, int ncv,
    int tail, T p0, T p1, T p2, int64_t rows_per_blk, int64_t nblk, const int* __restrict__ order,
    int remap, const T* __restrict__ R, const T* __restrict__ kap, MixedArgs ms) {
  __shared__ int s_rp[kMaxRpb + 1];
  __shared__ int s_col[kStageNz];
  __shared__ T s_val[kStageNz * (CX ? 2 : 1)];
  const int64_t lq = remap ? xcd_remap(blockIdx.x, gridDim.x) : (int64_t)blockIdx.x;
  if (lq >= nblk) return;  // uniform across the workgroup
  const int64_t lb = order ? (int64_t)order[lq] : lq;
  const int64_t i0 = lb * rows_per_blk;
  const int64_t i1 = min(n, i0 + rows_per_blk);
  csr_rows<T, G, NV, MODE, RPI, CX, csr_chunk<T, CX>()>(n, rowptr, col, val, X, Z, out, ld, ncv,
                                                       tail, p0, p1, p2, i0, i1, R, kap, s_rp,
                                                       s_col, s_val, ms);
}

#ifndef RCG_CSR_RPI
#define RCG_CSR_RPI 1
#endif
// lanes per row and vectors per lane for rows of 17-32 16-byte vectors
// (b = 64 FP64, b = 128 FP32)
#ifndef RCG_CSR32_G
#define RCG_CSR32_G 16
#endif
#ifndef RCG_CSR32_NV
#define RCG_CSR32_NV 2
#endif
// and for rows of 9-16 vectors (b = 64 FP32: 8 x 2 with the tuned 16x16 tile
// order 548 us per correction step at 128^3; 16 x 1 655 us, 4 x 4 718 us)
#ifndef RCG_CSR16_G
#define RCG_CSR16_G 8
#endif
#ifndef RCG_CSR16_NV
#define RCG_CSR16_NV 2
#endif


template <typename T, int MODE, bool CX, int G, int NV>
void csr_launch_g(int64_t n, const int* rp, const int* ci, const T* va, const T* X, const T* Z,
                  T* out, int ld, int ncv, int tail, T p0, T p1, T p2, hipStream_t st,
                  const CsrSched* sc, const T* R, const T* kap, const MixedArgs& ms) {
  constexpr int RS = kThreads / G;
  int64_t rows_per_blk, nblk;
  const int* order = nullptr;
  if (sc && sc->order) {
    rows_per_blk = sc->rows_per_blk;
    nblk = sc->nblk;
    order = sc->order;
  } else {
    // ~128-row blocks (their nonzeros fit the LDS stage for stencils) keep
    // the grid >> 256 CUs at large n; small problems use one row pass.
    rows_per_blk = std::min<int64_t>(std::max<int64_t>(RS, 128), kMaxRpb);
    nblk = (n + rows_per_blk - 1) / rows_per_blk;
    if (nblk < 2048) {
      rows_per_blk = RS;
      nblk = (n + rows_per_blk - 1) / rows_per_blk;
    }
  }
  if (rows_per_blk > kMaxRpb) throw Error(1, "CSR row block exceeds the staged row-pointer range");
  const int remap = sc ? sc->remap : 1;
  const int64_t grid = round_up(nblk, kXcds);
  hipLaunchKernelGGL((csr_block_kernel<T, G, NV, MODE, RCG_CSR_RPI, CX>), dim3((unsigned)grid), dim3(kThreads), 0,
                     st, n, rp, ci, va, X, Z, out, ld, ncv, tail, p0, p1, p2, rows_per_blk, nblk, order,
                     remap, R, kap, ms);
  RCG_HIP(hipGetLastError());
}

template <typename T, int MODE, bool CX>
void csr_launch_cx(int64_t n, const int* rp, const int* ci, const T* va, const T* X, const T* Z,
                   T* out, int ld, int ncols, T p0, T p1, T p2, hipStream_t st, const CsrSched* sc,
                   const T* R, const T* kap, const MixedArgs& ms) {
  constexpr int W = V16<T>::W;
  const int ncv = (ncols + W - 1) / W;
  const int tail = ncols - (ncv - 1) * W;
  if (ld % 4 != 0) throw Error(1, "block leading dimension must be a multiple of 4");
#define RCG_CSR_CASE(LIM, GG, NN) \
  if (ncv <= LIM) return csr_launch_g<T, MODE, CX, GG, NN>(n, rp, ci, va, X, Z, out, ld, ncv, tail, p0, p1, p2, st, sc, R, kap, ms);
  // (16-byte vectors per row, lanes per row G, vectors per lane NV).  From 8
  // vectors on, each lane carries two or more vectors: half the lanes per row
  // of one vector each, twice the rows per wave (FP64 step at 128^3, b = 64:
  // 942 -> 867 us; 1024^2 complex, b = 96: 1351 -> 1343 us).  Four vectors
  // per lane from 33 vectors on: the complex64 step at b = 96 (48 vectors),
  // 925 -> 709 us; four per lane at 16-32 vectors and eight at 65-128 were
  // slower.  A column's sum runs over the row's nonzeros in the same
  // order for any (G, NV), so results do not depend on this table.  The
  // batched step (rcg_batch.hip) keeps one vector per lane: the same change
  // there served 1168-1182 against 1181-1186 eigenpairs/s (and, while both
  // kernels shared this file, made the single-operator FP64 step 3% slower).
  // Lane counts that do not divide the workgroup (3, 6, 12, 24 lanes at 3-6,
  // 9-12, 17-24, 65-96 vectors and so on), which the batched step uses, were
  // flat or slower here: 1024^2 complex FP64 solve 29.7 -> 29.7, complex64
  // mixed 33.5 -> 32.3 eigenpairs/s, plain FP64 solves of served requests +1.4%.
  RCG_CSR_CASE(1, 1, 1)
  RCG_CSR_CASE(2, 2, 1)
  RCG_CSR_CASE(4, 4, 1)
  RCG_CSR_CASE(8, 4, 2)
  RCG_CSR_CASE(16, RCG_CSR16_G, RCG_CSR16_NV)
  RCG_CSR_CASE(32, RCG_CSR32_G, RCG_CSR32_NV)
  RCG_CSR_CASE(64, 16, 4)
  RCG_CSR_CASE(128, 32, 4)
  RCG_CSR_CASE(256, 32, 8)
#undef RCG_CSR_CASE
  throw Error(1, "CSR launch without a width class");
}

// ncols counts real columns (2 per complex column when cx).
template <typename T, int MODE>
void csr_launch(int64_t n, const int* rp, const int* ci, const T* va, const T* X, const T* Z,
                T* out, int ld, int ncols, T p0, T p1, T p2, hipStream_t st, const CsrSched* sc,
                const T* R = nullptr, const T* kap = nullptr, bool cx = false,
                const MixedArgs& ms = MixedArgs{}) {
  // the limit of the row kernels' width classes, whichever kernel runs
  if ((ncols + V16<T>::W - 1) / V16<T>::W > 256)
    throw Error(6, "CSR block kernels support at most 256 16-byte column vectors per row");
  if (sc && sc->tile &&
      launch_tile_step<T>(*sc->tile, MODE, va, X, Z, out, ld, ncols, p0, p1, p2, R, kap, cx, ms,
                          st))
    return;
  if (cx) {
    if (ncols % 2 != 0) throw Error(1, "complex blocks have an even number of real columns");
    csr_launch_cx<T, MODE, true>(n, rp, ci, va, X, Z, out, ld, ncols, p0, p1, p2, st, sc, R, kap, ms);
  } else {
    csr_launch_cx<T, MODE, false>(n, rp, ci, va, X, Z, out, ld, ncols, p0, p1, p2, st, sc, R, kap, ms);
  }
}

// ------------------------------------------------------ tall-skinny Gram
// Partial X^H Y over a row range for one 64x64 output tile.
constexpr int kTile = 64;
constexpr int kRb = 32;  // rows staged per LDS round

template <typename T>
__global__ __launch_bounds__(kThreads) void gram_partial_kernel(
    int64_t n, const T* __restrict__ X, int ldx, int bx, const T* __restrict__ Y, int ldy, int by,
    T* __restrict__ P, int64_t rows_per_blk, int ntb) {
  __shared__ T xs[kRb][kTile + 1];
  __shared__ T ys[kRb][kTile + 1];
  const int tile = blockIdx.y;
  const int ta = tile % ((bx + kTile - 1) / kTile);
  const int tb = tile / ((bx + kTile - 1) / kTile);
  const int a0 = ta * kTile;
  const int b0 = tb * kTile;
  const int tx = threadIdx.x % 16;
  const int ty = threadIdx.x / 16;
  const int64_t blk = blockIdx.x;
  const int64_t i0 = blk * rows_per_blk;
  const int64_t i1 = min(n, i0 + rows_per_blk);
  T acc[4][4];
#pragma unroll
  for (int p = 0; p < 4; ++p)
#pragma unroll
    for (int q = 0; q < 4; ++q) acc[p][q] = T(0);
  for (int64_t r0 = i0; r0 < i1; r0 += kRb) {
#pragma unroll
    for (int e = threadIdx.x; e < kRb * kTile; e += kThreads) {
      const int rr = e / kTile;
      const int cc = e % kTile;
      const int64_t i = r0 + rr;
      const bool rowok = i < i1;
      xs[rr][cc] = (rowok && a0 + cc < bx) ? X[i * ldx + a0 + cc] : T(0);
      ys[rr][cc] = (rowok && b0 + cc < by) ? Y[i * ldy + b0 + cc] : T(0);
    }
    __syncthreads();
#pragma unroll 8
    for (int rr = 0; rr < kRb; ++rr) {
      T xa[4], yb[4];
#pragma unroll
      for (int p = 0; p < 4; ++p) xa[p] = xs[rr][tx * 4 + p];
#pragma unroll
      for (int q = 0; q < 4; ++q) yb[q] = ys[rr][ty * 4 + q];
#pragma unroll
      for (int p = 0; p < 4; ++p)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[p][q] = fma(xa[p], yb[q], acc[p][q]);
    }
    __syncthreads();
  }
  T* Pb = P + blk * (int64_t)bx * by;
#pragma unroll
  for (int p = 0; p < 4; ++p)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int a = a0 + tx * 4 + p;
      const int b = b0 + ty * 4 + q;
      if (a < bx && b < by) Pb[a + (int64_t)b * bx] = acc[p][q];
    }
}

// out[o] = sum_b P[b*m + o].  A workgroup owns 64 outputs; its 4 waves take
// the partial blocks b = s (mod 4) with four interleaved accumulators each and
// are combined in a fixed order, so the result does not depend on scheduling.
template <typename T, typename TO>
__global__ __launch_bounds__(kThreads) void reduce_partials_kernel(const T* __restrict__ P,
                                                                   int64_t nblk, int64_t m,
                                                                   TO* __restrict__ out) {
  __shared__ T red[4][64];
  const int ol = threadIdx.x % 64;
  const int sl = threadIdx.x / 64;
  const int64_t o = blockIdx.x * (int64_t)64 + ol;
  T a0 = T(0), a1 = T(0), a2 = T(0), a3 = T(0);
  if (o < m) {
    int64_t b = sl;
    // four rounds' loads in flight, added in the order of the one-round loop
    for (; b + 60 < nblk; b += 64) {
      T x[16];
#pragma unroll
      for (int k = 0; k < 16; ++k) x[k] = P[(b + 4 * k) * m + o];
#pragma unroll
      for (int k = 0; k < 16; k += 4) {
        a0 += x[k];
        a1 += x[k + 1];
        a2 += x[k + 2];
        a3 += x[k + 3];
      }
    }
    for (; b + 12 < nblk; b += 16) {
      a0 += P[b * m + o];
      a1 += P[(b + 4) * m + o];
      a2 += P[(b + 8) * m + o];
      a3 += P[(b + 12) * m + o];
    }
    for (; b < nblk; b += 4) a0 += P[b * m + o];
  }
  red[sl][ol] = (a0 + a1) + (a2 + a3);
  __syncthreads();
  if (sl == 0 && o < m) out[o] = TO((red[0][ol] + red[1][ol]) + (red[2][ol] + red[3][ol]));
}

// The partial sums of a b x b Gram matrix (b <= B) and its Cholesky factor, in one
// workgroup: G = R^T R of the matrix scaled to unit diagonal, C = D R^{-1} (b x b
// column-major; V C is orthonormal), so that a CholQR pass needs no trip to the
// host.  *inv2 = ||R^{-1}||_F^2, which bounds the block's condition (one_pass_enough
// in rcg_dense.hpp), or 0 where a pivot is not positive; C is then the identity.
//
// One wave factors, without a barrier: lane c < 32 holds column c of the trailing
// matrix, lane 32 + c column c of M = R^{-T} (the same eliminations applied to the
// identity), and row j reaches every lane by lane reads.  A version with the
// matrix in LDS and three barriers per column took 13 us at 16 columns and 23 at
// 24, more than the host's factor with its wait and copies (21).
constexpr int kCholMax = 32;
constexpr int kCholThreads = 1024;
__device__ __forceinline__ double lane_of(double v, int l) {
  const long long b = __double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(b & 0xffffffffll), l);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), l);
  return __longlong_as_double(((long long)hi << 32) | lo);
}
// 1/sqrt(d), d > 0 and normal: the hardware's estimate and three Newton steps
// (it sits in the factor's serial chain; sqrt and divide take four times as long)
__device__ __forceinline__ double rsqrt_newton(double d) {
  double r = __builtin_amdgcn_rsq(d);
#pragma unroll
  for (int k = 0; k < 3; ++k) r = fma(r * 0.5, fma(-d * r, r, 1.0), r);
  return r;
}
template <int B>
__global__ __launch_bounds__(kCholThreads) void reduce_chol_kernel(const double* __restrict__ P,
                                                                   int64_t nblk, int b,
                                                                   double* __restrict__ C,
                                                                   double* inv2) {
  constexpr int NO = (B * B + 255) / 256;  // outputs per thread
  constexpr int NU = B <= 24 ? 8 : 4;      // partials of each in flight
  __shared__ double part[4][NO * 256];
  const int m = b * b;
  {
    const int t = threadIdx.x % 256;
    const int sl = threadIdx.x / 256;
    double s[NO];
#pragma unroll
    for (int k = 0; k < NO; ++k) s[k] = 0.0;
    for (int64_t q = sl; q < nblk; q += 4 * NU) {
      double x[NO][NU];
#pragma unroll
      for (int k = 0; k < NO; ++k)
#pragma unroll
        for (int u = 0; u < NU; ++u) {
          const int64_t blk = q + 4 * u;
          x[k][u] = (blk < nblk && t + 256 * k < m) ? P[blk * m + t + 256 * k] : 0.0;
        }
#pragma unroll
      for (int k = 0; k < NO; ++k)
#pragma unroll
        for (int u = 0; u < NU; ++u) s[k] += x[k][u];
    }
#pragma unroll
    for (int k = 0; k < NO; ++k) part[sl][t + 256 * k] = s[k];
  }
  __syncthreads();
  if (threadIdx.x >= 64) return;
  const int lane = threadIdx.x;
  const bool right = lane >= 32;  // a column of M
  const int c = lane & 31;
  auto g = [&](int i, int k) {
    const int e = i + k * b;
    return (part[0][e] + part[1][e]) + (part[2][e] + part[3][e]);
  };
  double dg = 1.0;
  if (c < b) {
    const double d = g(c, c);
    dg = (d > 0.0 && isfinite(d)) ? 1.0 / sqrt(d) : 1.0;
  }
  double a[B];
#pragma unroll
  for (int i = 0; i < B; ++i) {
    const double di = lane_of(dg, i);
    a[i] = i == c ? 1.0 : 0.0;
    if (!right && i < b && c < b) a[i] = g(i, c) * (di * dg);
  }
  bool ok = true;
  double sum = 0.0;  // |column c of M|^2
#pragma unroll
  for (int j = 0; j < B; ++j) {
    const double d = lane_of(a[j], j);
    // unit diagonal before elimination: a pivot below 1e-200 is no pivot
    const bool fine = d > 1e-200 && isfinite(d);
    ok = ok && fine;
    a[j] *= rsqrt_newton(fine ? d : 1.0);
    sum = fma(a[j], a[j], sum);
#pragma unroll
    for (int i = j + 1; i < B; ++i) a[i] = fma(-lane_of(a[j], i), a[j], a[i]);
  }
  if (right && c < b) {
    // R^{-1}[c][k] = M[k][c], zero below the diagonal
#pragma unroll
    for (int k = 0; k < B; ++k)
      if (k < b) C[c + k * b] = ok ? (c <= k ? a[k] * dg : 0.0) : (c == k ? 1.0 : 0.0);
  }
  sum = right && c < b ? sum : 0.0;
#pragma unroll
  for (int h = 16; h > 0; h /= 2) sum += __shfl_xor(sum, h);
  if (lane == 32) *inv2 = ok ? sum : 0.0;
}

inline unsigned reduce_grid(int64_t m) { return (unsigned)((m + 63) / 64); }

template <typename T>
int64_t gram_blocks(int64_t n, int bx, int by, int64_t* rows_per_blk) {
  const int ntiles = ((bx + kTile - 1) / kTile) * ((by + kTile - 1) / kTile);
  // row blocks: 1024 over the tiles, 512 from 2^20 rows (half the partials to
  // write and reduce: the 128^3 x 64 FP64 solve 1977 -> 1967 ms; 256: 1973 ms)
  const int64_t blocks = n >= (int64_t(1) << 20) ? 512 : 1024;
  int64_t target = std::max<int64_t>(1, blocks / ntiles);
  int64_t rpb = round_up((n + target - 1) / target, kRb);
  // at least 4 rows per output column, so a block's bx x by partial is at
  // most a quarter of the rows it reads (small n would otherwise write about
  // as many partial bytes as it reads), and at least 256 rows: the small
  // operators of a served stream (n ~ 1e4) then launch tens of workgroups with
  // fewer partials to reduce (served throughput +4%; 512 and 1024 were slower)
  rpb = std::max<int64_t>(rpb, round_up(4 * (int64_t)std::max(bx, by), kRb));
  rpb = std::max<int64_t>(rpb, 256);
  *rows_per_blk = rpb;
  return (n + rpb - 1) / rpb;
}

// -------------------------------------------------------- tall x small GEMM
template <typename T>
__global__ __launch_bounds__(kThreads) void tall_gemm_kernel(
    int64_t n, const T* __restrict__ X, int ldx, int bx, const T* __restrict__ C, int ldc, int by,
    T alpha, T beta, const T* Z, T* out, int ldo, int64_t nrb) {
  constexpr int KC = 16;
  __shared__ T xs[kTile][KC + 1];
  __shared__ T cs[KC][kTile + 1];
  const int64_t rb = xcd_remap(blockIdx.x, gridDim.x);
  if (rb >= nrb) return;
  const int c0 = blockIdx.y * kTile;
  const int tc = threadIdx.x % 16;
  const int tr = threadIdx.x / 16;
  const int64_t i0 = rb * kTile;
  T acc[4][4];
#pragma unroll
  for (int p = 0; p < 4; ++p)
#pragma unroll
    for (int q = 0; q < 4; ++q) acc[p][q] = T(0);
  for (int k0 = 0; k0 < bx; k0 += KC) {
    for (int e = threadIdx.x; e < kTile * KC; e += kThreads) {
      const int rr = e / KC;
      const int kk = e % KC;
      const int64_t i = i0 + rr;
      xs[rr][kk] = (i < n && k0 + kk < bx) ? X[i * ldx + k0 + kk] : T(0);
    }
    for (int e = threadIdx.x; e < KC * kTile; e += kThreads) {
      const int kk = e / kTile;
      const int cc = e % kTile;
      cs[kk][cc] = (k0 + kk < bx && c0 + cc < by) ? C[(k0 + kk) + (int64_t)(c0 + cc) * ldc] : T(0);
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < KC; ++kk) {
      T xr[4], cr[4];
#pragma unroll
      for (int p = 0; p < 4; ++p) xr[p] = xs[tr * 4 + p][kk];
#pragma unroll
      for (int q = 0; q < 4; ++q) cr[q] = cs[kk][tc * 4 + q];
#pragma unroll
      for (int p = 0; p < 4; ++p)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[p][q] = fma(xr[p], cr[q], acc[p][q]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const int64_t i = i0 + tr * 4 + p;
    if (i >= n) continue;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = c0 + tc * 4 + q;
      if (c >= by) continue;
      const int64_t off = i * ldo + c;
      T v = alpha * acc[p][q];
      if (beta != T(0)) v = fma(beta, Z[off], v);
      out[off] = v;
    }
  }
}

// ---------------------------------------------------- FP64 MFMA versions
// v_mfma_f64_16x16x4f64 computes D(16x16) += A(16x4) B(4x16); lane l supplies
// A[l%16][l/16] and B[l/16][l%16] and holds D[4j + l/16][l%16] in register j.
typedef double d4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ d4v mfma16x16x4(double a, double b, d4v c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Which tile column lane cc of a 16x16 subtile t holds.  With an even number
// of subtiles the columns are taken in pairs: lane cc reads columns 2cc and
// 2cc+1 of each 32-column half with one 16-byte load, subtile 2h holding the
// even and 2h+1 the odd ones; otherwise subtile t holds columns 16t..16t+15.
// The output tile is the same sums with its rows and columns permuted.
template <int NT>
__device__ __forceinline__ int gram_col(int t, int cc) {
  if constexpr (NT % 2 == 0) return 32 * (t >> 1) + 2 * cc + (t & 1);
  return 16 * t + cc;
}
// the subtile that holds tile column c (the inverse of gram_col)
template <int NT>
__device__ __forceinline__ int gram_sub(int c) {
  if constexpr (NT % 2 == 0) return 2 * (c >> 5) + (c & 1);
  return c >> 4;
}

// Partial X^T Y of one 64x64 output tile over a row range.  Wave w takes the
// 4-row groups i0 + 4w + 16t; lane (kr = l/16, cc = l%16) loads row row+kr of
// X at the tile columns gram_col(p, cc) and of Y at gram_col(q, cc), which are
// the A and B fragments of the NT x NT MFMA subtiles (16-byte loads of column
// pairs when NT is even, 128-byte row segments across the 16 lanes either
// way).  A wave's rows and the order it sums them in do not depend on the
// column order, so every entry is the same sum as with 8-byte loads.  DIAG (a
// tile on the diagonal of X^T X) multiplies only subtiles p <= q and needs
// no Y loads.
template <bool DIAG, int NT>
__device__ __forceinline__ void gram_tile_accumulate(d4v (&acc)[NT][NT], const double* __restrict__ X,
                                                     int ldx, int bx, const double* __restrict__ Y,
                                                     int ldy, int by, int a0, int b0, int64_t ib,
                                                     int64_t i1, int kr, int cc) {
  // U 16-row groups per pass: all of their loads are issued before the MFMAs
  // that consume them, and the next pass's loads before this pass's MFMAs.
  // A wave's rows and the order it sums them in do not depend on U.  Two
  // groups at NT = 3 (142 instead of 198 VGPRs for X^T Y: served stream
  // 1602 -> 1611 eigenpairs/s); at NT = 4 two groups made the 128^3 x 64
  // solve 1975 -> 1989 ms.
  constexpr int U = NT == 3 ? 2 : 4;
  double xa[U][NT], yb[U][NT], xn[U][NT], yn[U][NT];
  auto row_load = [&](const double* __restrict__ B, int ldb, int bw, int c0, int64_t row, bool ok,
                      double (&v)[NT]) {
    if constexpr (NT % 2 == 0) {
#pragma unroll
      for (int h = 0; h < NT / 2; ++h) {
        const int c = c0 + gram_col<NT>(2 * h, cc);
        v[2 * h] = (ok && c < bw) ? B[row * ldb + c] : 0.0;
        v[2 * h + 1] = (ok && c + 1 < bw) ? B[row * ldb + c + 1] : 0.0;
      }
    } else {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int c = c0 + gram_col<NT>(t, cc);
        v[t] = (ok && c < bw) ? B[row * ldb + c] : 0.0;
      }
    }
  };
  auto load = [&](int64_t jb, double (&xv)[U][NT], double (&yv)[U][NT]) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t row = jb + 16 * u + kr;
      const bool ok = row < i1;
      row_load(X, ldx, bx, a0, row, ok, xv[u]);
      if constexpr (!DIAG) row_load(Y, ldy, by, b0, row, ok, yv[u]);
    }
  };
  // Without guards: lanes past the last column (pair) load that one, which
  // reaches no output; an odd block's last column is the second of its pair.  A
  // block of one column is the first of a pair with the row's padding.
  typedef double pair __attribute__((ext_vector_type(2), aligned(8)));
  auto row_full = [&](const double* __restrict__ B, int ldb, int bw, int c0, int64_t row,
                      double (&v)[NT]) {
    if constexpr (NT % 2 == 0) {
#pragma unroll
      for (int h = 0; h < NT / 2; ++h) {
        const int c = c0 + gram_col<NT>(2 * h, cc);
        const pair t = *reinterpret_cast<const pair*>(B + row * ldb + max(0, min(c, bw - 2)));
        v[2 * h] = t[0];
        v[2 * h + 1] = t[1];
      }
    } else {
#pragma unroll
      for (int t = 0; t < NT; ++t)
        v[t] = B[row * ldb + min(c0 + gram_col<NT>(t, cc), bw - 1)];
    }
  };
  auto load_full = [&](int64_t jb, double (&xv)[U][NT], double (&yv)[U][NT]) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t row = jb + 16 * u + kr;
      row_full(X, ldx, bx, a0, row, xv[u]);
      if constexpr (!DIAG) row_full(Y, ldy, by, b0, row, yv[u]);
    }
  };
  bool sx[NT], sy[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    sx[t] = NT % 2 == 0 && bx > 1 && a0 + gram_col<NT>(t, cc) == bx - 1;
    sy[t] = NT % 2 == 0 && by > 1 && b0 + gram_col<NT>(t, cc) == by - 1;
  }
  auto mul = [&](const double (&xv)[U][NT], const double (&yv)[U][NT], bool shift) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      double xs[NT], ys[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        xs[t] = (t % 2 == 0 && shift && sx[t]) ? xv[u][(t + 1) % NT] : xv[u][t];
        if constexpr (!DIAG) ys[t] = (t % 2 == 0 && shift && sy[t]) ? yv[u][(t + 1) % NT] : yv[u][t];
      }
#pragma unroll
      for (int p = 0; p < NT; ++p)
#pragma unroll
        for (int q = 0; q < NT; ++q) {
          if (DIAG && p > q) continue;
          acc[p][q] = mfma16x16x4(xs[p], DIAG ? xs[q] : ys[q], acc[p][q]);
        }
    }
  };
  // Whole passes, the next one's loads in flight during a pass's MFMAs: with guards
  // the compiler waits for every load in flight before a set is used (X^T Y at
  // 128^3 x 64 511 -> 384 us, 5.6 TB/s; X^T X 280 -> 245; the pair of them at
  // 17576 x 24 13.2 -> 10.0).
  const int64_t last = i1 - ib - 16 * (U - 1) - 4;
  const bool any = last >= 0 && (NT % 2 != 0 || (ldx > 1 && (DIAG || ldy > 1)));
  const int np = __builtin_amdgcn_readfirstlane(any ? (int)(last / (16 * U)) + 1 : 0);
  if (np > 0) {
    load_full(ib, xa, yb);
    int k = 0;
    for (; k + 2 < np; k += 2) {
      load_full(ib + (k + 1) * (16 * U), xn, yn);
      mul(xa, yb, true);
      load_full(ib + (k + 2) * (16 * U), xa, yb);
      mul(xn, yn, true);
    }
    if (k + 1 < np) {
      load_full(ib + (k + 1) * (16 * U), xn, yn);
      mul(xa, yb, true);
      mul(xn, yn, true);
    } else {
      mul(xa, yb, true);
    }
    ib += (int64_t)np * (16 * U);
  }
  for (; ib < i1; ib += 16 * U) {
    load(ib, xa, yb);
    mul(xa, yb, false);
  }
}

// Which 64x64 tiles of X^H Y a Gram launch multiplies.  kGramFull: all of
// them.  kGramSym (X == Y): only the tiles ta <= tb of the upper triangle,
// ntiles = nta (nta+1)/2, each written at (a, b) and mirrored at (b, a).
// kGramLower (bx == by, X != Y): the tiles on and below the diagonal, for
// callers that read only the lower triangle of X^H Y (the Hermitian
// projection); the upper tiles get the transposed lower values so that every
// entry of the result is defined.  kGramDiag: the one tile of X^T X when
// bx <= 64.  kGramPair (bx == by <= 64): X^T X and X^T Y in one launch, tile 0
// and tile 1 of each row block, with the partials of both side by side.
enum { kGramFull = 0, kGramSym = 1, kGramDiag = 2, kGramLower = 3, kGramPair = 4 };

// Partial Gram matrices of one 64x64 tile, one bx x by block per row block:
// the one-tile launches (kGramFull with bx, by <= 64, or kGramDiag, compiled
// without the general path so that it keeps two waves per SIMD; kGramPair
// runs either per workgroup).  A row block's partials land at
// P + (rblk * ntiles + tile) * bx * by.  NT = ceil(max(bx, by) / 16): only
// the NT x NT 16x16 subtiles that hold output are multiplied, with registers
// for those alone (the sums of the others were zero).
template <int MODE, int NT>
__global__ __launch_bounds__(kThreads) void gram_mfma_kernel(
    int64_t n, const double* __restrict__ X, int ldx, int bx, const double* __restrict__ Y, int ldy,
    int by, double* __restrict__ P, int64_t rows_per_blk, int nta, int ntiles, int64_t nblk) {
  static_assert(MODE == kGramFull || MODE == kGramDiag || MODE == kGramPair,
                "one-tile launches only");
  __shared__ double red[kTile * kTile];
  // one 1-D grid: the tiles of a row block are consecutive logical workgroups,
  // which the remap keeps on one XCD, so its rows are read from HBM once
  const int64_t L = xcd_remap(blockIdx.x, gridDim.x);
  if (L >= nblk * ntiles) return;
  const int tile = (int)(L % ntiles);
  const int64_t rblk = L / ntiles;
  const int ta = MODE == kGramPair ? 0 : tile % nta;
  const int tb = MODE == kGramPair ? 0 : tile / nta;
  // uniform per workgroup: kGramPair's tile 0 is X^T X
  const bool diag = MODE == kGramDiag || (MODE == kGramPair && tile == 0);
  const int a0 = ta * kTile;
  const int b0 = tb * kTile;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int kr = lane >> 4;
  const int cc = lane & 15;
  const int64_t i0 = rblk * rows_per_blk;
  const int64_t i1 = min(n, i0 + rows_per_blk);
  d4v acc[NT][NT];
#pragma unroll
  for (int p = 0; p < NT; ++p)
#pragma unroll
    for (int q = 0; q < NT; ++q) acc[p][q] = d4v{0.0, 0.0, 0.0, 0.0};
  if constexpr (MODE == kGramPair) {
    if (diag)
      gram_tile_accumulate<true, NT>(acc, X, ldx, bx, X, ldx, bx, a0, b0, i0 + 4 * wave, i1, kr,
                                     cc);
    else
      gram_tile_accumulate<false, NT>(acc, X, ldx, bx, Y, ldy, by, a0, b0, i0 + 4 * wave, i1, kr,
                                      cc);
  } else {
    gram_tile_accumulate<MODE == kGramDiag, NT>(acc, X, ldx, bx, Y, ldy, by, a0, b0,
                                                i0 + 4 * wave, i1, kr, cc);
  }
  // the four waves' tiles are summed in LDS in wave order
  for (int w = 0; w < 4; ++w) {
    if (wave == w) {
#pragma unroll
      for (int p = 0; p < NT; ++p)
#pragma unroll
        for (int q = 0; q < NT; ++q) {
          if (diag && p > q) continue;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int idx = gram_col<NT>(p, 4 * j + kr) + kTile * gram_col<NT>(q, cc);
            red[idx] = (w == 0) ? acc[p][q][j] : red[idx] + acc[p][q][j];
          }
        }
    }
    __syncthreads();
  }
  double* Pb = P + (rblk * (MODE == kGramPair ? ntiles : 1) + (MODE == kGramPair ? tile : 0)) *
                      (int64_t)bx * by;
  for (int e = threadIdx.x; e < kTile * kTile; e += kThreads) {
    const int al = e % kTile;
    const int bl = e / kTile;
    const int a = a0 + al;
    const int b = b0 + bl;
    if (a >= bx || b >= by) continue;
    // a diagonal tile holds the subtiles p <= q; the others are their mirror
    if (diag)
      Pb[a + (int64_t)b * bx] = (gram_sub<NT>(al) <= gram_sub<NT>(bl)) ? red[al + kTile * bl]
                                                                        : red[bl + kTile * al];
    else
      Pb[a + (int64_t)b * bx] = red[al + kTile * bl];
  }
}

// Gram partials for blocks wider than one tile (bx or by > 64), through LDS.
// Each workgroup owns one 64x64 output tile (enumerated as in gram_mfma_kernel)
// and one row block; 32-row chunks of X[:, a0:a0+64] and Y[:, b0:b0+64] are
// loaded as pairs, two chunks ahead, without guards, and staged in double-buffered
// LDS (one barrier per chunk).  FP64 MFMA issue bounds it; with guarded loads one
// chunk ahead and rows padded to 65 entries the waves waited on memory and banks:
// X^T Y at 2^20 x 192 1.75 -> 1.47 ms (44 -> 53 TFLOP/s), X^T X 1.15 -> 0.95; 20000 x
// 256, X^T X, 69 -> 49 us.  Wave w owns the 32x32 quadrant (w & 1, w >> 1) of
// the tile, so no cross-wave reduction is needed; in a diagonal tile of X^T X
// the quadrant below the diagonal is the mirror of the one above and its wave
// idles.  (Each wave multiplying a quarter of every chunk's rows into the
// whole tile, four MFMAs per fragment read instead of one and no idle wave,
// then a sum over the waves in LDS, measured the same at 1024^2 x 192.)  Row
// blocks are sized so that all workgroups are resident at once
// (two or four times as many smaller blocks, so that compute units done with
// the cheaper diagonal tiles take more, gave the same time at 1024^2 x 192: a
// workgroup's time is its chunks' latency, not its compute unit's MFMA load).
constexpr int kGramKr = 32;
template <int MODE>
__global__ __launch_bounds__(kThreads, 2) void gram_lds_kernel(
    int64_t n, const double* __restrict__ X, int ldx, int bx, const double* __restrict__ Y, int ldy,
    int by, double* __restrict__ P, int64_t rows_per_blk, int nta, int ntiles, int64_t nblk) {
  __shared__ __align__(16) double xs[2][kGramKr][kTile];
  __shared__ __align__(16) double ys[2][kGramKr][kTile];
  const int64_t L = xcd_remap(blockIdx.x, gridDim.x);
  if (L >= nblk * ntiles) return;
  const int tile = (int)(L % ntiles);
  const int64_t rblk = L / ntiles;
  int ta, tb;
  if constexpr (MODE != kGramFull) {
    tb = 0;
    while ((tb + 1) * (tb + 2) / 2 <= tile) ++tb;
    ta = tile - tb * (tb + 1) / 2;
    if constexpr (MODE == kGramLower) {
      const int t = ta;
      ta = tb;
      tb = t;
    }
  } else {
    ta = tile % nta;
    tb = tile / nta;
  }
  const bool diag = MODE == kGramSym && ta == tb;
  const int a0 = ta * kTile;
  const int b0 = tb * kTile;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int kr = lane >> 4;
  const int cc = lane & 15;
  const int qa = wave & 1;
  const int qb = wave >> 1;
  const bool idle = diag && qa == 1 && qb == 0;
  const int64_t i0 = rblk * rows_per_blk;
  const int64_t i1 = min(n, i0 + rows_per_blk);
  // thread t moves pairs of columns: chunk rows t / 32 + 8 m, m < 4, columns 2 (t % 32)
  // and 2 (t % 32) + 1 of the tile's 64
  const int er = threadIdx.x / 32, ec = 2 * (threadIdx.x % 32);
  auto ld2 = [&](const double* B, int ldb, int bw, int64_t row, int col) -> dvec2 {
    if (row >= i1) return dvec2{0.0, 0.0};
    const double* ptr = B + row * ldb + col;
    return dvec2{col < bw ? ptr[0] : 0.0, col + 1 < bw ? ptr[1] : 0.0};
  };
  // Without guards: columns past the block's last pair are loaded from that pair (their
  // products reach no output), an odd block's last column as the pair's second, a
  // block's only column as the first of a pair with the row's padding.
  const int cx = max(0, min(a0 + ec, bx - 2)), cy = max(0, min(b0 + ec, by - 2));
  const bool shx = bx > 1 && a0 + ec == bx - 1, shy = by > 1 && b0 + ec == by - 1;
  typedef double pair __attribute__((ext_vector_type(2), aligned(8)));
  d4v acc[2][2];
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int q = 0; q < 2; ++q) acc[p][q] = d4v{0.0, 0.0, 0.0, 0.0};
  const bool dquad = diag && qa == qb;  // quadrant on the diagonal: subtiles p <= q
  // column of a row in LDS: rows of 64 with the halves of each 32 columns exchanged
  // in odd rows, so that a half-wave's fragment (2 rows x 16 columns) covers all
  // banks and a pair is stored by one 16-byte write
  const int swz = 16 * (kr & 1);
  auto run = [&](auto dg) {
    constexpr bool DG = decltype(dg)::value;
    dvec2 sx[2][4], sy[2][4];
    auto fetch_full = [&](int64_t r0, int s) {
      const double* xp = X + (r0 + er) * ldx + cx;
      const double* yp = Y + (r0 + er) * ldy + cy;
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const pair v = *reinterpret_cast<const pair*>(xp + (int64_t)(8 * m) * ldx);
        sx[s][m] = dvec2{v[0], v[1]};
        if constexpr (!DG) {
          const pair w = *reinterpret_cast<const pair*>(yp + (int64_t)(8 * m) * ldy);
          sy[s][m] = dvec2{w[0], w[1]};
        }
      }
    };
    auto put = [&](int buf, int s, bool ox, bool oy) {
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const int rr = er + 8 * m, c = ec ^ (16 * (rr & 1));
        dvec2 v = sx[s][m];
        if (ox) v.x = v.y;
        *reinterpret_cast<dvec2*>(&xs[buf][rr][c]) = v;
        if constexpr (!DG) {
          dvec2 w = sy[s][m];
          if (oy) w.x = w.y;
          *reinterpret_cast<dvec2*>(&ys[buf][rr][c]) = w;
        }
      }
    };
    auto chunk = [&](int buf) {
      if (DG && idle) return;
      const double(*yb)[kTile] = DG ? xs[buf] : ys[buf];
#pragma unroll
      for (int k4 = 0; k4 < kGramKr; k4 += 4) {
        const int kk = k4 + kr;
        double af[2], bf[2];
#pragma unroll
        for (int p = 0; p < 2; ++p) af[p] = xs[buf][kk][32 * qa + ((16 * p + cc) ^ swz)];
#pragma unroll
        for (int q = 0; q < 2; ++q) bf[q] = yb[kk][32 * qb + ((16 * q + cc) ^ swz)];
        acc[0][0] = mfma16x16x4(af[0], bf[0], acc[0][0]);
        acc[0][1] = mfma16x16x4(af[0], bf[1], acc[0][1]);
        if (!DG || !dquad) acc[1][0] = mfma16x16x4(af[1], bf[0], acc[1][0]);
        acc[1][1] = mfma16x16x4(af[1], bf[1], acc[1][1]);
      }
    };
    // whole chunks, loaded two ahead into register set c % 2 with no branch between
    // a set's loads and its stores (with one the compiler waits for all loads in flight)
    const int64_t nf = ldx > 1 && ldy > 1 ? (i1 - i0) / kGramKr : 0;
    int64_t done = i0;
    if (nf >= 4) {
      fetch_full(i0, 0);
      put(0, 0, shx, shy);
      fetch_full(i0 + kGramKr, 1);
      __syncthreads();
      int64_t c = 0;
      for (; c + 3 < nf; c += 2) {
        fetch_full(i0 + (c + 2) * kGramKr, 0);
        chunk(0);
        put(1, 1, shx, shy);
        __syncthreads();
        fetch_full(i0 + (c + 3) * kGramKr, 1);
        chunk(1);
        put(0, 0, shx, shy);
        __syncthreads();
      }
      const bool three = c + 2 < nf;
      if (three) fetch_full(i0 + (c + 2) * kGramKr, 0);
      chunk(0);
      put(1, 1, shx, shy);
      __syncthreads();
      chunk(1);
      if (three) {
        put(0, 0, shx, shy);
        __syncthreads();
        chunk(0);
      }
      done = i0 + nf * kGramKr;
    }
    for (int64_t r0 = done; r0 < i1; r0 += kGramKr) {
      __syncthreads();  // buffer 0 is free
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        sx[0][m] = ld2(X, ldx, bx, r0 + er + 8 * m, a0 + ec);
        if constexpr (!DG) sy[0][m] = ld2(Y, ldy, by, r0 + er + 8 * m, b0 + ec);
      }
      put(0, 0, false, false);
      __syncthreads();
      chunk(0);
    }
  };
  if (diag) run(std::true_type{});
  else run(std::false_type{});
  if (idle) return;
  double* Pb = P + rblk * (int64_t)bx * by;
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      if (dquad && p > q) continue;
      const int as = a0 + 32 * qa + 16 * p;
      const int bs = b0 + 32 * qb + 16 * q;
      const bool mirror = (MODE == kGramSym && as != bs) || (MODE == kGramLower && ta != tb);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int a = as + 4 * j + kr;
        const int b = bs + cc;
        if (a >= bx || b >= by) continue;
        const double v = acc[p][q][j];
        Pb[a + (int64_t)b * bx] = v;
        if (mirror) Pb[b + (int64_t)a * bx] = v;
      }
    }
}

enum TallAfter { kTallNone = 0, kTallSums = 1, kTallGram = 2, kTallCross = 3 };

// out = alpha X C + beta Z (X: n x bx, C: bx x by column-major).  A wave owns
// 16 rows of a 64-row tile; lane (kk = l/16, r = l%16) loads the 16
// consecutive entries [16kk, 16kk+16) of row r of a 64-wide k chunk with
// 16-byte loads, and MFMA step s contracts k = 16kk + s: A[r][kk] =
// X[r][16kk+s], B[kk][c] = C[16kk+s][c] (LDS).  D[4j+kk][c] lands in register
// j, so 16 lanes store 16 consecutive columns of one row.  Workgroups loop
// over row tiles; C is staged once when bx <= 64.  blockIdx.y selects 64
// output columns.
//
// AFTER: what is also formed from the rows while they are in registers, so that
// no pass over the block follows for it (one partial per workgroup in P):
//   kTallSums: out's column sums of squares (by values);
//   kTallGram: out^T out (by x by, bx and by <= 64): a register of D is the A and
//     the B fragment of the rows' Gram product as it stands (lane (kk, r) holds
//     row 4j+kk of column 16t+r), so it costs MFMAs only;
//   kTallCross: X^T out (bx x by, both <= 64), X read again in D's layout.
template <bool BETA, int NTC, int AFTER, int NTX>
__global__ __launch_bounds__(kThreads) void tall_gemm_mfma_kernel(
    int64_t n, const double* __restrict__ X, int ldx, int bx, const double* __restrict__ C,
    int ldc, int by, double alpha, double beta, const double* Z, double* out, int ldo,
    int64_t ntiles, int ct, int64_t nstripe, double* __restrict__ P) {
  __shared__ double cs[kTile][kTile + 1];  // [k][c]
  // 1-D grid of nstripe x ct workgroups: the ct column tiles of a row stripe are
  // consecutive logical workgroups on one XCD, so X rows are read from HBM once
  const int64_t L = xcd_remap(blockIdx.x, gridDim.x);
  if (L >= nstripe * ct) return;
  const int c0 = (int)(L % ct) * kTile;
  const int64_t stripe = L / ct;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int kk = lane >> 4;
  const int r = lane & 15;
  const int nk = (bx + kTile - 1) / kTile;
  const bool vec_ok = ((reinterpret_cast<uintptr_t>(X) & 15) == 0) && (ldx % 2 == 0);
  auto stage = [&](int k0) {
    for (int e = threadIdx.x; e < kTile * kTile; e += kThreads) {
      const int k = e % kTile;
      const int c = e / kTile;
      cs[k][c] = (k0 + k < bx && c0 + c < by) ? C[(k0 + k) + (int64_t)(c0 + c) * ldc] : 0.0;
    }
  };
  if (nk == 1) {
    stage(0);
    __syncthreads();
  }
  double sum[AFTER == kTallSums ? NTC : 1];
  d4v gram[AFTER >= kTallGram ? NTX : 1][AFTER >= kTallGram ? NTC : 1];
  if constexpr (AFTER == kTallSums) {
#pragma unroll
    for (int t = 0; t < NTC; ++t) sum[t] = 0.0;
  }
  if constexpr (AFTER >= kTallGram) {
#pragma unroll
    for (int p = 0; p < NTX; ++p)
#pragma unroll
      for (int t = 0; t < NTC; ++t) gram[p][t] = d4v{0.0, 0.0, 0.0, 0.0};
  }
  for (int64_t tile = stripe; tile < ntiles; tile += nstripe) {
    const int64_t row = tile * kTile + wave * 16 + r;
    int zero = 0;
    d4v acc[NTC];
#pragma unroll
    for (int t = 0; t < NTC; ++t) acc[t] = d4v{0.0, 0.0, 0.0, 0.0};
    for (int ci = 0; ci < nk; ++ci) {
      const int k0 = ci * kTile;
      if (nk > 1) {
        __syncthreads();
        stage(k0);
        __syncthreads();
      }
      double xa[16];
      const int kb = k0 + 16 * kk;
      if (row < n && kb + 16 <= bx && vec_ok) {
        const double* xp = X + row * ldx + kb;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const dvec2 t = *reinterpret_cast<const dvec2*>(xp + 2 * q);
          xa[2 * q] = t.x;
          xa[2 * q + 1] = t.y;
        }
      } else {
#pragma unroll
        for (int q = 0; q < 16; ++q) xa[q] = (row < n && kb + q < bx) ? X[row * ldx + kb + q] : 0.0;
      }
#pragma unroll
      for (int sidx = 0; sidx < 16; ++sidx) {
        // as in tall_resid_kernel, where a Gram matrix needs the registers
        if (AFTER >= kTallGram && sidx % 4 == 0) asm volatile("" : "+s"(zero));
        // step sidx contracts k0 + sidx + {0, 16, 32, 48}: none is a column of X
        // once k0 + sidx >= bx (uniform)
        if (NTC == 4 || k0 + sidx < bx) {
          const int k = 16 * kk + sidx;
#pragma unroll
          for (int t = 0; t < NTC; ++t) acc[t] = mfma16x16x4(xa[sidx], cs[k][16 * t + r + zero], acc[t]);
        }
      }
    }
    // Z may be `out` itself: all of the lane's Z values are read before its
    // first store, so the loads are issued together
    double zv[4][NTC];
    if constexpr (BETA) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int64_t ro = tile * kTile + wave * 16 + 4 * j + kk;
#pragma unroll
        for (int t = 0; t < NTC; ++t) {
          const int c = c0 + 16 * t + r;
          zv[j][t] = (ro < n && c < by) ? Z[ro * ldo + c] : 0.0;
        }
      }
    }
    // X in D's layout: rows 4j+kk, columns 16p+r (read before the stores)
    double ya[AFTER == kTallCross ? 4 : 1][NTX];
    if constexpr (AFTER == kTallCross) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int64_t ro = tile * kTile + wave * 16 + 4 * j + kk;
#pragma unroll
        for (int p = 0; p < NTX; ++p)
          ya[j][p] = (ro < n && 16 * p + r < bx) ? X[ro * ldx + 16 * p + r] : 0.0;
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t ro = tile * kTile + wave * 16 + 4 * j + kk;
#pragma unroll
      for (int t = 0; t < NTC; ++t) {
        const int c = c0 + 16 * t + r;
        double v = alpha * acc[t][j];
        if constexpr (BETA) v = fma(beta, zv[j][t], v);
        if (ro < n && c < by) out[ro * ldo + c] = v;
        // rows past n and columns past by are zero here
        if constexpr (AFTER == kTallSums) sum[t] = fma(v, v, sum[t]);
        if constexpr (AFTER >= kTallGram) acc[t][j] = v;
      }
    }
    if constexpr (AFTER >= kTallGram) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int p = 0; p < NTX; ++p)
#pragma unroll
          for (int t = 0; t < NTC; ++t) {
            if (AFTER == kTallGram && p > t) continue;
            gram[p][t] =
                mfma16x16x4(AFTER == kTallGram ? acc[p][j] : ya[j][p], acc[t][j], gram[p][t]);
          }
    }
  }
  if constexpr (AFTER == kTallSums) {
    // over the 4 row groups of a wave, then the waves in order
#pragma unroll
    for (int t = 0; t < NTC; ++t) {
      sum[t] += __shfl_xor(sum[t], 16);
      sum[t] += __shfl_xor(sum[t], 32);
    }
    __syncthreads();  // C is no longer read
    double* red = &cs[0][0];
    if (kk == 0) {
#pragma unroll
      for (int t = 0; t < NTC; ++t) red[wave * kTile + 16 * t + r] = sum[t];
    }
    __syncthreads();
    const int c = (int)threadIdx.x;
    if (c < 16 * NTC && c0 + c < by)
      P[stripe * by + c0 + c] =
          ((red[c] + red[kTile + c]) + red[2 * kTile + c]) + red[3 * kTile + c];
  }
  if constexpr (AFTER >= kTallGram) {
    __syncthreads();
    double* red = &cs[0][0];
    for (int w = 0; w < 4; ++w) {
      if (wave == w) {
#pragma unroll
        for (int p = 0; p < NTX; ++p)
#pragma unroll
          for (int t = 0; t < NTC; ++t) {
            if (AFTER == kTallGram && p > t) continue;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const int e = (16 * p + 4 * j + kk) + kTile * (16 * t + r);
              red[e] = (w == 0) ? gram[p][t][j] : red[e] + gram[p][t][j];
            }
          }
      }
      __syncthreads();
    }
    const int rows = AFTER == kTallGram ? by : bx;
    double* Pb = P + stripe * (int64_t)rows * by;
    for (int e = threadIdx.x; e < kTile * kTile; e += kThreads) {
      const int a = e % kTile, b = e / kTile;
      if (a >= rows || b >= by) continue;
      // out^T out: the subtiles above the diagonal, and their mirror
      Pb[a + (int64_t)b * rows] = (AFTER == kTallGram && (a >> 4) > (b >> 4))
                                      ? red[b + kTile * a]
                                      : red[a + kTile * b];
    }
  }
}

// out = V C and, for its first nc columns, the sums of |theta_c out_c - (W C)_c|^2
// and |out_c|^2 (V, W: n x b, C: b x b column-major, b <= 64): the Ritz rotation
// and its residuals in one pass.  With W = A V, W C is A out, so the operator is
// not applied again: reads V and W and writes out, against a product, an apply and
// a pass over both results (128^3 x 64, 32 residuals: 0.42 + 0.46 + 0.18 ms -> 0.61;
// n = 17576, 24 columns: 10 + 6 + 6 us -> 14).  Lanes and
// fragments as in tall_gemm_mfma_kernel, C feeding both products.  NTC, NTR: 16-column
// subtiles of out and of its residual columns (constants: a branch on nc between
// the MFMAs made the accumulators spill, 1.43 ms).
template <int NTC, int NTR>
__global__ __launch_bounds__(kThreads, 2) void tall_resid_kernel(
    int64_t n, const double* __restrict__ V, const double* __restrict__ W, int ld, int b,
    const double* __restrict__ C, double* __restrict__ out, const ThetaArgs theta, int nc,
    int64_t ntiles, int64_t nstripe, double* __restrict__ P) {
  __shared__ double cs[kTile][kTile + 1];  // [k][c]
  const int64_t stripe = xcd_remap(blockIdx.x, gridDim.x);
  if (stripe >= nstripe) return;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int kk = lane >> 4;
  const int r = lane & 15;
  const bool vec_ok = ld % 2 == 0 && ((reinterpret_cast<uintptr_t>(V) & 15) == 0) &&
                      ((reinterpret_cast<uintptr_t>(W) & 15) == 0);
  for (int e = threadIdx.x; e < kTile * kTile; e += kThreads) {
    const int k = e % kTile;
    const int c = e / kTile;
    cs[k][c] = (k < b && c < b) ? C[k + (int64_t)c * b] : 0.0;
  }
  double th[NTR], res[NTR], nrm[NTR];
#pragma unroll
  for (int t = 0; t < NTR; ++t) {
    th[t] = 16 * t + r < nc ? theta.v[16 * t + r] : 0.0;
    res[t] = nrm[t] = 0.0;
  }
  __syncthreads();
  for (int64_t tile = stripe; tile < ntiles; tile += nstripe) {
    const int64_t row = tile * kTile + wave * 16 + r;
    double xa[16], wa[16];
    const int kb = 16 * kk;
    if (row < n && kb + 16 <= b && vec_ok) {
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const dvec2 x = *reinterpret_cast<const dvec2*>(V + row * ld + kb + 2 * q);
        const dvec2 w = *reinterpret_cast<const dvec2*>(W + row * ld + kb + 2 * q);
        xa[2 * q] = x.x;
        xa[2 * q + 1] = x.y;
        wa[2 * q] = w.x;
        wa[2 * q + 1] = w.y;
      }
    } else {
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        const bool in = row < n && kb + q < b;
        xa[q] = in ? V[row * ld + kb + q] : 0.0;
        wa[q] = in ? W[row * ld + kb + q] : 0.0;
      }
    }
    int zero = 0;
    d4v av[NTC], aw[NTR];
#pragma unroll
    for (int t = 0; t < NTC; ++t) av[t] = d4v{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int t = 0; t < NTR; ++t) aw[t] = d4v{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int sidx = 0; sidx < 16; ++sidx) {
      // C's fragments are read from LDS four steps at a time (an offset of zero
      // that the compiler cannot see through): held in registers for all steps, or
      // over the tiles, as it would, they spill
      if (sidx % 4 == 0) asm volatile("" : "+s"(zero));
      // step sidx contracts sidx + {0, 16, 32, 48}: none below b once sidx >= b
      if (NTC == 4 || sidx < b) {
#pragma unroll
        for (int t = 0; t < NTC; ++t) {
          const double f = cs[16 * kk + sidx][16 * t + r + zero];
          av[t] = mfma16x16x4(xa[sidx], f, av[t]);
          if (t < NTR) aw[t < NTR ? t : 0] = mfma16x16x4(wa[sidx], f, aw[t < NTR ? t : 0]);
        }
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t ro = tile * kTile + wave * 16 + 4 * j + kk;
#pragma unroll
      for (int t = 0; t < NTC; ++t) {
        const double v = av[t][j];
        if (ro < n && 16 * t + r < b) out[ro * ld + 16 * t + r] = v;
        if (t < NTR) {  // zero in rows past n
          constexpr int last = NTR - 1;
          const int u = t < NTR ? t : last;
          const double d = th[u] * v - aw[u][j];
          res[u] = fma(d, d, res[u]);
          nrm[u] = fma(v, v, nrm[u]);
        }
      }
    }
  }
  // over the 4 row groups of a wave, then the waves in order
#pragma unroll
  for (int t = 0; t < NTR; ++t) {
    res[t] += __shfl_xor(res[t], 16);
    res[t] += __shfl_xor(res[t], 32);
    nrm[t] += __shfl_xor(nrm[t], 16);
    nrm[t] += __shfl_xor(nrm[t], 32);
  }
  __syncthreads();  // C is no longer read
  double* red = &cs[0][0];
  if (kk == 0) {
#pragma unroll
    for (int t = 0; t < NTR; ++t) {
      red[(2 * wave) * kTile + 16 * t + r] = res[t];
      red[(2 * wave + 1) * kTile + 16 * t + r] = nrm[t];
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < 2 * nc; e += kThreads) {
    const int c = e % nc, h = e / nc;  // h: 0 residuals, 1 norms
    P[stripe * 2 * nc + e] = ((red[h * kTile + c] + red[(2 + h) * kTile + c]) +
                              red[(4 + h) * kTile + c]) + red[(6 + h) * kTile + c];
  }
}

// out = alpha X C + beta Z for 64 < bx <= 64 KCH (the Gram-sized products of
// blocks of up to 256 columns).  The workgroup's whole 64-column slice of C
// (64 KCH x 64) is staged in LDS once; the workgroup then walks 128-row tiles
// with no further barrier.  Each wave owns 32 rows (two 16-row MFMA groups),
// so every B fragment read from LDS feeds two MFMAs, and the next 64-wide k
// chunk of its X rows -- in the last chunk, the next tile's first -- is loaded
// while the current one is multiplied.  Whether every row and column of a
// wave's chunk exists is decided once per wave (a scalar branch): loads that
// lanes take or skip on their own would make the wave wait for the loads in
// flight where the paths join, which takes the prefetch's overlap away.
// SUMS: also out's column sums of squares, a partial per workgroup in P.
template <int KCH, bool SUMS>
__global__ __launch_bounds__(kThreads) void tall_gemm_wide_kernel(
    int64_t n, const double* __restrict__ X, int ldx, int bx, const double* __restrict__ C,
    int ldc, int by, double alpha, double beta, const double* Z, double* out, int ldo,
    int64_t ntiles, int ct, int64_t nstripe, double* __restrict__ P) {
  constexpr int KP = KCH * kTile;
  __shared__ double cs[KP][kTile + 1];  // [k][c]
  const int64_t L = xcd_remap(blockIdx.x, gridDim.x);
  if (L >= nstripe * ct) return;
  const int c0 = (int)(L % ct) * kTile;
  const int64_t stripe = L / ct;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int kk = lane >> 4;
  const int r = lane & 15;
  const bool vec_ok = ((reinterpret_cast<uintptr_t>(X) & 15) == 0) && (ldx % 2 == 0);
  for (int e = threadIdx.x; e < KP * kTile; e += kThreads) {
    const int k = e % KP;
    const int c = e / KP;
    cs[k][c] = (k < bx && c0 + c < by) ? C[k + (int64_t)(c0 + c) * ldc] : 0.0;
  }
  __syncthreads();
  // lane (kk, r) of group g holds X[row_g][k0 + 16kk + q], q < 16; r0 and k0
  // are the same for the whole wave
  auto load = [&](int64_t r0, int k0, double (&xv)[2][16]) {
    const int kb = k0 + 16 * kk;
    const bool full = __builtin_amdgcn_readfirstlane(
                          (int)(vec_ok && r0 + 32 <= n && k0 + kTile <= bx)) != 0;
    if (full) {
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const double* xp = X + (r0 + 16 * g + r) * ldx + kb;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const dvec2 t = *reinterpret_cast<const dvec2*>(xp + 2 * q);
          xv[g][2 * q] = t.x;
          xv[g][2 * q + 1] = t.y;
        }
      }
    } else {
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const int64_t row = r0 + 16 * g + r;
#pragma unroll
        for (int q = 0; q < 16; ++q)
          xv[g][q] = (row < n && kb + q < bx) ? X[row * ldx + kb + q] : 0.0;
      }
    }
  };
  // xn receives every load and xa is only ever written from it by copies: a
  // register that entered the loops with a load in flight would make every
  // chunk wait for the loads issued ahead of its MFMAs
  double xa[2][16], xn[2][16];
  double sum[4] = {0.0, 0.0, 0.0, 0.0};
  if (stripe < ntiles) load(stripe * (2 * kTile) + wave * 32, 0, xn);
  for (int64_t tile = stripe; tile < ntiles; tile += nstripe) {
    const int64_t r0 = tile * (2 * kTile) + wave * 32;
    const bool next = tile + nstripe < ntiles;
    // every output row and column of the wave's tile exists (Z reads and the
    // stores then take no per-lane branches)
    const bool ofull =
        __builtin_amdgcn_readfirstlane((int)(r0 + 32 <= n && c0 + kTile <= by)) != 0;
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int q = 0; q < 16; ++q) xa[g][q] = xn[g][q];
    d4v acc[2][4];
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int t = 0; t < 4; ++t) acc[g][t] = d4v{0.0, 0.0, 0.0, 0.0};
    // beta Z of the epilogue, read at the start of the last chunk: Z may be
    // `out` itself, so loads issued between the stores would each wait for
    // the one before
    double zv[2][4][4];
#pragma unroll 1
    for (int ci = 0; ci < KCH; ++ci) {
      // one load site for both prefetches, so that they land in the same
      // registers and need no copies (which would wait for them) to merge
      if (ci + 1 < KCH || next)
        load(ci + 1 < KCH ? r0 : r0 + nstripe * (2 * kTile), ci + 1 < KCH ? (ci + 1) * kTile : 0,
             xn);
      if (ci + 1 == KCH && beta != 0.0) {
        if (ofull) {
#pragma unroll
          for (int g = 0; g < 2; ++g)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
              for (int t = 0; t < 4; ++t)
                zv[g][j][t] = Z[(r0 + 16 * g + 4 * j + kk) * ldo + c0 + 16 * t + r];
        } else {
#pragma unroll
          for (int g = 0; g < 2; ++g)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const int64_t ro = r0 + 16 * g + 4 * j + kk;
#pragma unroll
              for (int t = 0; t < 4; ++t) {
                const int c = c0 + 16 * t + r;
                zv[g][j][t] = (ro < n && c < by) ? Z[ro * ldo + c] : 0.0;
              }
            }
        }
      }
#pragma unroll
      for (int sidx = 0; sidx < 16; ++sidx) {
        const int k = ci * kTile + 16 * kk + sidx;
        double b[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) b[t] = cs[k][16 * t + r];
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
          for (int t = 0; t < 4; ++t) acc[g][t] = mfma16x16x4(xa[g][sidx], b[t], acc[g][t]);
      }
      if (ci + 1 < KCH) {
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
          for (int q = 0; q < 16; ++q) xa[g][q] = xn[g][q];
      }
    }
    if (ofull) {
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            double v = alpha * acc[g][t][j];
            if (beta != 0.0) v = fma(beta, zv[g][j][t], v);
            out[(r0 + 16 * g + 4 * j + kk) * ldo + c0 + 16 * t + r] = v;
            if constexpr (SUMS) sum[t] = fma(v, v, sum[t]);
          }
    } else {
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int64_t ro = r0 + 16 * g + 4 * j + kk;
          if (ro >= n) continue;
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const int c = c0 + 16 * t + r;
            if (c >= by) continue;
            double v = alpha * acc[g][t][j];
            if (beta != 0.0) v = fma(beta, zv[g][j][t], v);
            out[ro * ldo + c] = v;
            if constexpr (SUMS) sum[t] = fma(v, v, sum[t]);
          }
        }
    }
  }
  if constexpr (SUMS) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      sum[t] += __shfl_xor(sum[t], 16);
      sum[t] += __shfl_xor(sum[t], 32);
    }
    __syncthreads();  // C is no longer read
    double* red = &cs[0][0];
    if (kk == 0) {
#pragma unroll
      for (int t = 0; t < 4; ++t) red[wave * kTile + 16 * t + r] = sum[t];
    }
    __syncthreads();
    const int c = (int)threadIdx.x;
    if (c < kTile && c0 + c < by)
      P[stripe * by + c0 + c] =
          ((red[c] + red[kTile + c]) + red[2 * kTile + c]) + red[3 * kTile + c];
  }
}

// ------------------------------------------------ dense operator (MFMA)
// v_mfma_f32_16x16x4f32: lane l supplies A[l%16][l/16] and B[l/16][l%16] as
// for FP64; register j holds D[4(l/16) + j][l%16].
typedef float f4v __attribute__((ext_vector_type(4)));
__device__ __forceinline__ f4v mfma16x16x4(float a, float b, f4v c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
template <typename T>
struct MfmaAcc;
template <>
struct MfmaAcc<double> {
  typedef d4v type;
  // row within the 16x16 tile of register j of lane l
  __device__ static int row(int j, int l) { return 4 * j + (l >> 4); }
};
template <>
struct MfmaAcc<float> {
  typedef f4v type;
  __device__ static int row(int j, int l) { return 4 * (l >> 4) + j; }
};

// One filter step (or apply) of a dense symmetric operator A (n x n,
// row-major = column-major) on a row-interleaved block:
//   kApply: out = p0 A X;  kApplyBeta: out = p0 A X + p1 out;
//   kChebFirst: out = p2 p1 (p0 A X + X);  kCheb: out = p2 (p1 (p0 A X + X) - Z);
//   kChebSrc: kCheb + kap[c] R.
// BM x 64 output tile per workgroup; wave w owns rows [w BM/4, (w+1) BM/4), all
// 64 columns: FP64 (BM = 128) 2 x 4 MFMA 16x16x4 tiles, 6 LDS fragment reads
// per 8 MFMAs; FP32 (BM = 64) 1 x 4 tiles.
// K runs in chunks of BK through two LDS buffers and two register sets: a
// chunk's global loads are issued two chunks before its MFMAs and stored into
// the free LDS buffer after the MFMAs of the chunk before it, one barrier per
// chunk.  The column tiles of a row
// tile are consecutive logical workgroups, kept on one XCD, so the A rows
// they share come from the same L2.  The step is made on columns [cfirst, ncols),
// cfirst a multiple of 4.
template <typename T>
struct DenseCfg {
  // FP32 runs 64-row tiles (16 rows per wave): at n = 16384, b = 256 that is
  // 1024 workgroups instead of 512, 4.5% faster per step than 128 rows; 32-column
  // tiles, K chunks of 16 or 64, and 32x32 per wave were slower
  // (FP64 in 64-row tiles too, 4 waves per SIMD: 2.44 -> 2.69 ms per step)
  static constexpr int BM = sizeof(T) == 8 ? 128 : 64;
  static constexpr int BN = 64;
  static constexpr int BK = sizeof(T) == 8 ? 16 : 32;
  // LDS row padding (elements) of the A and X tiles.  FP32: rows of 34 and 80
  // floats put the 16 rows x 2 K of a half-wave's A fragment reads, and the
  // 16 columns x 2 K of its X reads, in distinct banks; with 33 and 65 bank
  // conflicts took 25% of the step's cycles, but removing them gains only 1%
  // (1403 -> 1384 us at n = 16384, b = 256): the MFMA issue, not LDS, binds.
  static constexpr int PA = sizeof(T) == 8 ? 1 : 2;
  static constexpr int PX = sizeof(T) == 8 ? 1 : 16;
};
// The products of one K split, summed by dense_combine_kernel.
constexpr int kDensePartial = 7;
template <typename T, int MODE>
__global__ __launch_bounds__(kThreads, 2) void dense_step_kernel(
    int64_t n, const T* __restrict__ A, int64_t lda, const T* __restrict__ X, const T* Z, T* out,
    int ld, int ncols, T p0, T p1, T p2, const T* __restrict__ R, const T* __restrict__ kap,
    int cfirst, int ntn, int nsplit, T* __restrict__ P) {
  constexpr int BK = DenseCfg<T>::BK;
  constexpr int BM = DenseCfg<T>::BM, BN = DenseCfg<T>::BN;
  constexpr int AE = BM * BK / kThreads;  // A elements per thread per chunk
  constexpr int XE = BK * BN / kThreads;  // X elements per thread per chunk
  constexpr int WR = BM / 4;              // rows per wave
  constexpr int NA = WR / 16, NB = BN / 16;
  __shared__ T As[2][BM][BK + DenseCfg<T>::PA];
  __shared__ T Xs[2][BK][BN + DenseCfg<T>::PX];
  using Acc = typename MfmaAcc<T>::type;
  const int64_t L = xcd_remap(blockIdx.x, gridDim.x);
  const int64_t ntm = (n + BM - 1) / BM;
  if (L >= ntm * ntn * nsplit) return;
  // K range of this split, whole chunks but for the last one's end
  const int64_t split = L / (ntm * ntn), T0 = L % (ntm * ntn);
  const int64_t kper = (n + (int64_t)nsplit * BK - 1) / ((int64_t)nsplit * BK) * BK;
  const int64_t kbeg = min(n, split * kper), kend = min(n, kbeg + kper);
  const int64_t i0 = (T0 / ntn) * BM;
  const int c0 = cfirst + (int)(T0 % ntn) * BN;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  Acc acc[NA][NB];
#pragma unroll
  for (int a = 0; a < NA; ++a)
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[a][b] = Acc{0, 0, 0, 0};
  // Each thread loads AE consecutive A entries of one row and XE consecutive
  // X entries of one K row, in 16-byte vectors when they are whole and
  // aligned (the chunk offset moves along K).
  using VT = V16<T>;
  constexpr int W = VT::W;
  static_assert(AE % W == 0 && XE % W == 0 && WR % 16 == 0 && BN % 16 == 0, "dense tile shape");
  constexpr int TPA = BK / AE;  // threads per A row
  constexpr int TPX = BN / XE;  // threads per X row
  const int ar = threadIdx.x / TPA, ak = (threadIdx.x % TPA) * AE;
  const int xk = threadIdx.x / TPX, xc = (threadIdx.x % TPX) * XE;
  const int64_t ai = i0 + ar;
  const bool a_vec = ((reinterpret_cast<uintptr_t>(A) & 15) == 0) && (lda % W == 0);
  const bool x_vec = ((reinterpret_cast<uintptr_t>(X) & 15) == 0) && (ld % W == 0) &&
                     (c0 + xc + XE <= ncols);
  // Whole chunks are loaded with no guard: a row past n reads row n - 1 and a
  // column vector past the rows' padding the last one, whose products land in
  // entries that are not stored.  A's rows may start at any multiple of an element.
  const bool x_ok = ((reinterpret_cast<uintptr_t>(X) & 15) == 0) && (ld % W == 0);
  const T* arow = A + min(ai, n - 1) * lda + ak;
  int xcol[XE / W];
#pragma unroll
  for (int q = 0; q < XE / W; ++q) xcol[q] = min(c0 + xc + q * W, ld - W);
  typedef T VecU __attribute__((ext_vector_type(W), aligned(sizeof(T))));
  T ra2[2][AE], rx2[2][XE];
  auto fetch_full = [&](int64_t k0, T (&ra)[AE], T (&rx)[XE]) {
#pragma unroll
    for (int q = 0; q < AE / W; ++q) {
      const VecU t = *reinterpret_cast<const VecU*>(arow + k0 + q * W);
#pragma unroll
      for (int w = 0; w < W; ++w) ra[q * W + w] = t[w];
    }
#pragma unroll
    for (int q = 0; q < XE / W; ++q) {
      T t[W];
      VT::ld(X + (k0 + xk) * ld + xcol[q], t);
#pragma unroll
      for (int w = 0; w < W; ++w) rx[q * W + w] = t[w];
    }
  };
  auto fetch_to = [&](int64_t k0, T (&ra)[AE], T (&rx)[XE]) {
    const int64_t ka = k0 + ak;
    if (a_vec && ai < n && ka + AE <= kend) {
      const T* ap = A + ai * lda + ka;
#pragma unroll
      for (int q = 0; q < AE / W; ++q) {
        T t[W];
        VT::ld(ap + q * W, t);
#pragma unroll
        for (int w = 0; w < W; ++w) ra[q * W + w] = t[w];
      }
    } else {
#pragma unroll
      for (int q = 0; q < AE; ++q) ra[q] = (ai < n && ka + q < kend) ? A[ai * lda + ka + q] : T(0);
    }
    const int64_t kx = k0 + xk;
    if (x_vec && kx < kend) {
      const T* xp = X + kx * ld + c0 + xc;
#pragma unroll
      for (int q = 0; q < XE / W; ++q) {
        T t[W];
        VT::ld(xp + q * W, t);
#pragma unroll
        for (int w = 0; w < W; ++w) rx[q * W + w] = t[w];
      }
    } else {
#pragma unroll
      for (int q = 0; q < XE; ++q) {
        const int c = c0 + xc + q;
        rx[q] = (kx < kend && c < ncols) ? X[kx * ld + c] : T(0);
      }
    }
  };
  auto chunk = [&](int buf) {
#pragma unroll
    for (int ks = 0; ks < BK; ks += 4) {
      const int kk = ks + (lane >> 4);
      T af[NA], bf[NB];
#pragma unroll
      for (int a = 0; a < NA; ++a) af[a] = As[buf][WR * wave + 16 * a + (lane & 15)][kk];
#pragma unroll
      for (int b = 0; b < NB; ++b) bf[b] = Xs[buf][kk][16 * b + (lane & 15)];
#pragma unroll
      for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[a][b] = mfma16x16x4(af[a], bf[b], acc[a][b]);
    }
  };
  // Chunk c is loaded into register set c % 2 two chunks before its MFMAs
  // and stored to LDS buffer c % 2 at the end of chunk c - 1, so its global
  // loads have two chunks of MFMAs to arrive in (FP64 step at n = 16384,
  // b = 256: 2.77 -> 2.45 ms, 49.6 -> 56.1 TFLOP/s; one chunk ahead left the
  // MFMA pipes idle 37% of the kernel, waves waiting on loads).
  auto put = [&](int buf, const T (&sa)[AE], const T (&sx)[XE]) {
#pragma unroll
    for (int q = 0; q < AE; ++q) As[buf][ar][ak + q] = sa[q];
#pragma unroll
    for (int q = 0; q < XE; ++q) Xs[buf][xk][xc + q] = sx[q];
  };
  // Chunks [0, done) without guards.  The loop has no branch between a set's loads
  // and its LDS stores: with one (whole chunk or not, last chunk or not) the
  // compiler cannot count the loads in flight and waits for all of them, the set
  // just issued included, before every store -- the loads were then one chunk
  // of MFMAs ahead, not two (FP64 step at n = 16384, b = 256: 2.38 -> 2.05 ms, 67
  // TFLOP/s; FP32 1.19 -> 1.13; n = 9001, b = 64, whose rows are not 16-byte
  // aligned: 1.22 -> 0.70 and 0.54 -> 0.23).
  int64_t done = kbeg;
  if (__builtin_amdgcn_readfirstlane((int)(x_ok && kend - kbeg >= 4 * BK)) != 0) {
    const int64_t nf = (kend - kbeg) / BK;
    fetch_full(kbeg, ra2[0], rx2[0]);
    put(0, ra2[0], rx2[0]);
    fetch_full(kbeg + BK, ra2[1], rx2[1]);
    __syncthreads();
    int64_t c = 0;
    for (; c + 3 < nf; c += 2) {
      fetch_full(kbeg + (c + 2) * BK, ra2[0], rx2[0]);
      chunk(0);
      put(1, ra2[1], rx2[1]);
      __syncthreads();
      fetch_full(kbeg + (c + 3) * BK, ra2[1], rx2[1]);
      chunk(1);
      put(0, ra2[0], rx2[0]);
      __syncthreads();
    }
    // the last two or three: c in buffer 0, c + 1 in set 1
    const bool three = c + 2 < nf;
    if (three) fetch_full(kbeg + (c + 2) * BK, ra2[0], rx2[0]);
    chunk(0);
    put(1, ra2[1], rx2[1]);
    __syncthreads();
    chunk(1);
    if (three) {
      put(0, ra2[0], rx2[0]);
      __syncthreads();
      chunk(0);
    }
    done = kbeg + nf * BK;
    __syncthreads();  // both buffers are free
  }
  if (done < kend) {
    fetch_to(done, ra2[0], rx2[0]);
    put(0, ra2[0], rx2[0]);
    if (done + BK < kend) fetch_to(done + BK, ra2[1], rx2[1]);
    __syncthreads();
  }
  for (int64_t k0 = done; k0 < kend; k0 += 2 * BK) {
    // even chunk: buffer 0, its successor in set 1; fetch chunk + 2 into set 0
    if (k0 + 2 * BK < kend) fetch_to(k0 + 2 * BK, ra2[0], rx2[0]);
    chunk(0);
    if (k0 + BK < kend) put(1, ra2[1], rx2[1]);
    __syncthreads();
    if (k0 + BK >= kend) break;
    // odd chunk: buffer 1, its successor in set 0; fetch chunk + 2 into set 1
    if (k0 + 3 * BK < kend) fetch_to(k0 + 3 * BK, ra2[1], rx2[1]);
    chunk(1);
    if (k0 + 2 * BK < kend) put(0, ra2[0], rx2[0]);
    __syncthreads();
  }
#pragma unroll
  for (int a = 0; a < NA; ++a)
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int64_t i = i0 + WR * wave + 16 * a + MfmaAcc<T>::row(j, lane);
        const int c = c0 + 16 * b + (lane & 15);
        if (i >= n || c >= ncols) continue;
        const int64_t off = i * ld + c;
        const T v = acc[a][b][j];
        if constexpr (MODE == kDensePartial) {
          P[(split * n + i) * (ncols - cfirst) + c - cfirst] = v;
          continue;
        }
        T o;
        if constexpr (MODE == kApply || MODE == kDensePartial) o = p0 * v;
        else if constexpr (MODE == kApplyBeta) o = fma(p0, v, p1 * out[off]);
        else if constexpr (MODE == kChebFirst) o = p2 * (p1 * fma(p0, v, X[off]));
        else if constexpr (MODE == kCheb) o = p2 * fma(p1, fma(p0, v, X[off]), -Z[off]);
        else o = p2 * fma(kap[c], R[off], fma(p1, fma(p0, v, X[off]), -Z[off]));
        out[off] = o;
      }
}

// The step from the K splits' partial products, summed in their order.
template <int MODE>
__global__ __launch_bounds__(kThreads) void dense_combine_kernel(
    int64_t n, const double* __restrict__ P, int nsplit, const double* X, const double* Z,
    double* out, int ld, int cfirst, int ncols, double p0, double p1, double p2) {
  const int64_t e = blockIdx.x * (int64_t)kThreads + threadIdx.x;
  const int nc = ncols - cfirst;
  const int64_t m = n * nc;
  if (e >= m) return;
  double v = 0.0;
  for (int s = 0; s < nsplit; s += 4) {
    double x[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) x[u] = s + u < nsplit ? P[(s + u) * m + e] : 0.0;
#pragma unroll
    for (int u = 0; u < 4; ++u) v += x[u];
  }
  const int64_t off = (e / nc) * ld + cfirst + e % nc;
  double o;
  if constexpr (MODE == kApply) o = p0 * v;
  else if constexpr (MODE == kApplyBeta) o = fma(p0, v, p1 * out[off]);
  else if constexpr (MODE == kChebFirst) o = p2 * (p1 * fma(p0, v, X[off]));
  else o = p2 * fma(p1, fma(p0, v, X[off]), -Z[off]);
  out[off] = o;
}

// One column of a dense operator (the dense Lanczos matrix-vector products):
// out = p0 A x (+ p1 out with kApplyBeta).  A wave owns a row: its lanes read
// 16-byte pieces of the row in order and sum them, then a fixed shuffle tree
// adds the lanes.
template <int MODE>
__global__ __launch_bounds__(kThreads) void dense_gemv_kernel(int64_t n,
                                                              const double* __restrict__ A,
                                                              int64_t lda,
                                                              const double* __restrict__ x,
                                                              double* out, double p0, double p1) {
  const int lane = threadIdx.x & 63;
  const int64_t i = blockIdx.x * (int64_t)(kThreads / 64) + (threadIdx.x >> 6);
  if (i >= n) return;  // uniform across the wave
  const double* a = A + i * lda;
  const bool vec = ((reinterpret_cast<uintptr_t>(a) & 15) == 0) &&
                   ((reinterpret_cast<uintptr_t>(x) & 15) == 0);
  double s0 = 0.0, s1 = 0.0;
  int64_t k = 2 * (int64_t)lane;
  if (vec) {
    for (; k + 1 < n; k += 128) {
      const dvec2 av = *reinterpret_cast<const dvec2*>(a + k);
      const dvec2 xv = *reinterpret_cast<const dvec2*>(x + k);
      s0 = fma(av.x, xv.x, s0);
      s1 = fma(av.y, xv.y, s1);
    }
    if (k < n) s0 = fma(a[k], x[k], s0);
  } else {
    for (; k < n; k += 128) {
      s0 = fma(a[k], x[k], s0);
      if (k + 1 < n) s1 = fma(a[k + 1], x[k + 1], s1);
    }
  }
  double s = s0 + s1;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
  if (lane == 0) {
    if constexpr (MODE == kApplyBeta) out[i] = fma(p0, s, p1 * out[i]);
    else out[i] = p0 * s;
  }
}

// ------------------------------------------------------ column reductions
// Threads are laid out as (row slot, column): CW columns per pass.
constexpr int kColRows = 512;  // rows per partial block
// Rows whose loads a column-reduction thread issues together before adding
// them in row order (the sums are those of the one-row loop): at n ~ 5e4,
// b = 24 a thread walks ~50 rows, one load latency each when taken singly.
constexpr int kColDepth = 8;

template <typename T, bool RESID>
__global__ __launch_bounds__(kThreads) void col_sumsq_kernel(int64_t n, const T* __restrict__ V,
                                                             const T* __restrict__ Wm, int ld,
                                                             int nc, const double* theta,
                                                             double* __restrict__ P) {
  __shared__ double red[kThreads];
  const int64_t blk = blockIdx.x;
  const int cw = min(nc, kThreads);  // columns per pass
  const int slots = kThreads / cw;
  const int c_in = threadIdx.x % cw;
  const int slot = threadIdx.x / cw;
  const int64_t i0 = blk * kColRows;
  const int64_t i1 = min(n, i0 + kColRows);
  for (int cbase = 0; cbase < nc; cbase += cw) {
    const int c = cbase + c_in;
    double s = 0.0;
    if (slot < slots && c < nc) {
      const double th = RESID ? theta[c] : 0.0;
      int64_t i = i0 + slot;
      // kColDepth rows' loads in flight, summed in row order as one at a time
      for (; i + (kColDepth - 1) * slots < i1; i += kColDepth * slots) {
        double v[kColDepth], w[kColDepth];
#pragma unroll
        for (int k = 0; k < kColDepth; ++k) {
          v[k] = double(V[(i + k * slots) * ld + c]);
          if (RESID) w[k] = double(Wm[(i + k * slots) * ld + c]);
        }
#pragma unroll
        for (int k = 0; k < kColDepth; ++k) {
          double x = v[k];
          if (RESID) x = th * x - w[k];
          s += x * x;
        }
      }
      for (; i < i1; i += slots) {
        double v = double(V[i * ld + c]);
        if (RESID) v = th * v - double(Wm[i * ld + c]);
        s += v * v;
      }
    }
    red[threadIdx.x] = s;
    __syncthreads();
    if (slot == 0 && c < nc) {
      double t = red[threadIdx.x];
      for (int q = 1; q < slots; ++q) t += red[threadIdx.x + q * cw];
      P[blk * nc + c] = t;
    }
    __syncthreads();
  }
}

// Residual and norm sums together: P[blk*2nc + c] = sum_i |theta_c V - W|^2,
// P[blk*2nc + nc + c] = sum_i |V|^2 over the block's rows.
// TH: const double* (theta in device memory) or ThetaArgs (in the arguments)
template <typename T, typename TH>
__global__ __launch_bounds__(kThreads) void resid_norm_kernel(int64_t n, const T* __restrict__ V,
                                                              const T* __restrict__ Wm, int ld,
                                                              int nc, const TH theta,
                                                              double* __restrict__ P) {
  __shared__ double red[2 * kThreads];
  const int64_t blk = blockIdx.x;
  const int cw = min(nc, kThreads);
  const int slots = kThreads / cw;
  const int c_in = threadIdx.x % cw;
  const int slot = threadIdx.x / cw;
  const int64_t i0 = blk * kColRows;
  const int64_t i1 = min(n, i0 + kColRows);
  for (int cbase = 0; cbase < nc; cbase += cw) {
    const int c = cbase + c_in;
    double s = 0.0, q = 0.0;
    if (slot < slots && c < nc) {
      const double th = theta[c];
      int64_t i = i0 + slot;
      for (; i + (kColDepth - 1) * slots < i1; i += kColDepth * slots) {
        double v[kColDepth], w[kColDepth];
#pragma unroll
        for (int k = 0; k < kColDepth; ++k) {
          v[k] = double(V[(i + k * slots) * ld + c]);
          w[k] = double(Wm[(i + k * slots) * ld + c]);
        }
#pragma unroll
        for (int k = 0; k < kColDepth; ++k) {
          const double r = th * v[k] - w[k];
          s += r * r;
          q += v[k] * v[k];
        }
      }
      for (; i < i1; i += slots) {
        const double v = double(V[i * ld + c]);
        const double r = th * v - double(Wm[i * ld + c]);
        s += r * r;
        q += v * v;
      }
    }
    red[threadIdx.x] = s;
    red[kThreads + threadIdx.x] = q;
    __syncthreads();
    if (slot == 0 && c < nc) {
      double t = red[threadIdx.x], u = red[kThreads + threadIdx.x];
      for (int k = 1; k < slots; ++k) {
        t += red[threadIdx.x + k * cw];
        u += red[kThreads + threadIdx.x + k * cw];
      }
      P[blk * 2 * nc + c] = t;
      P[blk * 2 * nc + nc + c] = u;
    }
    __syncthreads();
  }
}

template <typename T>
__global__ __launch_bounds__(kThreads) void normalize_cols_kernel(int64_t n, T* X, int ld, int nc,
                                                                  const double* __restrict__ sums) {
  const int64_t e = blockIdx.x * (int64_t)kThreads + threadIdx.x;
  const int64_t i = e / nc;
  const int c = (int)(e % nc);
  if (i >= n) return;
  const double s = 1.0 / sqrt(fabs(sums[c]));
  X[i * ld + c] = T(double(X[i * ld + c]) * s);
}

// out[i,c] = X[i,c] / sqrt(|sums[c]|) (out may be X)
__global__ __launch_bounds__(kThreads) void scale_cols_kernel(int64_t n, const double* X, int ld,
                                                              int nc,
                                                              const double* __restrict__ sums,
                                                              double* out) {
  const int64_t e = blockIdx.x * (int64_t)kThreads + threadIdx.x;
  const int64_t i = e / nc;
  const int c = (int)(e % nc);
  if (i >= n) return;
  const double s = 1.0 / sqrt(fabs(sums[c]));
  out[i * ld + c] = X[i * ld + c] * s;
}

template <typename T>
__global__ __launch_bounds__(kThreads) void copy_cols_kernel(int64_t n, const T* __restrict__ src,
                                                             int lds, int s0, T* __restrict__ dst,
                                                             int ldd, int d0, int cnt) {
  const int64_t e = blockIdx.x * (int64_t)kThreads + threadIdx.x;
  const int64_t i = e / cnt;
  const int j = (int)(e % cnt);
  if (i >= n) return;
  dst[i * ldd + d0 + j] = src[i * lds + s0 + j];
}

__device__ __forceinline__ uint64_t mix64(uint64_t z) {
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
  return z ^ (z >> 31);
}
__device__ __forceinline__ double sym_draw(uint64_t key, uint64_t idx) {
  const uint64_t z = mix64(key + (idx + 1) * 0x9E3779B97F4A7C15ULL);
  return -1.0 + 2.0 * (double(z >> 11) * 0x1.0p-53);
}

template <typename T>
__global__ __launch_bounds__(kThreads) void randomize_cols_kernel(int64_t n, T* X, int ld, int c0,
                                                                  int cnt, uint64_t key,
                                                                  uint64_t counter) {
  // thread per (row, column): column-fastest so stores are coalesced.
  const int64_t e = blockIdx.x * (int64_t)kThreads + threadIdx.x;
  const int64_t i = e / cnt;
  const int j = (int)(e % cnt);
  if (i >= n) return;
  X[i * ld + c0 + j] = T(sym_draw(key, counter + (uint64_t)j * (uint64_t)n + (uint64_t)i));
}

template <typename T>
__global__ __launch_bounds__(kThreads) void fill_cols_kernel(int64_t n, T* X, int ld, int c0,
                                                             int cnt, T value) {
  const int64_t e = blockIdx.x * (int64_t)kThreads + threadIdx.x;
  const int64_t i = e / cnt;
  const int j = (int)(e % cnt);
  if (i >= n) return;
  X[i * ld + c0 + j] = value;
}

// ------------------------------------------------ mixed-precision filter
// Start of the correction recurrence X_j = u_j(theta_c) v + E_j: from
// V (FP64) and AV (FP64), per column c < nc with cp[c] = theta_c and
// cp[nc + c] = 1 (Ritz column) or 0 (plain column):
//   Ritz : R = AV - theta V, E0 = 0, E1 = e1 * R
//   plain: R = 0,            E0 = V, E1 = g2*(g1*AV + V)
// E0, E1, R are FP32 blocks of the same ld.
__global__ __launch_bounds__(kThreads) void mixed_start_kernel(
    int64_t n, const double* __restrict__ V, const double* __restrict__ AV, int ld, int nc,
    const double* __restrict__ cp, double e1, double g1, double g2, float* __restrict__ E0,
    float* __restrict__ E1, float* __restrict__ R) {
  const int64_t e = blockIdx.x * (int64_t)kThreads + threadIdx.x;
  const int64_t i = e / nc;
  const int c = (int)(e % nc);
  if (i >= n) return;
  const int64_t k = i * ld + c;
  float e0, e1v, r;
  mixed_start_elem(V[k], AV[k], cp[c], cp[nc + c], e1, g1, g2, e0, e1v, r);
  R[k] = r;
  E0[k] = e0;
  E1[k] = e1v;
}

// V <- s * (um[c] * V + E), c < nc (E FP32).
__global__ __launch_bounds__(kThreads) void mixed_combine_kernel(int64_t n, double* V, int ld,
                                                                 int nc, const double* __restrict__ um,
                                                                 double s, const float* __restrict__ E) {
  const int64_t e = blockIdx.x * (int64_t)kThreads + threadIdx.x;
  const int64_t i = e / nc;
  const int c = (int)(e % nc);
  if (i >= n) return;
  const int64_t k = i * ld + c;
  V[k] = s * fma(um[c], V[k], double(E[k]));
}

__global__ __launch_bounds__(kThreads) void to_f32_kernel(int64_t n, const double* __restrict__ x,
                                                          float* __restrict__ y) {
  const int64_t i = blockIdx.x * (int64_t)kThreads + threadIdx.x;
  if (i < n) y[i] = float(x[i]);
}

// ------------------------------------------------------- complex helpers
// Complex block columns are pairs of real columns (re, im).  Start vectors:
// complex column c0+j, row i takes draws counter + 2(j*n + i) + {0 re, 1 im}.
__global__ __launch_bounds__(kThreads) void randomize_cplx_kernel(int64_t n, double* X, int ld,
                                                                  int c0, int cnt, uint64_t key,
                                                                  uint64_t counter) {
  const int64_t e = blockIdx.x * (int64_t)kThreads + threadIdx.x;
  const int64_t i = e / (2 * cnt);
  const int r = (int)(e % (2 * cnt));
  if (i >= n) return;
  const int j = r >> 1;
  const int part = r & 1;
  X[i * ld + 2 * (c0 + j) + part] =
      sym_draw(key, counter + 2 * ((uint64_t)j * (uint64_t)n + (uint64_t)i) + (uint64_t)part);
}

// s[2c] = s[2c+1] = s[2c] + s[2c+1], c < nc: squared norms of complex columns
// from those of their real and imaginary parts.
__global__ void pair_sums_kernel(double* s, int nc) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nc) return;
  const double t = s[2 * c] + s[2 * c + 1];
  s[2 * c] = t;
  s[2 * c + 1] = t;
}

// In place, per 2x2 block: the real Gram G~ = Y~^T V~ of interleaved complex
// blocks (2f x 2b, column-major, ld 2f) becomes the real embedding of
// C = Y^H V, so that V~ C~ is the interleaved form of V C:
//   C = (G~[2a,2c] + G~[2a+1,2c+1]) + i (G~[2a,2c+1] - G~[2a+1,2c]),
//   C~[2a,2c] = C~[2a+1,2c+1] = Re C, C~[2a,2c+1] = Im C, C~[2a+1,2c] = -Im C.
__global__ void herm_embed_kernel(double* G, int f, int b) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= f * b) return;
  const int a = e % f;
  const int c = e / f;
  const int64_t ld = 2 * f;
  double* g00 = G + 2 * a + (int64_t)(2 * c) * ld;
  double* g10 = g00 + 1;
  double* g01 = G + 2 * a + (int64_t)(2 * c + 1) * ld;
  double* g11 = g01 + 1;
  const double re = *g00 + *g11;
  const double im = *g01 - *g10;
  *g00 = re;
  *g11 = re;
  *g01 = im;
  *g10 = -im;
}

// ----------------------------------------------------------------- Lanczos
// rows per partial block of the Lanczos kernels: 256, a row per thread, below 2^17
// rows (more blocks for small operators), then 512, and 2048 from 2^20 (fewer
// partials to reduce)
inline int64_t lz_rows(int64_t n) {
  return n >= (int64_t(1) << 20) ? 2048 : (n >= (int64_t(1) << 17) ? 512 : kThreads);
}

__device__ __forceinline__ double block_sum(double v, double* red) {
  red[threadIdx.x] = v;
  __syncthreads();
  for (int s = kThreads / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  const double r = red[0];
  __syncthreads();
  return r;
}

// v = v/||v||, w = v, v = 0 (LanczosMaxMinFinder.h:272-279) -- two phases.
__global__ __launch_bounds__(kThreads) void lz_sumsq_kernel(int64_t n, const double* v, double* P, int64_t rpb) {
  __shared__ double red[kThreads];
  const int64_t i0 = blockIdx.x * rpb;
  const int64_t i1 = min(n, i0 + rpb);
  double s = 0.0;
  for (int64_t i = i0 + threadIdx.x; i < i1; i += kThreads) s += v[i] * v[i];
  s = block_sum(s, red);
  if (threadIdx.x == 0) P[blockIdx.x] = s;
}
__global__ __launch_bounds__(kThreads) void lz_finalize_kernel(const double* P, int64_t nblk,
                                                               double* out, int take_sqrt) {
  __shared__ double red[kThreads];
  // fixed-order: each thread sums a strided subset, then a tree.
  double s = 0.0;
  for (int64_t b = threadIdx.x; b < nblk; b += kThreads) s += P[b];
  s = block_sum(s, red);
  if (threadIdx.x == 0) *out = take_sqrt ? sqrt(fabs(s)) : s;
}
__global__ __launch_bounds__(kThreads) void lz_init_kernel(int64_t n, double* v, double* w,
                                                           const double* nrm) {
  const int64_t i = blockIdx.x * (int64_t)kThreads + threadIdx.x;
  if (i >= n) return;
  const double s = 1.0 / *nrm;
  w[i] = v[i] * s;
  v[i] = 0.0;
}
// if |beta| > 1e-14: w <- v/beta, v <- -beta*w_old (LanczosMaxMinFinder.h:329-339)
__global__ __launch_bounds__(kThreads) void lz_swap_kernel(int64_t n, double* v, double* w,
                                                           const double* beta_prev) {
  const double b = *beta_prev;
  if (!(fabs(b) > 1.0e-14)) return;
  const int64_t i = blockIdx.x * (int64_t)kThreads + threadIdx.x;
  if (i >= n) return;
  const double t = w[i];
  w[i] = v[i] * (1.0 / b);
  v[i] = t * (-b);
}
// v += A w; partial dot(w, v)
__global__ __launch_bounds__(kThreads) void lz_apply_dot_kernel(int64_t n,
                                                                const int* __restrict__ rowptr,
                                                                const int* __restrict__ col,
                                                                const double* __restrict__ val,
                                                                const double* __restrict__ w,
                                                                double* v, double* P, int64_t rpb) {
  __shared__ double red[kThreads];
  const int64_t i0 = blockIdx.x * rpb;
  const int64_t i1 = min(n, i0 + rpb);
  double s = 0.0;
  for (int64_t i = i0 + threadIdx.x; i < i1; i += kThreads) {
    double a = 0.0;
    for (int p = rowptr[i]; p < rowptr[i + 1]; ++p) a = fma(val[p], w[col[p]], a);
    const double vn = v[i] + a;
    v[i] = vn;
    s = fma(w[i], vn, s);
  }
  s = block_sum(s, red);
  if (threadIdx.x == 0) P[blockIdx.x] = s;
}
// complex: v += A w (interleaved re, im), partials of Re and Im of sum conj(w) v
__global__ __launch_bounds__(kThreads) void lz_apply_dot_c_kernel(
    int64_t n, const int* __restrict__ rowptr, const int* __restrict__ col,
    const double* __restrict__ val, const double* __restrict__ w, double* v, double* P,
    int64_t nblk, int64_t rpb) {
  __shared__ double red[kThreads];
  const int64_t i0 = blockIdx.x * rpb;
  const int64_t i1 = min(n, i0 + rpb);
  double sr = 0.0, si = 0.0;
  for (int64_t i = i0 + threadIdx.x; i < i1; i += kThreads) {
    double ar = 0.0, ai = 0.0;
    for (int p = rowptr[i]; p < rowptr[i + 1]; ++p) {
      const double vr = val[2 * (int64_t)p], vi = val[2 * (int64_t)p + 1];
      const double xr = w[2 * (int64_t)col[p]], xi = w[2 * (int64_t)col[p] + 1];
      ar = fma(vr, xr, fma(-vi, xi, ar));
      ai = fma(vr, xi, fma(vi, xr, ai));
    }
    const double nr = v[2 * i] + ar, ni = v[2 * i + 1] + ai;
    v[2 * i] = nr;
    v[2 * i + 1] = ni;
    const double wr = w[2 * i], wi = w[2 * i + 1];
    sr = fma(wr, nr, fma(wi, ni, sr));
    si = fma(wr, ni, fma(-wi, nr, si));
  }
  sr = block_sum(sr, red);
  si = block_sum(si, red);
  if (threadIdx.x == 0) {
    P[blockIdx.x] = sr;
    P[nblk + blockIdx.x] = si;
  }
}

// partial sum w . v (the dense operator's Lanczos alpha)
__global__ __launch_bounds__(kThreads) void lz_dot_kernel(int64_t n, const double* w,
                                                          const double* v, double* P, int64_t rpb) {
  __shared__ double red[kThreads];
  const int64_t i0 = blockIdx.x * rpb;
  const int64_t i1 = min(n, i0 + rpb);
  double s = 0.0;
  for (int64_t i = i0 + threadIdx.x; i < i1; i += kThreads) s = fma(w[i], v[i], s);
  s = block_sum(s, red);
  if (threadIdx.x == 0) P[blockIdx.x] = s;
}

// v += (-alpha) w; partial |v|^2
__global__ __launch_bounds__(kThreads) void lz_axpy_norm_kernel(int64_t n, const double* w,
                                                                double* v, const double* alpha,
                                                                double* P, int64_t rpb) {
  __shared__ double red[kThreads];
  const double a = -*alpha;
  const int64_t i0 = blockIdx.x * rpb;
  const int64_t i1 = min(n, i0 + rpb);
  double s = 0.0;
  for (int64_t i = i0 + threadIdx.x; i < i1; i += kThreads) {
    const double vn = fma(w[i], a, v[i]);
    v[i] = vn;
    s = fma(vn, vn, s);
  }
  s = block_sum(s, red);
  if (threadIdx.x == 0) P[blockIdx.x] = s;
}

// The block's partial sum goes to P[blockIdx.x]; the last block to finish
// (counted on *cnt, which it resets) adds the partials in block order -- the
// order lz_finalize_kernel uses -- and writes the total (or its square root).
// No block waits for another.
__device__ void last_block_total(double s, double* P, unsigned* cnt, double* out, int take_sqrt,
                                 double* red) {
  __shared__ int am_last;
  if (threadIdx.x == 0) {
    P[blockIdx.x] = s;
    __threadfence();
    const unsigned t = atomicAdd(cnt, 1u);
    am_last = (t == gridDim.x - 1);
  }
  __syncthreads();
  if (!am_last) return;
  __threadfence();
  double a = 0.0;
  for (int64_t b = threadIdx.x; b < (int64_t)gridDim.x; b += kThreads) a += P[b];
  a = block_sum(a, red);
  if (threadIdx.x == 0) {
    *out = take_sqrt ? sqrt(fabs(a)) : a;
    *cnt = 0u;
  }
}

// One Lanczos step on a ping-pong pair of vectors (LanczosMaxMinFinder.h:
// 300-345), for real CSR operators.  The previous step's swap (when
// |beta_{k-1}| > 1e-14: w' = v / beta, v' = -beta w) is folded into the
// operator application, whose gathers read v / beta directly; the result
// goes to the other pair (vn = v' + A w', wn = w'), and alpha_k = w' . vn.
// Same arithmetic, in the same order, as lz_swap + lz_apply_dot + finalize.
__global__ __launch_bounds__(kThreads) void lz_step_kernel(
    int64_t n, const int* __restrict__ rowptr, const int* __restrict__ col,
    const double* __restrict__ val, const double* __restrict__ v, const double* __restrict__ w,
    double* __restrict__ vn, double* __restrict__ wn, const double* beta_prev, double* P,
    unsigned* cnt, double* alpha_k, int64_t rpb) {
  __shared__ double red[kThreads];
  const double b = beta_prev ? *beta_prev : 0.0;
  const bool sw = beta_prev != nullptr && fabs(b) > 1.0e-14;
  const double rb = sw ? 1.0 / b : 1.0;
  const int64_t i0 = blockIdx.x * rpb;
  const int64_t i1 = min(n, i0 + rpb);
  double s = 0.0;
  for (int64_t i = i0 + threadIdx.x; i < i1; i += kThreads) {
    const double a = sw ? lz_row<true>(rowptr, col, val, v, i, rb)
                        : lz_row<false>(rowptr, col, val, w, i, 1.0);
    const double wi = sw ? v[i] * rb : w[i];
    const double vi = sw ? w[i] * (-b) : v[i];
    const double vnew = vi + a;
    vn[i] = vnew;
    wn[i] = wi;
    s = fma(wi, vnew, s);
  }
  s = block_sum(s, red);
  last_block_total(s, P, cnt, alpha_k, 0, red);
}

// v -= alpha w; beta_k = ||v|| (lz_axpy_norm + finalize in one launch)
__global__ __launch_bounds__(kThreads) void lz_axpy_beta_kernel(int64_t n, const double* w,
                                                                double* v, const double* alpha,
                                                                double* P, unsigned* cnt,
                                                                double* beta_k, int64_t rpb) {
  __shared__ double red[kThreads];
  const double a = -*alpha;
  const int64_t i0 = blockIdx.x * rpb;
  const int64_t i1 = min(n, i0 + rpb);
  double s = 0.0;
  for (int64_t i = i0 + threadIdx.x; i < i1; i += kThreads) {
    const double vn = fma(w[i], a, v[i]);
    v[i] = vn;
    s = fma(vn, vn, s);
  }
  s = block_sum(s, red);
  last_block_total(s, P, cnt, beta_k, 1, red);
}

inline unsigned grid_for(int64_t work) {
  return (unsigned)((work + kThreads - 1) / kThreads);
}

}  // namespace

// ============================================================== launchers
template <typename T>
void launch_csr_apply(int64_t n, const int* rowptr, const int* col, const T* val, const T* X,
                      T* out, int ld, int ncols, T alpha, T beta, hipStream_t st,
                      const CsrSched* sc, bool cx) {
  if (n <= 0 || ncols <= 0) return;
  if (beta == T(0))
    csr_launch<T, kApply>(n, rowptr, col, val, X, nullptr, out, ld, ncols, alpha, T(0), T(0), st, sc,
                          nullptr, nullptr, cx);
  else
    csr_launch<T, kApplyBeta>(n, rowptr, col, val, X, nullptr, out, ld, ncols, alpha, beta, T(0), st,
                              sc, nullptr, nullptr, cx);
}

void launch_csr_apply_start(int64_t n, const int* rowptr, const int* col, const double* val,
                            const double* V, int ld, int ncols, const MixedArgs& ms,
                            hipStream_t st, const CsrSched* sc, bool cx) {
  if (n <= 0 || ncols <= 0) return;
  if (ms.nc != ncols || !ms.cp || !ms.e0 || !ms.e1 || !ms.r)
    throw Error(1, "fused start: coefficient table and FP32 blocks must cover the call's columns");
  csr_launch<double, kApplyStart>(n, rowptr, col, val, V, nullptr, nullptr, ld, ncols, 1.0, 0.0,
                                  0.0, st, sc, nullptr, nullptr, cx, ms);
}

template <typename T>
void launch_cheb_step(int64_t n, const int* rowptr, const int* col, const T* val, const T* X1,
                      const T* X0, T* out, int ld, int ncols, T g1, T g2, T s, bool first,
                      hipStream_t st, int panel, const CsrSched* sc, bool cx) {
  if (n <= 0 || ncols <= 0) return;
  // Column panels: each launch streams the CSR arrays once and touches only
  // `panel` columns of every row, which shrinks the per-plane footprint of
  // the gathered block so that neighbour rows stay in L2 between uses.
  if (panel <= 0 || panel >= ncols || (sc && sc->tile)) panel = ncols;
  if (panel % 4 != 0) panel = round_up(panel, 4);
  for (int c0 = 0; c0 < ncols; c0 += panel) {
    const int pc = std::min(panel, ncols - c0);
    if (first)
      csr_launch<T, kChebFirst>(n, rowptr, col, val, X1 + c0, nullptr, out + c0, ld, pc, g1, g2, s,
                                st, sc, nullptr, nullptr, cx);
    else
      csr_launch<T, kCheb>(n, rowptr, col, val, X1 + c0, X0 + c0, out + c0, ld, pc, g1, g2, s, st,
                           sc, nullptr, nullptr, cx);
  }
}

void launch_cheb_step_src(int64_t n, const int* rowptr, const int* col, const float* val,
                          const float* X1, const float* X0, float* out, const float* R,
                          const float* kap, int ld, int ncols, float g1, float g2, float s,
                          hipStream_t st, int panel, const CsrSched* sc, bool cx) {
  if (n <= 0 || ncols <= 0) return;
  if (panel <= 0 || panel >= ncols || (sc && sc->tile)) panel = ncols;
  if (panel % 4 != 0) panel = round_up(panel, 4);
  for (int c0 = 0; c0 < ncols; c0 += panel) {
    const int pc = std::min(panel, ncols - c0);
    csr_launch<float, kChebSrc>(n, rowptr, col, val, X1 + c0, X0 + c0, out + c0, ld, pc, g1, g2, s,
                                st, sc, R + c0, kap + c0, cx);
  }
}

void launch_cheb_step_src_end(int64_t n, const int* rowptr, const int* col, const float* val,
                              const float* X1, const float* X0, const float* R, const float* kap,
                              int ld, int ncols, float g1, float g2, const MixedArgs& end,
                              hipStream_t st, int panel, const CsrSched* sc, bool cx) {
  if (n <= 0 || ncols <= 0) return;
  if (!end.v_end || !end.um) throw Error(1, "fused recombination: V and um are required");
  if (panel <= 0 || panel >= ncols || (sc && sc->tile)) panel = ncols;
  if (panel % 4 != 0) panel = round_up(panel, 4);
  for (int c0 = 0; c0 < ncols; c0 += panel) {
    const int pc = std::min(panel, ncols - c0);
    MixedArgs e = end;
    e.v_end = end.v_end + c0;
    e.um = end.um + c0;
    csr_launch<float, kChebSrcEnd>(n, rowptr, col, val, X1 + c0, X0 + c0, nullptr, ld, pc, g1, g2,
                                   1.0f, st, sc, R + c0, kap + c0, cx, e);
  }
}

void launch_mixed_start(int64_t n, const double* V, const double* AV, int ld, int nc,
                        const double* cp, double e1, double g1, double g2, float* E0, float* E1,
                        float* R, hipStream_t st) {
  if (n <= 0 || nc <= 0) return;
  const int64_t tot = n * nc;
  hipLaunchKernelGGL(mixed_start_kernel, dim3((unsigned)((tot + kThreads - 1) / kThreads)),
                     dim3(kThreads), 0, st, n, V, AV, ld, nc, cp, e1, g1, g2, E0, E1, R);
  RCG_HIP(hipGetLastError());
}

void launch_mixed_combine(int64_t n, double* V, int ld, int nc, const double* um, double s,
                          const float* E, hipStream_t st) {
  if (n <= 0 || nc <= 0) return;
  const int64_t tot = n * nc;
  hipLaunchKernelGGL(mixed_combine_kernel, dim3((unsigned)((tot + kThreads - 1) / kThreads)),
                     dim3(kThreads), 0, st, n, V, ld, nc, um, s, E);
  RCG_HIP(hipGetLastError());
}

void launch_to_f32(int64_t n, const double* x, float* y, hipStream_t st) {
  if (n <= 0) return;
  hipLaunchKernelGGL(to_f32_kernel, dim3((unsigned)((n + kThreads - 1) / kThreads)), dim3(kThreads),
                     0, st, n, x, y);
  RCG_HIP(hipGetLastError());
}

inline int64_t dense_tiles(int64_t n, int64_t ncols, int bm, int bn) {
  return ((n + bm - 1) / bm) * ((ncols + bn - 1) / bn);
}
// K splits of an FP64 dense step: with fewer tiles than the two workgroups that a
// CU holds, the tiles' K ranges are cut (at least 8 chunks each) and summed by a
// second kernel.  n = 2048, b = 64 (16 tiles): 157 -> 21.5 us; n = 700, b = 48: 59 ->
// 17; n = 6547, b = 119 (104 tiles): 499 -> 256.  The sizes alone decide, so that
// the order of the sums, and with it the bits, never depends on what a workspace
// happens to hold.
inline int dense_splits(int64_t n, int64_t ncols) {
  const int64_t fill = 512 / dense_tiles(n, ncols, DenseCfg<double>::BM, DenseCfg<double>::BN);
  const int64_t depth = n / (8 * DenseCfg<double>::BK);
  return (int)std::max<int64_t>(1, std::min({fill, depth, (int64_t)32}));
}
size_t dense_ws_elems(int64_t n, int ncols) {
  // fewer columns can take more splits: the most columns of every number of tiles
  size_t most = 0;
  for (int64_t c = 0; c < ncols;) {
    c = std::min<int64_t>(ncols, c + DenseCfg<double>::BN);
    const int s = dense_splits(n, c);
    if (s > 1) most = std::max(most, (size_t)s * (size_t)n * (size_t)c);
  }
  return most;
}

template <typename T>
void launch_dense_step(int64_t n, const T* A, int64_t lda, const T* X, const T* Z, T* out, int ld,
                       int ncols, T p0, T p1, T p2, int mode, const T* R, const T* kap,
                       hipStream_t st, T* ws, size_t ws_elems) {
  if (n <= 0 || ncols <= 0) return;
  if constexpr (std::is_same<T, double>::value) {
    if (ncols == 1 && ld == 1 && (mode == kApply || mode == kApplyBeta)) {
      const dim3 g1((unsigned)((n + kThreads / 64 - 1) / (kThreads / 64)));
      if (mode == kApply)
        hipLaunchKernelGGL(dense_gemv_kernel<kApply>, g1, dim3(kThreads), 0, st, n, A, lda, X,
                           out, p0, p1);
      else
        hipLaunchKernelGGL(dense_gemv_kernel<kApplyBeta>, g1, dim3(kThreads), 0, st, n, A, lda, X,
                           out, p0, p1);
      RCG_HIP(hipGetLastError());
      return;
    }
  }
  const int ntn = (ncols + DenseCfg<T>::BN - 1) / DenseCfg<T>::BN;
  const int64_t tiles = dense_tiles(n, ncols, DenseCfg<T>::BM, DenseCfg<T>::BN);
  if constexpr (std::is_same<T, double>::value) {
    const int nsplit = dense_splits(n, ncols);
    // as many columns at a time as the workspace holds the partial products of: all
    // of them where dense_ws_elems was reserved; fewer change no bits
    const int64_t room = (int64_t)(ws_elems / ((size_t)nsplit * (size_t)n));
    const int cper = room >= ncols ? ncols : (int)(room / 4 * 4);
    if (ws && nsplit > 1 && cper > 0 && mode != kChebSrc) {
      for (int c0 = 0; c0 < ncols; c0 += cper) {
        const int c1 = std::min(ncols, c0 + cper);
        const int tn = (c1 - c0 + DenseCfg<T>::BN - 1) / DenseCfg<T>::BN;
        const int64_t wgs = dense_tiles(n, c1 - c0, DenseCfg<T>::BM, DenseCfg<T>::BN) * nsplit;
        hipLaunchKernelGGL((dense_step_kernel<T, kDensePartial>),
                           dim3((unsigned)round_up(wgs, kXcds)), dim3(kThreads), 0, st, n, A, lda,
                           X, Z, out, ld, c1, p0, p1, p2, R, kap, c0, tn, nsplit, ws);
        RCG_HIP(hipGetLastError());
        const dim3 g3((unsigned)((n * (c1 - c0) + kThreads - 1) / kThreads));
#define RCG_COMBINE(M)                                                                           \
  hipLaunchKernelGGL(dense_combine_kernel<M>, g3, dim3(kThreads), 0, st, n, ws, nsplit, X, Z, out, \
                     ld, c0, c1, p0, p1, p2)
        switch (mode) {
          case kApply: RCG_COMBINE(kApply); break;
          case kApplyBeta: RCG_COMBINE(kApplyBeta); break;
          case kChebFirst: RCG_COMBINE(kChebFirst); break;
          case kCheb: RCG_COMBINE(kCheb); break;
          default: throw Error(1, "unknown dense step mode");
        }
#undef RCG_COMBINE
        RCG_HIP(hipGetLastError());
      }
      return;
    }
  }
  const dim3 grid((unsigned)round_up(tiles, kXcds));
#define RCG_DENSE(M)                                                                           \
  hipLaunchKernelGGL((dense_step_kernel<T, M>), grid, dim3(kThreads), 0, st, n, A, lda, X, Z, out, \
                     ld, ncols, p0, p1, p2, R, kap, 0, ntn, 1, (T*)nullptr)
  switch (mode) {
    case kApply: RCG_DENSE(kApply); break;
    case kApplyBeta: RCG_DENSE(kApplyBeta); break;
    case kChebFirst: RCG_DENSE(kChebFirst); break;
    case kCheb: RCG_DENSE(kCheb); break;
    case kChebSrc: RCG_DENSE(kChebSrc); break;
    default: throw Error(1, "unknown dense step mode");
  }
#undef RCG_DENSE
  RCG_HIP(hipGetLastError());
}

template <typename T>
size_t gram_ws_elems(int64_t n, int bx, int by) {
  int64_t rpb;
  const int64_t nblk = gram_blocks<T>(n, bx, by, &rpb);
  return (size_t)nblk * bx * by;
}

// Upper bound of gram_ws_elems over every bx, by <= bmax: a launch has at
// most 1024/ntiles + 1 row blocks (and at most ceil(n/kRb)), each holding at
// most ntiles 64x64 tiles.
size_t gram_ws_bound(int64_t n, int bmax) {
  const int64_t t = (bmax + kTile - 1) / kTile;
  const int64_t by_tiles = (1024 + t * t) * (int64_t)kTile * kTile;
  const int64_t by_rows = ((n + kRb - 1) / kRb) * (int64_t)bmax * bmax;
  return (size_t)std::max<int64_t>(1, std::min(by_tiles, by_rows));
}

// 16x16 subtiles per side of a one-tile Gram launch
inline int gram_nt(int bx, int by) { return (std::max(bx, by) + 15) / 16; }
template <int MODE>
void gram_one_tile(int nt, dim3 grid, hipStream_t st, int64_t n, const double* X, int ldx, int bx,
                   const double* Y, int ldy, int by, double* P, int64_t rpb, int nta, int ntiles,
                   int64_t nblk) {
#define RCG_GRAM_NT(NT)                                                                          \
  case NT:                                                                                       \
    hipLaunchKernelGGL((gram_mfma_kernel<MODE, NT>), grid, dim3(kThreads), 0, st, n, X, ldx, bx, \
                       Y, ldy, by, P, rpb, nta, ntiles, nblk);                                   \
    break;
  switch (nt) {
    RCG_GRAM_NT(1)
    RCG_GRAM_NT(2)
    RCG_GRAM_NT(3)
    RCG_GRAM_NT(4)
    default: throw Error(1, "one-tile Gram launches take at most 64 columns");
  }
#undef RCG_GRAM_NT
}

template <typename T>
void launch_gram(int64_t n, const T* X, int ldx, int bx, const T* Y, int ldy, int by, T* G,
                 T* ws, size_t ws_elems, hipStream_t st, bool lower_only) {
  if (bx <= 0 || by <= 0) return;
  if (n <= 0) {
    RCG_HIP(hipMemsetAsync(G, 0, sizeof(T) * bx * by, st));
    return;
  }
  int64_t rpb;
  int64_t nblk = gram_blocks<T>(n, bx, by, &rpb);
  if ((size_t)nblk * bx * by > ws_elems) throw Error(3, "gram workspace too small");
  const int nta = (bx + kTile - 1) / kTile;
  const int ntb = (by + kTile - 1) / kTile;
  const int ntiles = nta * ntb;
  if constexpr (std::is_same<T, double>::value) {
    const bool sym = X == Y && bx == by && ldx == ldy;
    if (ntiles > 1) {
      // LDS-staged tiles; the launched tiles times the row blocks fill two
      // workgroups per CU of a 256-CU part once
      const bool low = !sym && lower_only && bx == by;
      const int nl = (sym || low) ? nta * (nta + 1) / 2 : ntiles;
      const int64_t target = std::max<int64_t>(1, 512 / nl);
      rpb = round_up((n + target - 1) / target, kRb);
      rpb = std::max<int64_t>(rpb, round_up(4 * (int64_t)std::max(bx, by), kRb));
      nblk = (n + rpb - 1) / rpb;
      if ((size_t)nblk * bx * by > ws_elems) throw Error(3, "gram workspace too small");
      const dim3 grid((unsigned)round_up(nblk * nl, kXcds));
      if (sym)
        hipLaunchKernelGGL(gram_lds_kernel<kGramSym>, grid, dim3(kThreads), 0, st, n, X, ldx, bx,
                           Y, ldy, by, ws, rpb, nta, nl, nblk);
      else if (low)
        hipLaunchKernelGGL(gram_lds_kernel<kGramLower>, grid, dim3(kThreads), 0, st, n, X, ldx, bx,
                           Y, ldy, by, ws, rpb, nta, nl, nblk);
      else
        hipLaunchKernelGGL(gram_lds_kernel<kGramFull>, grid, dim3(kThreads), 0, st, n, X, ldx, bx,
                           Y, ldy, by, ws, rpb, nta, nl, nblk);
    } else if (sym) {
      gram_one_tile<kGramDiag>(gram_nt(bx, by), dim3((unsigned)round_up(nblk, kXcds)), st, n, X,
                               ldx, bx, Y, ldy, by, ws, rpb, nta, 1, nblk);
    } else {
      gram_one_tile<kGramFull>(gram_nt(bx, by), dim3((unsigned)round_up(nblk * ntiles, kXcds)), st,
                               n, X, ldx, bx, Y, ldy, by, ws, rpb, nta, ntiles, nblk);
    }
  } else {
    hipLaunchKernelGGL(gram_partial_kernel<T>, dim3((unsigned)nblk, ntiles), dim3(kThreads), 0, st,
                       n, X, ldx, bx, Y, ldy, by, ws, rpb, ntiles);
  }
  RCG_HIP(hipGetLastError());
  const int64_t m = (int64_t)bx * by;
  hipLaunchKernelGGL((reduce_partials_kernel<T, T>), dim3(reduce_grid(m)), dim3(kThreads), 0, st, ws,
                     nblk, m, G);
  RCG_HIP(hipGetLastError());
}

// One workgroup reads all partials: up to 2^16 (0.5 MB) that is no slower than
// the workgroups of a reduction of its own.
bool chol_fits(int64_t n, int b) {
  int64_t rpb;
  return n > 0 && b >= 1 && b <= kCholMax && gram_blocks<double>(n, b, b, &rpb) * b * b <= 65536;
}

void launch_gram_chol(int64_t n, const double* X, int ldx, int b, double* C, double* inv2,
                      double* ws, size_t ws_elems, hipStream_t st) {
  if (!chol_fits(n, b)) throw Error(1, "block too large for the device factor");
  int64_t rpb;
  const int64_t nblk = gram_blocks<double>(n, b, b, &rpb);
  if ((size_t)nblk * b * b > ws_elems) throw Error(3, "gram workspace too small");
  gram_one_tile<kGramDiag>(gram_nt(b, b), dim3((unsigned)round_up(nblk, kXcds)), st, n, X, ldx, b,
                           X, ldx, b, ws, rpb, 1, 1, nblk);
  RCG_HIP(hipGetLastError());
#define RCG_CHOL(B)                                                                              \
  hipLaunchKernelGGL(reduce_chol_kernel<B>, dim3(1), dim3(kCholThreads), 0, st, ws, nblk, b, C, \
                     inv2)
  if (b <= 16) RCG_CHOL(16);
  else if (b <= 24) RCG_CHOL(24);
  else RCG_CHOL(32);
#undef RCG_CHOL
  RCG_HIP(hipGetLastError());
}

void launch_gram_pair(int64_t n, const double* X, int ldx, const double* Y, int ldy, int b,
                      double* G, double* ws, size_t ws_elems, hipStream_t st) {
  if (b <= 0) return;
  if (b > kTile) throw Error(1, "paired Gram products take at most 64 columns");
  if (n <= 0) {
    RCG_HIP(hipMemsetAsync(G, 0, sizeof(double) * 2 * b * b, st));
    return;
  }
  // the row blocks of the single launches, so that the partials and their
  // sums are the same
  int64_t rpb;
  const int64_t nblk = gram_blocks<double>(n, b, b, &rpb);
  if ((size_t)(2 * nblk) * b * b > ws_elems) throw Error(3, "gram workspace too small");
  gram_one_tile<kGramPair>(gram_nt(b, b), dim3((unsigned)round_up(2 * nblk, kXcds)), st, n, X, ldx,
                          b, Y, ldy, b, ws, rpb, 1, 2, nblk);
  RCG_HIP(hipGetLastError());
  const int64_t m = 2 * (int64_t)b * b;
  hipLaunchKernelGGL((reduce_partials_kernel<double, double>), dim3(reduce_grid(m)), dim3(kThreads),
                     0, st, ws, nblk, m, G);
  RCG_HIP(hipGetLastError());
}

namespace {
// Workgroups of the wide tall product: C slice resident in LDS (66.5, 100 or
// 133 KB) and about 300 registers per lane, one workgroup per CU, persistent
// over 128-row tiles.
int64_t wide_stripes(int64_t n, int ct) {
  const int64_t nrt = (n + 2 * kTile - 1) / (2 * kTile);
  return std::max<int64_t>(1, std::min<int64_t>(nrt, 256 / (int64_t)ct));
}
// Workgroups of the narrow one, persistent over 64-row tiles: as many as fit at
// once on a 256-CU part (four per CU, three with the registers that hold beta Z
// or column sums, two with a Gram matrix's).
int64_t tall_stripes(int64_t n, int ct, bool beta, int after) {
  const int64_t wgs = after >= kTallGram ? 512 : (beta || after == kTallSums ? 768 : 1024);
  return std::max<int64_t>(1, std::min<int64_t>((n + kTile - 1) / kTile, wgs / (int64_t)ct));
}
template <bool SUMS>
void tall_wide(int64_t n, const double* X, int ldx, int bx, const double* C, int ldc, int by,
               double alpha, double beta, const double* Z, double* out, int ldo, double* P,
               hipStream_t st) {
  const int ct = (by + kTile - 1) / kTile;
  const int kch = (bx + kTile - 1) / kTile;
  const int64_t nrt = (n + 2 * kTile - 1) / (2 * kTile);
  const int64_t nstripe = wide_stripes(n, ct);
  const dim3 grid((unsigned)round_up(nstripe * ct, kXcds));
#define RCG_WIDE(K)                                                                               \
  hipLaunchKernelGGL((tall_gemm_wide_kernel<K, SUMS>), grid, dim3(kThreads), 0, st, n, X, ldx, bx, \
                     C, ldc, by, alpha, beta, Z, out, ldo, nrt, ct, nstripe, P)
  if (kch == 2) RCG_WIDE(2);
  else if (kch == 3) RCG_WIDE(3);
  else RCG_WIDE(4);
#undef RCG_WIDE
  RCG_HIP(hipGetLastError());
}
template <int AFTER, int NTC, int NTX>
void tall_one(int64_t n, const double* X, int ldx, int bx, const double* C, int ldc, int by,
              double alpha, double beta, const double* Z, double* out, int ldo, double* P,
              hipStream_t st) {
  const int ct = (by + kTile - 1) / kTile;
  const int64_t nrb = (n + kTile - 1) / kTile;
  const int64_t nstripe = tall_stripes(n, ct, beta != 0.0, AFTER);
  const dim3 grid((unsigned)round_up(nstripe * ct, kXcds));
  // out^T out follows products without Z, X^T out the deflation's only
  if constexpr (AFTER != kTallGram)
    if (beta != 0.0)
      hipLaunchKernelGGL((tall_gemm_mfma_kernel<true, NTC, AFTER, NTX>), grid, dim3(kThreads), 0,
                         st, n, X, ldx, bx, C, ldc, by, alpha, beta, Z, out, ldo, nrb, ct, nstripe,
                         P);
  if constexpr (AFTER != kTallCross)
    if (beta == 0.0 || AFTER == kTallGram)
      hipLaunchKernelGGL((tall_gemm_mfma_kernel<false, NTC, AFTER, NTX>), grid, dim3(kThreads), 0,
                         st, n, X, ldx, bx, C, ldc, by, alpha, beta, Z, out, ldo, nrb, ct, nstripe,
                         P);
  RCG_HIP(hipGetLastError());
}
template <int AFTER>
void tall_narrow(int64_t n, const double* X, int ldx, int bx, const double* C, int ldc, int by,
                 double alpha, double beta, const double* Z, double* out, int ldo, double* P,
                 hipStream_t st) {
  const int ntc = by >= kTile ? 4 : (by + 15) / 16;
#define RCG_TALL(NTC, NTX) \
  tall_one<AFTER, NTC, NTX>(n, X, ldx, bx, C, ldc, by, alpha, beta, Z, out, ldo, P, st)
  if constexpr (AFTER == kTallCross) {
    const int ntx = bx <= 16 ? 1 : (bx <= 32 ? 2 : 4);
#define RCG_TALL_X(NTC)               \
  if (ntx == 1) RCG_TALL(NTC, 1);     \
  else if (ntx == 2) RCG_TALL(NTC, 2); \
  else RCG_TALL(NTC, 4);              \
  break;
    switch (ntc) {
      case 1: RCG_TALL_X(1)
      case 2: RCG_TALL_X(2)
      case 3: RCG_TALL_X(3)
      default: RCG_TALL_X(4)
    }
#undef RCG_TALL_X
  } else {
    switch (ntc) {
      case 1: RCG_TALL(1, 1); break;
      case 2: RCG_TALL(2, 2); break;
      case 3: RCG_TALL(3, 3); break;
      default: RCG_TALL(4, 4); break;
    }
  }
#undef RCG_TALL
}
}  // namespace

template <typename T>
void launch_tall_gemm(int64_t n, const T* X, int ldx, int bx, const T* C, int ldc, int by,
                      T alpha, T beta, const T* Z, T* out, int ldo, hipStream_t st) {
  if (n <= 0 || by <= 0) return;
  if constexpr (std::is_same<T, double>::value) {
    if (bx > kTile && bx <= 4 * kTile)
      tall_wide<false>(n, X, ldx, bx, C, ldc, by, alpha, beta, Z, out, ldo, nullptr, st);
    else
      tall_narrow<kTallNone>(n, X, ldx, bx, C, ldc, by, alpha, beta, Z, out, ldo, nullptr, st);
  } else {
    const int64_t nrb = (n + kTile - 1) / kTile;
    const unsigned ct = (unsigned)((by + kTile - 1) / kTile);
    hipLaunchKernelGGL(tall_gemm_kernel<T>, dim3((unsigned)round_up(nrb, kXcds), ct),
                       dim3(kThreads), 0, st, n, X, ldx, bx, C, ldc, by, alpha, beta, Z, out, ldo,
                       nrb);
    RCG_HIP(hipGetLastError());
  }
}

namespace {
void reduce_to(const double* P, int64_t nblk, int64_t m, double* out, hipStream_t st) {
  hipLaunchKernelGGL((reduce_partials_kernel<double, double>), dim3(reduce_grid(m)),
                     dim3(kThreads), 0, st, P, nblk, m, out);
  RCG_HIP(hipGetLastError());
}
}  // namespace

void launch_tall_gemm_sums(int64_t n, const double* X, int ldx, int bx, const double* C, int ldc,
                           int by, double alpha, double beta, const double* Z, double* out, int ldo,
                           double* sums, double* ws, size_t ws_elems, hipStream_t st) {
  if (n <= 0 || by <= 0) return;
  const bool wide = bx > kTile && bx <= 4 * kTile;
  const int ct = (by + kTile - 1) / kTile;
  const int64_t nblk = wide ? wide_stripes(n, ct) : tall_stripes(n, ct, beta != 0.0, kTallSums);
  if ((size_t)(nblk * by) > ws_elems) throw Error(3, "column-sum workspace too small");
  if (wide) tall_wide<true>(n, X, ldx, bx, C, ldc, by, alpha, beta, Z, out, ldo, ws, st);
  else tall_narrow<kTallSums>(n, X, ldx, bx, C, ldc, by, alpha, beta, Z, out, ldo, ws, st);
  reduce_to(ws, nblk, by, sums, st);
}

void launch_tall_resid(int64_t n, const double* V, const double* W, int ld, int b, const double* C,
                       double* out, const ThetaArgs& theta, int nc, double* sums, double* ws,
                       size_t ws_elems, hipStream_t st) {
  if (n <= 0 || b <= 0 || nc <= 0) throw Error(1, "residuals of an empty block");
  if (b > kTile || nc > b) throw Error(1, "fused residuals take at most 64 columns");
  const int64_t nrb = (n + kTile - 1) / kTile;
  const int64_t nblk = std::min<int64_t>(nrb, 512);  // two workgroups per CU
  if ((size_t)(nblk * 2 * nc) > ws_elems) throw Error(3, "column-sum workspace too small");
  const dim3 grid((unsigned)round_up(nblk, kXcds));
  // 16-column subtiles of the block and of its residual columns
#define RCG_RESID(N, R)                                                                            \
  case 10 * N + R:                                                                                 \
    hipLaunchKernelGGL((tall_resid_kernel<N, R>), grid, dim3(kThreads), 0, st, n, V, W, ld, b, C,  \
                       out, theta, nc, nrb, nblk, ws);                                             \
    break;
  switch (10 * ((b + 15) / 16) + (nc + 15) / 16) {
    RCG_RESID(1, 1)
    RCG_RESID(2, 1)
    RCG_RESID(2, 2)
    RCG_RESID(3, 1)
    RCG_RESID(3, 2)
    RCG_RESID(3, 3)
    RCG_RESID(4, 1)
    RCG_RESID(4, 2)
    RCG_RESID(4, 3)
    RCG_RESID(4, 4)
  }
#undef RCG_RESID
  RCG_HIP(hipGetLastError());
  reduce_to(ws, nblk, 2 * nc, sums, st);
}

// A partial per workgroup of 64-row tiles costs the fused forms more than a partial per
// 256 rows costs the Gram launch, until there are more tiles than workgroups; from
// 2^19 rows the Gram launch streams faster than the narrow product's two workgroups
// per CU.  us, fused / apart, out^T out of 8, 32 and 64 columns: n = 4000 9.6 / 11.1,
// 15.1 / 15.9, 23.3 / 27.2; 14000 11.1 / 11.8, 17.4 / 17.6, 27.4 / 29.7; 17576 12.2 / 12.5,
// 21.1 / 18.9, 38.2 / 31.8; 50000 15.8 / 15.0, 30.5 / 24.7, 52.1 / 42.0; 70000 17.1 /
// 17.9, 34.9 / 34.5, 57.5 / 62.2; 200000 24.8 / 32.8, 54.6 / 58.5, 85.9 / 114; 2^20 70 / 62,
// 194 / 193, 292 / 363.
bool tall_gram_pays(int64_t n, int by) {
  return n <= 14336 || (n >= 70000 && (n < (int64_t(1) << 19) || by > 40));
}
// X^T out reads X again, but the Gram launch it replaces reads X and out, and
// multiplies max(bx, by)^2 tiles.  us, fused / apart, 24 x 24, 64 x 16, 20 x 64 and 64 x
// 64 (bx x by): n = 4000 15.7 / 18.3, 14.3 / 31.1, 20.9 / 35.5, 29.3 / 35.9; 20000 23.7 /
// 21.3, 21.7 / 33.5, 34.3 / 39.9, 56.6 / 41.0; 50000 30.6 / 26.7, 27.7 / 38.8, 46.5 / 51.0,
// 75.8 / 54.2; 65536 30.7 / 34.8, 28.0 / 44.2, 48.1 / 60.4, 76.6 / 65.4; 75000 37.7 / 40.5,
// 31.4 / 66.5, 54.3 / 84.3, 87.8 / 88.3; 2^20 x (16 x 24) 209 / 237, (64 x 64) 492 / 575.
// With bx above 32 and 33-48 columns it spills: 48 x 48 at 75000 82.8 / 62.5.
bool tall_cross_pays(int64_t n, int bx, int by) {
  if (n <= 14336) return true;
  if (bx > 32 && by > 32 && by <= 48) return false;
  if (n >= 65536) return !(bx > 32 && by > 48) || n >= 70000;
  return std::max(bx, by) > 48 && std::min(bx, by) <= 32;
}

void launch_tall_gemm_gram(int64_t n, const double* X, int ldx, int bx, const double* C, int ldc,
                           int by, double* out, int ldo, double* G, double* ws, size_t ws_elems,
                           hipStream_t st) {
  if (n <= 0 || by <= 0) return;
  if (bx > kTile || by > kTile) throw Error(1, "fused Gram products take at most 64 columns");
  const int64_t nblk = tall_stripes(n, 1, false, kTallGram), m = (int64_t)by * by;
  if ((size_t)(nblk * m) > ws_elems) throw Error(3, "gram workspace too small");
  tall_narrow<kTallGram>(n, X, ldx, bx, C, ldc, by, 1.0, 0.0, nullptr, out, ldo, ws, st);
  reduce_to(ws, nblk, m, G, st);
}

void launch_tall_gemm_cross(int64_t n, const double* X, int ldx, int bx, const double* C, int ldc,
                            int by, double alpha, const double* Z, double* out, int ldo, double* G,
                            double* ws, size_t ws_elems, hipStream_t st) {
  if (n <= 0 || by <= 0) return;
  if (bx > kTile || by > kTile) throw Error(1, "fused Gram products take at most 64 columns");
  const int64_t nblk = tall_stripes(n, 1, true, kTallCross), m = (int64_t)bx * by;
  if ((size_t)(nblk * m) > ws_elems) throw Error(3, "gram workspace too small");
  tall_narrow<kTallCross>(n, X, ldx, bx, C, ldc, by, alpha, 1.0, Z, out, ldo, ws, st);
  reduce_to(ws, nblk, m, G, st);
}

size_t colred_ws_elems(int64_t n, int nc) {
  return (size_t)((n + kColRows - 1) / kColRows) * (size_t)std::max(nc, 1);
}

template <typename T>
void launch_col_sumsq(int64_t n, const T* X, int ld, int nc, double* sums, double* ws,
                      size_t ws_elems, hipStream_t st) {
  if (nc <= 0) return;
  const int64_t nblk = (n + kColRows - 1) / kColRows;
  if ((size_t)(nblk * nc) > ws_elems) throw Error(3, "column-reduction workspace too small");
  hipLaunchKernelGGL((col_sumsq_kernel<T, false>), dim3((unsigned)nblk), dim3(kThreads), 0, st, n,
                     X, (const T*)nullptr, ld, nc, (const double*)nullptr, ws);
  RCG_HIP(hipGetLastError());
  hipLaunchKernelGGL((reduce_partials_kernel<double, double>), dim3(reduce_grid(nc)), dim3(kThreads),
                     0, st, ws, nblk, (int64_t)nc, sums);
  RCG_HIP(hipGetLastError());
}

template <typename T>
void launch_residual_sumsq(int64_t n, const T* V, const T* W, int ld, int nc, const double* theta,
                           double* sums, double* ws, size_t ws_elems, hipStream_t st) {
  if (nc <= 0) return;
  const int64_t nblk = (n + kColRows - 1) / kColRows;
  if ((size_t)(nblk * nc) > ws_elems) throw Error(3, "column-reduction workspace too small");
  hipLaunchKernelGGL((col_sumsq_kernel<T, true>), dim3((unsigned)nblk), dim3(kThreads), 0, st, n, V,
                     W, ld, nc, theta, ws);
  RCG_HIP(hipGetLastError());
  hipLaunchKernelGGL((reduce_partials_kernel<double, double>), dim3(reduce_grid(nc)), dim3(kThreads),
                     0, st, ws, nblk, (int64_t)nc, sums);
  RCG_HIP(hipGetLastError());
}

__global__ __launch_bounds__(kThreads) void group_sqrt_kernel(const double* __restrict__ sums,
                                                              int cw, int count,
                                                              double* __restrict__ out) {
  const int c = blockIdx.x * kThreads + threadIdx.x;
  if (c >= count) return;
  double t = 0.0;
  for (int e = 0; e < cw; ++e) t += sums[cw * c + e];
  out[c] = sqrt(fabs(t));
}

void launch_group_sqrt(const double* sums, int cw, int count, double* out, hipStream_t st) {
  if (count <= 0) return;
  hipLaunchKernelGGL(group_sqrt_kernel, dim3((unsigned)((count + kThreads - 1) / kThreads)),
                     dim3(kThreads), 0, st, sums, cw, count, out);
  RCG_HIP(hipGetLastError());
}

template <typename T>
void launch_resid_norm_sumsq(int64_t n, const T* V, const T* W, int ld, int nc,
                             const double* theta, double* sums, double* ws, size_t ws_elems,
                             hipStream_t st) {
  if (nc <= 0) return;
  const int64_t nblk = (n + kColRows - 1) / kColRows;
  if ((size_t)(nblk * 2 * nc) > ws_elems) throw Error(3, "column-reduction workspace too small");
  hipLaunchKernelGGL((resid_norm_kernel<T, const double*>), dim3((unsigned)nblk), dim3(kThreads),
                     0, st, n, V, W, ld, nc, theta, ws);
  RCG_HIP(hipGetLastError());
  hipLaunchKernelGGL((reduce_partials_kernel<double, double>), dim3(reduce_grid(2 * nc)),
                     dim3(kThreads), 0, st, ws, nblk, (int64_t)(2 * nc), sums);
  RCG_HIP(hipGetLastError());
}

void launch_resid_norm_sumsq_args(int64_t n, const double* V, const double* W, int ld, int nc,
                                  const ThetaArgs& theta, double* sums, double* ws,
                                  size_t ws_elems, hipStream_t st) {
  if (nc <= 0) return;
  if (nc > kThetaArgs) throw Error(1, "more Ritz values than the argument block holds");
  const int64_t nblk = (n + kColRows - 1) / kColRows;
  if ((size_t)(nblk * 2 * nc) > ws_elems) throw Error(3, "column-reduction workspace too small");
  hipLaunchKernelGGL((resid_norm_kernel<double, ThetaArgs>), dim3((unsigned)nblk), dim3(kThreads),
                     0, st, n, V, W, ld, nc, theta, ws);
  RCG_HIP(hipGetLastError());
  hipLaunchKernelGGL((reduce_partials_kernel<double, double>), dim3(reduce_grid(2 * nc)),
                     dim3(kThreads), 0, st, ws, nblk, (int64_t)(2 * nc), sums);
  RCG_HIP(hipGetLastError());
}

template <typename T>
void launch_normalize_cols(int64_t n, T* X, int ld, int nc, const double* sums, hipStream_t st) {
  if (n <= 0 || nc <= 0) return;
  hipLaunchKernelGGL(normalize_cols_kernel<T>, dim3(grid_for(n * nc)), dim3(kThreads), 0, st, n, X,
                     ld, nc, sums);
  RCG_HIP(hipGetLastError());
}

void launch_scale_cols(int64_t n, const double* X, int ld, int nc, const double* sums, double* out,
                       hipStream_t st) {
  if (n <= 0 || nc <= 0) return;
  hipLaunchKernelGGL(scale_cols_kernel, dim3(grid_for(n * nc)), dim3(kThreads), 0, st, n, X, ld, nc,
                     sums, out);
  RCG_HIP(hipGetLastError());
}

template <typename T>
void launch_copy_cols(int64_t n, const T* src, int lds, int s0, T* dst, int ldd, int d0, int cnt,
                      hipStream_t st) {
  if (n <= 0 || cnt <= 0) return;
  hipLaunchKernelGGL(copy_cols_kernel<T>, dim3(grid_for(n * cnt)), dim3(kThreads), 0, st, n, src,
                     lds, s0, dst, ldd, d0, cnt);
  RCG_HIP(hipGetLastError());
}

template <typename T>
void launch_randomize_cols(int64_t n, T* X, int ld, int c0, int cnt, uint64_t seed,
                           uint64_t counter, hipStream_t st) {
  if (n <= 0 || cnt <= 0) return;
  const uint64_t key = [&] {
    uint64_t z = seed + 0x9E3779B97F4A7C15ULL;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
  }();
  hipLaunchKernelGGL(randomize_cols_kernel<T>, dim3(grid_for(n * cnt)), dim3(kThreads), 0, st, n,
                     X, ld, c0, cnt, key, counter);
  RCG_HIP(hipGetLastError());
}

template <typename T>
void launch_fill_cols(int64_t n, T* X, int ld, int c0, int cnt, T value, hipStream_t st) {
  if (n <= 0 || cnt <= 0) return;
  hipLaunchKernelGGL(fill_cols_kernel<T>, dim3(grid_for(n * cnt)), dim3(kThreads), 0, st, n, X, ld,
                     c0, cnt, value);
  RCG_HIP(hipGetLastError());
}

size_t lz_ws_elems(int64_t n) { return 2 * (size_t)((n + lz_rows(n) - 1) / lz_rows(n)) + 4; }

void launch_lz_dot(int64_t n, const double* w, const double* v, double* out, double* ws,
                   size_t ws_elems, hipStream_t st) {
  const int64_t rpb = lz_rows(n);
  const int64_t nblk = (n + rpb - 1) / rpb;
  if ((size_t)nblk > ws_elems) throw Error(3, "Lanczos workspace too small");
  hipLaunchKernelGGL(lz_dot_kernel, dim3((unsigned)nblk), dim3(kThreads), 0, st, n, w, v, ws, rpb);
  hipLaunchKernelGGL(lz_finalize_kernel, dim3(1), dim3(kThreads), 0, st, ws, nblk, out, 0);
  RCG_HIP(hipGetLastError());
}

void launch_randomize_cplx(int64_t n, double* X, int ld, int c0, int cnt, uint64_t seed,
                           uint64_t counter, hipStream_t st) {
  if (n <= 0 || cnt <= 0) return;
  const uint64_t key = [&] {
    uint64_t z = seed + 0x9E3779B97F4A7C15ULL;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
  }();
  hipLaunchKernelGGL(randomize_cplx_kernel, dim3(grid_for(n * 2 * cnt)), dim3(kThreads), 0, st, n, X,
                     ld, c0, cnt, key, counter);
  RCG_HIP(hipGetLastError());
}

void launch_pair_sums(double* s, int nc, hipStream_t st) {
  if (nc <= 0) return;
  hipLaunchKernelGGL(pair_sums_kernel, dim3((nc + 255) / 256), dim3(256), 0, st, s, nc);
  RCG_HIP(hipGetLastError());
}

void launch_herm_embed(double* G, int f, int b, hipStream_t st) {
  if (f <= 0 || b <= 0) return;
  hipLaunchKernelGGL(herm_embed_kernel, dim3((f * b + 255) / 256), dim3(256), 0, st, G, f, b);
  RCG_HIP(hipGetLastError());
}

void launch_lz_apply_dot_c(int64_t n, const int* rowptr, const int* col, const double* val,
                           const double* w, double* v, double* alpha_k, double* alpha_im_k,
                           double* ws, size_t ws_elems, hipStream_t st) {
  const int64_t rpb = lz_rows(n);
  const int64_t nblk = (n + rpb - 1) / rpb;
  if ((size_t)(2 * nblk) > ws_elems) throw Error(3, "Lanczos workspace too small");
  hipLaunchKernelGGL(lz_apply_dot_c_kernel, dim3((unsigned)nblk), dim3(kThreads), 0, st, n, rowptr,
                     col, val, w, v, ws, nblk, rpb);
  hipLaunchKernelGGL(lz_finalize_kernel, dim3(1), dim3(kThreads), 0, st, ws, nblk, alpha_k, 0);
  hipLaunchKernelGGL(lz_finalize_kernel, dim3(1), dim3(kThreads), 0, st, ws + nblk, nblk, alpha_im_k, 0);
  RCG_HIP(hipGetLastError());
}



void launch_lz_start(int64_t n, double* v, double* w, double* ws, size_t ws_elems,
                     double* scratch, hipStream_t st) {
  const int64_t rpb = lz_rows(n);
  const int64_t nblk = (n + rpb - 1) / rpb;
  if ((size_t)nblk > ws_elems) throw Error(3, "Lanczos workspace too small");
  hipLaunchKernelGGL(lz_sumsq_kernel, dim3((unsigned)nblk), dim3(kThreads), 0, st, n, v, ws, rpb);
  hipLaunchKernelGGL(lz_finalize_kernel, dim3(1), dim3(kThreads), 0, st, ws, nblk, scratch, 1);
  hipLaunchKernelGGL(lz_init_kernel, dim3(grid_for(n)), dim3(kThreads), 0, st, n, v, w, scratch);
  RCG_HIP(hipGetLastError());
}
void launch_lz_swap(int64_t n, double* v, double* w, const double* beta_prev, hipStream_t st) {
  hipLaunchKernelGGL(lz_swap_kernel, dim3(grid_for(n)), dim3(kThreads), 0, st, n, v, w, beta_prev);
  RCG_HIP(hipGetLastError());
}
void launch_lz_apply_dot(int64_t n, const int* rowptr, const int* col, const double* val,
                         const double* w, double* v, double* alpha_k, double* ws, size_t ws_elems,
                         hipStream_t st) {
  const int64_t rpb = lz_rows(n);
  const int64_t nblk = (n + rpb - 1) / rpb;
  if ((size_t)nblk > ws_elems) throw Error(3, "Lanczos workspace too small");
  hipLaunchKernelGGL(lz_apply_dot_kernel, dim3((unsigned)nblk), dim3(kThreads), 0, st, n, rowptr,
                     col, val, w, v, ws, rpb);
  hipLaunchKernelGGL(lz_finalize_kernel, dim3(1), dim3(kThreads), 0, st, ws, nblk, alpha_k, 0);
  RCG_HIP(hipGetLastError());
}
void launch_lz_axpy_norm(int64_t n, const double* w, double* v, const double* alpha_k,
                         double* beta_k, double* ws, size_t ws_elems, hipStream_t st) {
  const int64_t rpb = lz_rows(n);
  const int64_t nblk = (n + rpb - 1) / rpb;
  if ((size_t)nblk > ws_elems) throw Error(3, "Lanczos workspace too small");
  hipLaunchKernelGGL(lz_axpy_norm_kernel, dim3((unsigned)nblk), dim3(kThreads), 0, st, n, w, v,
                     alpha_k, ws, rpb);
  hipLaunchKernelGGL(lz_finalize_kernel, dim3(1), dim3(kThreads), 0, st, ws, nblk, beta_k, 1);
  RCG_HIP(hipGetLastError());
}

void launch_lz_step(int64_t n, const int* rowptr, const int* col, const double* val,
                    const double* v, const double* w, double* vn, double* wn,
                    const double* beta_prev, double* alpha_k, double* beta_k, unsigned* cnt,
                    double* ws, size_t ws_elems, hipStream_t st) {
  const int64_t rpb = lz_rows(n);
  const int64_t nblk = (n + rpb - 1) / rpb;
  if ((size_t)nblk > ws_elems) throw Error(3, "Lanczos workspace too small");
  hipLaunchKernelGGL(lz_step_kernel, dim3((unsigned)nblk), dim3(kThreads), 0, st, n, rowptr, col,
                     val, v, w, vn, wn, beta_prev, ws, cnt, alpha_k, rpb);
  hipLaunchKernelGGL(lz_axpy_beta_kernel, dim3((unsigned)nblk), dim3(kThreads), 0, st, n, wn, vn,
                     alpha_k, ws, cnt, beta_k, rpb);
  RCG_HIP(hipGetLastError());
}

// ------------------------------------------------------- instantiations
// ------------------------------------------ layouts for caller operators
// A caller-supplied operator works on column-major blocks (element (i, c) at
// C[c*ldc + i], the reference's AmatrixClassLMCuda layout); the solver's
// blocks are row-interleaved (element (i, c) at X[i*ldx + c]).  E is one
// block entry: double, or double2 for a complex entry (re, im).  32 x 32
// tiles through LDS keep both sides coalesced.
template <typename E>
struct EntryOps;
template <>
struct EntryOps<double> {
  __device__ static double comb(double p0, double p1, double p2, double ax, double x, double z) {
    return p2 * fma(p1, fma(p0, ax, x), -z);
  }
  __device__ static double zero() { return 0.0; }
};
template <>
struct EntryOps<double2> {
  __device__ static double2 comb(double p0, double p1, double p2, double2 ax, double2 x,
                                 double2 z) {
    return make_double2(p2 * fma(p1, fma(p0, ax.x, x.x), -z.x), p2 * fma(p1, fma(p0, ax.y, x.y), -z.y));
  }
  __device__ static double2 zero() { return make_double2(0.0, 0.0); }
};

constexpr int kLt = 32;  // layout tile

// TO_COLS: rows layout -> column-major; else the reverse.
template <typename E, bool TO_COLS>
__global__ __launch_bounds__(kThreads) void layout_kernel(int64_t n, int cols, E* R, int64_t ldr,
                                                          E* Cm, int64_t ldc) {
  __shared__ E tile[kLt][kLt + 1];
  const int64_t i0 = (int64_t)blockIdx.x * kLt;
  const int c0 = blockIdx.y * kLt;
  const int tx = threadIdx.x % kLt, ty = threadIdx.x / kLt;
  for (int r = ty; r < kLt; r += kThreads / kLt) {
    if (TO_COLS) {  // tile[row][col] from the rows layout
      const int64_t i = i0 + r;
      const int c = c0 + tx;
      if (i < n && c < cols) tile[r][tx] = R[i * ldr + c];
    } else {  // tile[col][row] from the column-major layout
      const int c = c0 + r;
      const int64_t i = i0 + tx;
      if (i < n && c < cols) tile[r][tx] = Cm[(int64_t)c * ldc + i];
    }
  }
  __syncthreads();
  for (int r = ty; r < kLt; r += kThreads / kLt) {
    if (TO_COLS) {
      const int c = c0 + r;
      const int64_t i = i0 + tx;
      if (i < n && c < cols) Cm[(int64_t)c * ldc + i] = tile[tx][r];
    } else {
      const int64_t i = i0 + r;
      const int c = c0 + tx;
      if (i < n && c < cols) R[i * ldr + c] = tile[tx][r];
    }
  }
}

// out = p2 (p1 (p0 AX + X) - Z) in the rows layout, AX column-major (Z may
// be null: no Z term; out may alias Z): the Chebyshev step around a caller
// operator's product, the same expression as the fused CSR step's epilogue.
template <typename E>
__global__ __launch_bounds__(kThreads) void cheb_combine_kernel(int64_t n, int cols,
                                                                const E* __restrict__ AX,
                                                                int64_t ldc, const E* X,
                                                                const E* Z, E* out, int64_t ldr,
                                                                double p0, double p1, double p2) {
  __shared__ E tile[kLt][kLt + 1];
  const int64_t i0 = (int64_t)blockIdx.x * kLt;
  const int c0 = blockIdx.y * kLt;
  const int tx = threadIdx.x % kLt, ty = threadIdx.x / kLt;
  for (int r = ty; r < kLt; r += kThreads / kLt) {
    const int c = c0 + r;
    const int64_t i = i0 + tx;
    if (i < n && c < cols) tile[r][tx] = AX[(int64_t)c * ldc + i];
  }
  __syncthreads();
  for (int r = ty; r < kLt; r += kThreads / kLt) {
    const int64_t i = i0 + r;
    const int c = c0 + tx;
    if (i < n && c < cols) {
      const int64_t o = i * ldr + c;
      const E z = Z ? Z[o] : EntryOps<E>::zero();
      out[o] = EntryOps<E>::comb(p0, p1, p2, tile[tx][r], X[o], z);
    }
  }
}

void launch_block_layout(int64_t n, int cols, int es, void* rows, int64_t ldr, void* colmaj,
                         int64_t ldc, bool to_cols, hipStream_t st) {
  if (n <= 0 || cols <= 0) return;
  const dim3 grid((unsigned)((n + kLt - 1) / kLt), (unsigned)((cols + kLt - 1) / kLt));
  auto go = [&](auto entry) {
    using E = decltype(entry);
    if (to_cols)
      hipLaunchKernelGGL((layout_kernel<E, true>), grid, dim3(kThreads), 0, st, n, cols,
                         static_cast<E*>(rows), ldr, static_cast<E*>(colmaj), ldc);
    else
      hipLaunchKernelGGL((layout_kernel<E, false>), grid, dim3(kThreads), 0, st, n, cols,
                         static_cast<E*>(rows), ldr, static_cast<E*>(colmaj), ldc);
  };
  if (es == 4) go(float());
  else if (es == 8) go(double());
  else if (es == 16) go(double2());
  else throw Error(1, "block entries are 4, 8 or 16 bytes");
  RCG_HIP(hipGetLastError());
}

void launch_layout(int64_t n, int cols, int cw, double* rows, int64_t ldr_real, double* colmaj,
                   int64_t ldc, bool to_cols, hipStream_t st) {
  if (cw != 1 && cw != 2) throw Error(1, "entries are real or complex");
  if (ldr_real % cw != 0) throw Error(1, "row stride is not a whole number of entries");
  launch_block_layout(n, cols, 8 * cw, rows, ldr_real / cw, colmaj, ldc, to_cols, st);
}

void launch_cheb_combine(int64_t n, int cols, int cw, const double* AX, int64_t ldc,
                         const double* X, const double* Z, double* out, int64_t ldr_real,
                         double p0, double p1, double p2, hipStream_t st) {
  if (n <= 0 || cols <= 0) return;
  if (cw != 1 && cw != 2) throw Error(1, "entries are real or complex");
  if (ldr_real % cw != 0) throw Error(1, "row stride is not a whole number of entries");
  const dim3 grid((unsigned)((n + kLt - 1) / kLt), (unsigned)((cols + kLt - 1) / kLt));
  const int64_t ldr = ldr_real / cw;
  if (cw == 1) {
    hipLaunchKernelGGL(cheb_combine_kernel<double>, grid, dim3(kThreads), 0, st, n, cols, AX, ldc,
                       X, Z, out, ldr, p0, p1, p2);
  } else {
    hipLaunchKernelGGL(cheb_combine_kernel<double2>, grid, dim3(kThreads), 0, st, n, cols,
                       reinterpret_cast<const double2*>(AX), ldc,
                       reinterpret_cast<const double2*>(X), reinterpret_cast<const double2*>(Z),
                       reinterpret_cast<double2*>(out), ldr, p0, p1, p2);
  }
  RCG_HIP(hipGetLastError());
}

// partial sums of Re and Im of sum conj(w) v over interleaved complex vectors
__global__ __launch_bounds__(kThreads) void lz_dot_c_kernel(int64_t n, const double* w,
                                                            const double* v, double* P,
                                                            int64_t nblk, int64_t rpb) {
  __shared__ double red[kThreads];
  const int64_t i0 = blockIdx.x * rpb;
  const int64_t i1 = min(n, i0 + rpb);
  double sr = 0.0, si = 0.0;
  for (int64_t i = i0 + threadIdx.x; i < i1; i += kThreads) {
    const double wr = w[2 * i], wi = w[2 * i + 1], vr = v[2 * i], vi = v[2 * i + 1];
    sr = fma(wr, vr, fma(wi, vi, sr));
    si = fma(wr, vi, fma(-wi, vr, si));
  }
  sr = block_sum(sr, red);
  si = block_sum(si, red);
  if (threadIdx.x == 0) {
    P[blockIdx.x] = sr;
    P[nblk + blockIdx.x] = si;
  }
}

void launch_lz_dot_c(int64_t n, const double* w, const double* v, double* alpha_k,
                     double* alpha_im_k, double* ws, size_t ws_elems, hipStream_t st) {
  const int64_t rpb = lz_rows(n);
  const int64_t nblk = (n + rpb - 1) / rpb;
  if ((size_t)(2 * nblk) > ws_elems) throw Error(3, "Lanczos workspace too small");
  hipLaunchKernelGGL(lz_dot_c_kernel, dim3((unsigned)nblk), dim3(kThreads), 0, st, n, w, v, ws,
                     nblk, rpb);
  hipLaunchKernelGGL(lz_finalize_kernel, dim3(1), dim3(kThreads), 0, st, ws, nblk, alpha_k, 0);
  hipLaunchKernelGGL(lz_finalize_kernel, dim3(1), dim3(kThreads), 0, st, ws + nblk, nblk,
                     alpha_im_k, 0);
  RCG_HIP(hipGetLastError());
}

#define RCG_INST(T)                                                                              \
  template void launch_csr_apply<T>(int64_t, const int*, const int*, const T*, const T*, T*, int, \
                                    int, T, T, hipStream_t, const CsrSched*, bool);               \
  template void launch_cheb_step<T>(int64_t, const int*, const int*, const T*, const T*,          \
                                    const T*, T*, int, int, T, T, T, bool, hipStream_t, int,      \
                                    const CsrSched*, bool);                                       \
  template size_t gram_ws_elems<T>(int64_t, int, int);                                           \
  template void launch_gram<T>(int64_t, const T*, int, int, const T*, int, int, T*, T*, size_t,   \
                               hipStream_t, bool);                                                \
  template void launch_tall_gemm<T>(int64_t, const T*, int, int, const T*, int, int, T, T,        \
                                    const T*, T*, int, hipStream_t);                              \
  template void launch_col_sumsq<T>(int64_t, const T*, int, int, double*, double*, size_t,        \
                                    hipStream_t);                                                 \
  template void launch_residual_sumsq<T>(int64_t, const T*, const T*, int, int, const double*,    \
                                         double*, double*, size_t, hipStream_t);                  \
  template void launch_normalize_cols<T>(int64_t, T*, int, int, const double*, hipStream_t);      \
  template void launch_resid_norm_sumsq<T>(int64_t, const T*, const T*, int, int, const double*,  \
                                           double*, double*, size_t, hipStream_t);                \
  template void launch_copy_cols<T>(int64_t, const T*, int, int, T*, int, int, int, hipStream_t); \
  template void launch_randomize_cols<T>(int64_t, T*, int, int, int, uint64_t, uint64_t,          \
                                         hipStream_t);                                            \
  template void launch_fill_cols<T>(int64_t, T*, int, int, int, T, hipStream_t);                 \
  template void launch_dense_step<T>(int64_t, const T*, int64_t, const T*, const T*, T*, int, int, \
                                     T, T, T, int, const T*, const T*, hipStream_t, T*, size_t);

RCG_INST(double)
RCG_INST(float)

}  // namespace rcg
