// rcg_tile.hip -- CSR steps over tiles of a structured grid whose rows are
// gathered from LDS.  A translation unit of its own, so that its kernels cannot
// change the code generated for the general step.
#include "rcg_csr_rows.hpp"

namespace rcg {
namespace {

constexpr int kTileRows = 64;    // rows of the operator per tile
constexpr int kTileNz = 8;       // nonzeros per row a tile holds
constexpr int kTileWaves = 8;    // waves per workgroup, kTileRows / kTileWaves rows each
constexpr int kTileThreads = 64 * kTileWaves;
constexpr int kWaveRows = kTileRows / kTileWaves;
constexpr int kHash = 1024;
static_assert(kWaveRows % 4 == 0 && kTileNz <= 16, "16 lanes to a row, a nonzero to a lane");

// Tile t of the visiting order -> its place in the grid of tiles: tiles march
// along x in bundles of sy x sz, so that the halo rows a tile shares with its y
// and z neighbours are still in the XCD's L2.
__device__ void tile_place(int64_t t, int ntx, int nty, int ntz, int sy, int sz, int& tx, int& ty,
                           int& tz) {
  // bundles in y-fastest order; the last ones of a row or layer are narrower
  const int64_t layer = (int64_t)ntx * nty * sz;  // tiles of a full z-layer of bundles
  const int bz = (int)(t / layer);
  const int dz = min(sz, ntz - bz * sz);
  int64_t q = t - bz * layer;
  const int64_t strip = (int64_t)ntx * sy * dz;
  const int by = (int)(q / strip);
  const int dy = min(sy, nty - by * sy);
  q -= by * strip;
  tx = (int)(q / (dy * dz));
  q -= (int64_t)tx * dy * dz;
  tz = bz * sz + (int)(q / dy);
  ty = by * sy + (int)(q % dy);
}

// One workgroup per tile: the tile's own rows, the distinct rows its nonzeros
// read (own rows first), and for every nonzero the place of its row among
// them.  *bad is set if a tile needs more than smax rows or a row holds more
// than kTileNz nonzeros; the plan is then not used.
__global__ __launch_bounds__(256) void tile_plan_kernel(
    int64_t n, const int* __restrict__ rowptr, const int* __restrict__ col, int gx, int gy, int gz,
    int ex, int ey, int ez, int sy, int sz, int smax, int* __restrict__ srow,
    int* __restrict__ pstart, unsigned char* __restrict__ lidx, int* bad) {
  __shared__ int key[kHash];
  __shared__ short pos[kHash];
  __shared__ int count, fail;
  const int64_t t = blockIdx.x;
  int tx, ty, tz;
  tile_place(t, (gx + ex - 1) / ex, (gy + ey - 1) / ey, (gz + ez - 1) / ez, sy, sz, tx, ty, tz);
  const int nx = min(ex, gx - tx * ex), ny = min(ey, gy - ty * ey), nz = min(ez, gz - tz * ez);
  const int own = nx * ny * nz;
  for (int h = threadIdx.x; h < kHash; h += 256) key[h] = -1;
  if (threadIdx.x == 0) {
    count = kTileRows;  // places past the tile's own rows, up to 64, stay empty
    fail = 0;
  }
  __syncthreads();
  int* s = srow + t * smax;
  auto row_of = [&](int k) -> int {
    const int x = tx * ex + k % nx, y = ty * ey + (k / nx) % ny, z = tz * ez + k / (nx * ny);
    return x + gx * (y + gy * z);
  };
  auto slot = [&](int j, bool& fresh) -> int {  // the hash slot of row j, taken if new
    unsigned h = ((unsigned)j * 2654435761u) >> 22;
    for (int probe = 0; probe < kHash; ++probe, h = (h + 1) & (kHash - 1)) {
      const int old = atomicCAS(&key[h], -1, j);
      if (old == -1 || old == j) {
        fresh = old == -1;
        return (int)h;
      }
    }
    fresh = false;
    return -1;
  };
  for (int k = threadIdx.x; k < smax; k += 256) s[k] = -1;
  __syncthreads();
  for (int k = threadIdx.x; k < own; k += 256) {
    bool fresh;
    const int r = row_of(k);
    pos[slot(r, fresh)] = (short)k;
    s[k] = r;
  }
  __syncthreads();
  for (int q = threadIdx.x; q < kTileRows * kTileNz; q += 256) {
    const int k = q / kTileNz, e = q % kTileNz;
    if (k >= own) continue;
    const int r = row_of(k);
    const int p0 = rowptr[r], len = rowptr[r + 1] - p0;
    if (e == 0 && len > kTileNz) fail = 1;
    if (e >= len || len > kTileNz) continue;
    const int j = col[p0 + e];
    bool fresh;
    const int h = slot(j, fresh);
    if (h < 0) {
      fail = 1;
    } else if (fresh) {
      const int at = atomicAdd(&count, 1);
      if (at < smax) {
        s[at] = j;
        pos[h] = (short)at;
      } else {
        fail = 1;
        pos[h] = 0;
      }
    }
  }
  __syncthreads();
  for (int q = threadIdx.x; q < kTileRows * kTileNz; q += 256) {
    const int k = q / kTileNz, e = q % kTileNz;
    int l = 255, p0 = 0;
    if (k < own) {
      const int r = row_of(k);
      p0 = rowptr[r];
      const int len = rowptr[r + 1] - p0;
      if (e < len && len <= kTileNz && !fail) {
        bool fresh;
        l = pos[slot(col[p0 + e], fresh)];
      }
    }
    lidx[t * (kTileRows * kTileNz) + q] = (unsigned char)l;
    if (e == 0) pstart[t * kTileRows + k] = p0;
  }
  if (threadIdx.x == 0 && fail) *bad = 1;
}

// lane E of each 16 lanes, for all of them
template <int E>
__device__ __forceinline__ int row_bcast(int v) {
  return __builtin_amdgcn_update_dpp(0, v, 0x150 + E, 0xf, 0xf, true);
}
template <int E>
__device__ __forceinline__ float row_bcast(float v) {
  return __int_as_float(row_bcast<E>(__float_as_int(v)));
}
template <int E>
__device__ __forceinline__ double row_bcast(double v) {
  const long long b = __double_as_longlong(v);
  const unsigned lo = (unsigned)row_bcast<E>((int)(b & 0xffffffffll));
  const unsigned hi = (unsigned)row_bcast<E>((int)(b >> 32));
  return __longlong_as_double(((long long)hi << 32) | lo);
}

// nonzeros E..N-1 of the row: its entries of the copied rows from LDS (lo: this
// lane's nonzero's byte offset there, at: this lane's place in a row) ...
template <int E, int N, typename T, int NV>
__device__ __forceinline__ void tile_read(const char* at, int lo,
                                          T (&u)[kTileNz][NV][V16<T>::W]) {
  if constexpr (E < N) {
    const char* p = at + row_bcast<E>(lo);
#pragma unroll
    for (int k = 0; k < NV; ++k) V16<T>::ld(reinterpret_cast<const T*>(p + 256 * k), u[E][k]);
    tile_read<E + 1, N, T, NV>(at, lo, u);
  }
}
// ... and their products, in order.  ALL: every row of the wave has N nonzeros;
// else this lane's row has cnt of them.
template <int E, int N, bool ALL, bool CX, typename T, int NV>
__device__ __forceinline__ void tile_fma(const T (&u)[kTileNz][NV][V16<T>::W], T av, T ai, int cnt,
                                         T (&acc)[NV][V16<T>::W]) {
  if constexpr (E < N) {
    const T a = row_bcast<E>(av);
    const bool live = ALL || E < cnt;
    if constexpr (CX) {
      const T b = row_bcast<E>(ai);
#pragma unroll
      for (int k = 0; k < NV; ++k)
#pragma unroll
        for (int w = 0; w < V16<T>::W; w += 2) {
          T re = fma(a, u[E][k][w], acc[k][w]);
          re = fma(-b, u[E][k][w + 1], re);
          T im = fma(a, u[E][k][w + 1], acc[k][w + 1]);
          im = fma(b, u[E][k][w], im);
          acc[k][w] = live ? re : acc[k][w];
          acc[k][w + 1] = live ? im : acc[k][w + 1];
        }
    } else {
#pragma unroll
      for (int k = 0; k < NV; ++k)
#pragma unroll
        for (int w = 0; w < V16<T>::W; ++w) {
          const T v = fma(a, u[E][k][w], acc[k][w]);
          acc[k][w] = live ? v : acc[k][w];
        }
    }
    tile_fma<E + 1, N, ALL, CX, T, NV>(u, av, ai, cnt, acc);
  }
}

// One step on the 64 rows of a tile and 16 NV vectors of 16 bytes of each.  The
// tile's own rows and their halo (the distinct rows its nonzeros read) are copied
// to LDS once, directly from memory; the general step requests a row once per
// nonzero instead (7 times for a 7-point stencil; 2.5 times with 4 x 4 x 4
// tiles), and the vector-memory address path, not HBM, bounds it.  16 lanes
// own a row, as many as a DPP broadcast reaches: lane e of them holds the row's
// nonzero e.
//
// A row's nonzeros are summed in their order with the arithmetic of csr_rows
// and absent ones are skipped, so the result is the general step's bit for bit.
template <typename T, bool CX, int MODE, int SMAX, int NV>
__global__ __launch_bounds__(kTileThreads) void csr_tile_kernel(
    const int* __restrict__ srow, const int* __restrict__ pstart,
    const unsigned char* __restrict__ lidx, const T* __restrict__ val, const T* X, const T* Z,
    T* out, int ld, int ncols, int c_first, T p0, T p1, T p2, int64_t ntile, int npanel, const T* R,
    const T* __restrict__ kap, MixedArgs ms) {
  constexpr bool kSrc = MODE == kChebSrc || MODE == kChebSrcEnd;
  using VT = V16<T>;
  constexpr int W = VT::W;
  constexpr int PAN = 16 * NV * W;           // elements of a row per workgroup
  constexpr int LPR = 16 * NV, RPI = 64 / LPR;  // lanes that copy a row, rows per instruction
  constexpr int IT = kWaveRows / 4;          // a wave computes 4 rows at a time
  __shared__ __align__(16) T xs[SMAX * PAN];
  const int64_t L = xcd_remap(blockIdx.x, gridDim.x);
  if (L >= ntile * npanel) return;  // uniform across the workgroup
  const int64_t tile = L / npanel;
  const int c0 = c_first + (int)(L % npanel) * PAN;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int g = lane & 15;
  const int* s = srow + tile * SMAX;
  // rows into LDS: a copy instruction moves RPI consecutive ones.  Columns up
  // to the row's padding (ld, a multiple of 4) are read.
  {
    const int cl = c0 + (lane % LPR) * W;
    constexpr int NC = (SMAX / RPI + kTileWaves - 1) / kTileWaves;
    static_assert(SMAX % RPI == 0, "whole copy instructions");
    int cr[NC];
#pragma unroll
    for (int k = 0; k < NC; ++k) {
      const int q = wave + k * kTileWaves;
      cr[k] = q < SMAX / RPI ? s[q * RPI + lane / LPR] : -1;
    }
#pragma unroll
    for (int k = 0; k < NC; ++k) {
      const int q = wave + k * kTileWaves, r = cr[k];
      if (r >= 0 && cl < ld)
        __builtin_amdgcn_global_load_lds(
            (const __attribute__((address_space(1))) void*)(X + (int64_t)r * ld + cl),
            (__attribute__((address_space(3))) void*)(xs + q * RPI * PAN), 16, 0, 0);
    }
  }
  // nonzeros, one to a lane, and the rows' own operands
  int row[IT], lo[IT];
  T av[IT], ai[CX ? IT : 1];
  unsigned long long there[IT];
  T zs[IT][NV][W], rs[kSrc ? IT : 1][NV][W], kv[kSrc ? NV : 1][W];
  // kChebSrcEnd: V and its columns' factors, in whole 16-byte vectors and ahead of the
  // gathers, as Z and R
  constexpr bool kEnd = MODE == kChebSrcEnd;
  double vs[kEnd ? IT : 1][kEnd ? NV : 1][W], uv[kEnd ? NV : 1][W];
#pragma unroll
  for (int q = 0; q < IT; ++q) {
    const int k = wave * kWaveRows + q * 4 + (lane >> 4);
    row[q] = s[k];  // -1: a tile cut by the grid's end has fewer rows
    const int li = g < kTileNz ? (int)lidx[(tile * kTileRows + k) * kTileNz + g] : 255;
    const int64_t p = (int64_t)pstart[tile * kTileRows + k] + g;
    there[q] = __ballot(li != 255);
    lo[q] = (li != 255 ? li : k) * (int)(PAN * sizeof(T));
    av[q] = T(0);
    if (li != 255) {
      if constexpr (CX) {
        av[q] = ld_once(val + 2 * p);
        ai[q] = ld_once(val + 2 * p + 1);
      } else {
        av[q] = ld_once(val + p);
      }
    } else if constexpr (CX) {
      ai[q] = T(0);
    }
  }
  // kApplyStart: the columns' (theta, Ritz flag)
  double th[MODE == kApplyStart ? NV : 1][W], fl[MODE == kApplyStart ? NV : 1][W];
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int c = c0 + (g + 16 * k) * W;
    if constexpr (MODE == kApplyStart) {
#pragma unroll
      for (int w = 0; w < W; ++w) {
        th[k][w] = c + w < ms.nc ? ms.cp[c + w] : 0.0;
        fl[k][w] = c + w < ms.nc ? ms.cp[ms.nc + c + w] : 0.0;
      }
    }
    if constexpr (kSrc) {
#pragma unroll
      for (int w = 0; w < W; ++w) kv[k][w] = c < ld ? kap[c + w] : T(0);
    }
    if constexpr (kEnd) {
#pragma unroll
      for (int w = 0; w < W; ++w) uv[k][w] = c + w < ncols ? ms.um[c + w] : 0.0;
    }
#pragma unroll
    for (int q = 0; q < IT; ++q) {
      const int64_t o = (int64_t)row[q] * ld + c;
      if (row[q] >= 0 && c < ncols) {
        if constexpr (MODE == kCheb || kSrc) VT::ld_stream(Z + o, zs[q][k]);
        if constexpr (kSrc) VT::ld_stream(R + o, rs[q][k]);
        if constexpr (kEnd) {
#pragma unroll
          for (int h = 0; h < W / 2; ++h) {
            const dvec2 v = reinterpret_cast<const dvec2*>(ms.v_end + o)[h];
            vs[q][k][2 * h] = v.x;
            vs[q][k][2 * h + 1] = v.y;
          }
        }
      }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's copies have landed
  __syncthreads();
  const char* at = reinterpret_cast<const char*>(xs) + 16 * g;
#pragma unroll
  for (int q = 0; q < IT; ++q) {
    T acc[NV][W], u[kTileNz][NV][W];
#pragma unroll
    for (int k = 0; k < NV; ++k)
#pragma unroll
      for (int w = 0; w < W; ++w) acc[k][w] = T(0);
    const T aq = av[q], bq = CX ? ai[q] : T(0);
    const unsigned long long one = 0x0001000100010001ull, m = there[q];
    if (m == 0x7full * one) {
      tile_read<0, 7, T, NV>(at, lo[q], u);
      tile_fma<0, 7, true, CX, T, NV>(u, aq, bq, 7, acc);
    } else if (m == 0x1full * one) {
      tile_read<0, 5, T, NV>(at, lo[q], u);
      tile_fma<0, 5, true, CX, T, NV>(u, aq, bq, 5, acc);
    } else {
      const int cnt = __popcll((m >> (lane & 48)) & 255ull);
      tile_read<0, kTileNz, T, NV>(at, lo[q], u);
      tile_fma<0, kTileNz, false, CX, T, NV>(u, aq, bq, cnt, acc);
    }
    const char* own = at + (wave * kWaveRows + q * 4 + (lane >> 4)) * (int)(PAN * sizeof(T));
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const int c = c0 + (g + 16 * k) * W;
      T x[W], o[W];
      VT::ld(reinterpret_cast<const T*>(own + 256 * k), x);
      if constexpr (MODE == kApplyStart) {
        // W = A V straight into the mixed filter's start
        if (row[q] < 0 || c >= ncols) continue;
        const int64_t at0 = (int64_t)row[q] * ld + c;
        float e0[W], e1[W], rr[W];
#pragma unroll
        for (int w = 0; w < W; ++w)
          mixed_start_elem(x[w], p0 * acc[k][w], th[k][w], fl[k][w], ms.e1c, ms.g1, ms.g2, e0[w],
                           e1[w], rr[w]);
        if (c + W <= ncols) {
          typedef float fvec2 __attribute__((ext_vector_type(2)));
          *reinterpret_cast<fvec2*>(ms.e0 + at0) = fvec2{e0[0], e0[1]};
          *reinterpret_cast<fvec2*>(ms.e1 + at0) = fvec2{e1[0], e1[1]};
          *reinterpret_cast<fvec2*>(ms.r + at0) = fvec2{rr[0], rr[1]};
        } else {
          ms.e0[at0] = e0[0];
          ms.e1[at0] = e1[0];
          ms.r[at0] = rr[0];
        }
        continue;
      }
#pragma unroll
      for (int w = 0; w < W; ++w) {
        if constexpr (MODE == kApply) o[w] = p0 * acc[k][w];
        else if constexpr (MODE == kChebFirst) o[w] = p2 * (p1 * fma(p0, acc[k][w], x[w]));
        else if constexpr (kSrc)
          o[w] = p2 * fma(kv[k][w], rs[q][k][w], fma(p1, fma(p0, acc[k][w], x[w]), -zs[q][k][w]));
        else o[w] = p2 * fma(p1, fma(p0, acc[k][w], x[w]), -zs[q][k][w]);
      }
      if (row[q] < 0 || c >= ncols) continue;
      if constexpr (MODE == kChebSrcEnd) {
        // V <- s_end (um V + x), V FP64; x itself is not stored
        double* v = ms.v_end + (int64_t)row[q] * ld + c;
        double e[W];
#pragma unroll
        for (int w = 0; w < W; ++w) e[w] = ms.s_end * fma(uv[k][w], vs[q][k][w], double(o[w]));
        if (c + W <= ncols) {
#pragma unroll
          for (int h = 0; h < W / 2; ++h)
            reinterpret_cast<dvec2*>(v)[h] = dvec2{e[2 * h], e[2 * h + 1]};
        } else {
#pragma unroll
          for (int w = 0; w < W; ++w)
            if (c + w < ncols) v[w] = e[w];
        }
        continue;
      }
      T* y = out + (int64_t)row[q] * ld + c;
      if (c + W <= ncols) {
        VT::st_stream(y, o);
      } else {
#pragma unroll
        for (int w = 0; w < W; ++w)
          if (c + w < ncols) y[w] = o[w];
      }
    }
  }
}

template <typename T, bool CX, int MODE, int NV>
void tile_launch_nv(const TilePlan& t, const T* val, const T* X, const T* Z, T* out, int ld,
                    int ncols, int c_first, int npanel, T p0, T p1, T p2, const T* R, const T* kap,
                    const MixedArgs& ms, hipStream_t st) {
  const dim3 grid((unsigned)round_up(t.ntile * npanel, kXcds));
#define RCG_TILE(S)                                                                               \
  hipLaunchKernelGGL((csr_tile_kernel<T, CX, MODE, S, NV>), grid, dim3(kTileThreads), 0, st,      \
                     t.srow, t.pstart, t.lidx, val, X, Z, out, ld, ncols, c_first, p0, p1, p2,    \
                     t.ntile, npanel, R, kap, ms)
  if (t.smax == 96) RCG_TILE(96);
  else RCG_TILE(160);
#undef RCG_TILE
  RCG_HIP(hipGetLastError());
}

// Panels of 64 elements: FP64 rows of 512 bytes (two workgroups of 80 KB per
// CU), FP32 rows of 256.  FP64 columns left over, up to 32, take a launch with
// half the lanes' work and half the LDS.
inline int fp64_full_panels(int ncols) { return ncols / 64 + (ncols % 64 > 32 ? 1 : 0); }
template <typename T, bool CX, int MODE>
void tile_launch(const TilePlan& t, const T* val, const T* X, const T* Z, T* out, int ld, int ncols,
                 T p0, T p1, T p2, const T* R, const T* kap, const MixedArgs& ms, hipStream_t st) {
  if constexpr (std::is_same<T, double>::value) {
    const int rest = ncols % 64;
    const int full = fp64_full_panels(ncols);
    if (full > 0)
      tile_launch_nv<T, CX, MODE, 2>(t, val, X, Z, out, ld, ncols, 0, full, p0, p1, p2, R, kap, ms,
                                     st);
    if (rest > 0 && rest <= 32)
      tile_launch_nv<T, CX, MODE, 1>(t, val, X, Z, out, ld, ncols, 64 * full, 1, p0, p1, p2, R, kap,
                                     ms, st);
  } else {
    tile_launch_nv<T, CX, MODE, 1>(t, val, X, Z, out, ld, ncols, 0, (ncols + 63) / 64, p0, p1, p2, R,
                                   kap, ms, st);
  }
}

}  // namespace

TileShape tile_shape(int64_t gx, int64_t gy, int64_t gz) {
  TileShape t;
  t.gx = gx;
  t.gy = gy;
  t.gz = gz;
  t.rows = kTileRows;
  if (gz > 1) {
    t.ex = t.ey = t.ez = 4;
    t.sy = 32;
    t.sz = 8;
    t.smax = 160;  // 64 rows and 6 faces of 16
  } else {
    t.ex = t.ey = 8;
    t.ez = 1;
    t.sy = 16;
    t.sz = 1;
    t.smax = 96;  // 64 rows and 4 sides of 8
  }
  t.ntile = ((gx + t.ex - 1) / t.ex) * ((gy + t.ey - 1) / t.ey) * ((gz + t.ez - 1) / t.ez);
  t.srow = (size_t)t.ntile * t.smax;
  t.pstart = (size_t)t.ntile * kTileRows;
  t.lidx = (size_t)t.ntile * kTileRows * kTileNz;
  return t;
}

void launch_tile_plan(const TileShape& t, int64_t n, const int* rowptr, const int* col, int* srow,
                      int* pstart, unsigned char* lidx, int* bad, hipStream_t st) {
  if (t.gx * t.gy * t.gz != n || t.ntile > INT32_MAX) throw Error(1, "tile plan: grid does not match");
  hipLaunchKernelGGL(tile_plan_kernel, dim3((unsigned)t.ntile), dim3(256), 0, st, n, rowptr, col,
                     (int)t.gx, (int)t.gy, (int)t.gz, t.ex, t.ey, t.ez, t.sy, t.sz, t.smax, srow, pstart,
                     lidx, bad);
  RCG_HIP(hipGetLastError());
}

template <typename T>
bool launch_tile_step(const TilePlan& t, int mode, const T* val, const T* X, const T* Z, T* out,
                      int ld, int ncols, T p0, T p1, T p2, const T* R, const T* kap, bool cx,
                      const MixedArgs& ms, hipStream_t st) {
#define RCG_TILE_MODE(M)                                                                       \
  case M:                                                                                      \
    if (cx)                                                                                    \
      tile_launch<T, true, M>(t, val, X, Z, out, ld, ncols, p0, p1, p2, R, kap, ms, st);       \
    else                                                                                       \
      tile_launch<T, false, M>(t, val, X, Z, out, ld, ncols, p0, p1, p2, R, kap, ms, st);      \
    return true;
  if constexpr (std::is_same<T, double>::value) {
    switch (mode) {
      RCG_TILE_MODE(kApply)
      RCG_TILE_MODE(kChebFirst)
      RCG_TILE_MODE(kCheb)
      RCG_TILE_MODE(kApplyStart)
      default: return false;
    }
  } else {
    switch (mode) {
      RCG_TILE_MODE(kChebSrc)
      RCG_TILE_MODE(kChebSrcEnd)
      default: return false;
    }
  }
#undef RCG_TILE_MODE
}
template <typename T>
int tile_step_launches(int ncols) {
  if constexpr (std::is_same<T, float>::value) return ncols > 0 ? 1 : 0;
  const int full = fp64_full_panels(ncols);
  return (full > 0 ? 1 : 0) + (ncols > 64 * full ? 1 : 0);
}
template int tile_step_launches<double>(int);
template int tile_step_launches<float>(int);

template bool launch_tile_step<double>(const TilePlan&, int, const double*, const double*,
                                       const double*, double*, int, int, double, double, double,
                                       const double*, const double*, bool, const MixedArgs&,
                                       hipStream_t);
template bool launch_tile_step<float>(const TilePlan&, int, const float*, const float*,
                                      const float*, float*, int, int, float, float, float,
                                      const float*, const float*, bool, const MixedArgs&,
                                      hipStream_t);

}  // namespace rcg
