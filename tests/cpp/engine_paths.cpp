// The solve's engine (csrc/rcg_solver.cpp, compiled into this library) driven
// piece by piece, for tests of branches that a whole solve reaches only with
// unusual blocks or little memory.  The C entry points are this library's own
// copies; the kernels come from librcg.so.  Launches are counted, and device
// allocations can be made to fail from a size on.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <complex>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <thread>
#include <type_traits>
#include <vector>

#include "../../rayleighchebyshevgpgpu_amd/csrc/rcg_internal.hpp"

namespace {
size_t g_alloc_limit = ~size_t(0);  // allocations above fail
int g_device_factors = 0, g_pairs = 0, g_grams = 0;

hipError_t limited_malloc(void** p, size_t bytes) {
  if (bytes > g_alloc_limit) return hipErrorOutOfMemory;
  return hipMalloc(p, bytes);
}
}  // namespace
namespace rcg {
inline void counted_gram_chol(int64_t n, const double* X, int ldx, int b, double* C, double* inv2,
                              double* ws, size_t ws_elems, hipStream_t st) {
  ++g_device_factors;
  launch_gram_chol(n, X, ldx, b, C, inv2, ws, ws_elems, st);
}
inline void counted_gram_pair(int64_t n, const double* X, int ldx, const double* Y, int ldy, int b,
                              double* G, double* ws, size_t ws_elems, hipStream_t st) {
  ++g_pairs;
  launch_gram_pair(n, X, ldx, Y, ldy, b, G, ws, ws_elems, st);
}
template <typename T, typename... Args>
void counted_gram(int64_t n, const T* X, Args... args) {
  ++g_grams;
  launch_gram<T>(n, X, args...);
}
}  // namespace rcg
#define hipMalloc limited_malloc
#define launch_gram counted_gram
#define launch_gram_chol counted_gram_chol
#define launch_gram_pair counted_gram_pair
#include "../../rayleighchebyshevgpgpu_amd/csrc/rcg_solver.cpp"

namespace {
template <class S>
void project_and_rotate(Engine& e, int64_t b, double* H_out, double* res) {
  std::vector<S> H, I(b * b, S(0.0));
  e.ortho_project<S>(b, H);
  std::memcpy(H_out, H.data(), sizeof(S) * b * b);
  std::vector<double> th(b), r;
  for (int64_t j = 0; j < b; ++j) {
    I[j + j * b] = S(1.0);
    th[j] = std::real(H[j + j * b]);
  }
  e.rotate_residuals(b, I, th, b, r);
  std::memcpy(res, r.data(), sizeof(double) * b);
}
}  // namespace

extern "C" {
void test_alloc_limit(int64_t bytes) { g_alloc_limit = bytes < 0 ? ~size_t(0) : (size_t)bytes; }

// An iteration's orthonormalisation and projection of V (H, b x b), then its
// rotation by the identity: V holds the orthonormal basis, res the residuals with
// the diagonal of H.  prime (or null) goes first through the same engine, as the
// iteration before.  counts: device factors, paired and single
// Gram products for V.
int test_ortho_project(rcg_operator op, rcg_block prime, rcg_block V, rcg_block T, rcg_block W,
                       int64_t b, double* H, double* res, int32_t* counts) {
  return guarded([&] {
    Engine e(op->ctx, op, op->n);
    e.reserve(real_ld(V), real_ld(V));
    auto run = [&](rcg_block X) {
      e.attach(static_cast<double*>(X->d()), static_cast<double*>(T->d()),
               static_cast<double*>(W->d()), real_ld(X), nullptr, 0);
      g_device_factors = g_pairs = g_grams = 0;
      if (e.cx()) project_and_rotate<cplx>(e, b, H, res);
      else project_and_rotate<double>(e, b, H, res);
    };
    if (prime) run(prime);
    run(V);
    counts[0] = g_device_factors;
    counts[1] = g_pairs;
    counts[2] = g_grams;
    if (!e.v_is_first())
      rcg::launch_copy_cols<double>(V->n, e.V(), (int)real_ld(V), 0, static_cast<double*>(V->d()),
                                    (int)real_ld(V), 0, (int)(e.cw() * b), e.stream());
    e.sync();
  });
}

// Whether a product of cols columns goes over LDS tiles.
int test_apply_tiles(rcg_operator op, int64_t cols, int32_t* tiles) {
  return guarded([&] {
    Engine e(op->ctx, op, op->n);
    e.attach(nullptr, nullptr, nullptr, e.cw() * block_ld(cols), nullptr, 0);
    const rcg::CsrSched* sc = e.sched_for(e.cw() * cols);
    *tiles = sc && sc->tile;
  });
}

// An FP64 filter of degree m: the schedule it took, its column panel and launches.
int test_filter_route(rcg_operator op, rcg_block X, rcg_block T, int64_t cols, int64_t m,
                      char* sched, int64_t cap, int64_t* panel, int64_t* launches) {
  return guarded([&] {
    Piece pc(X, T, op);
    pc.eng.filter(cols, (long)m, 1, 14.0, 1.0);
    std::snprintf(sched, (size_t)cap, "%s", pc.eng.last_sched().c_str());
    *panel = pc.eng.last_panel();
    *launches = pc.eng.step_launches();
    pc.settle(X, cols);
  });
}

int test_tall_gram_pays(int64_t n, int by) { return rcg::tall_gram_pays(n, by) ? 1 : 0; }
int test_tall_cross_pays(int64_t n, int bx, int by) {
  return rcg::tall_cross_pays(n, bx, by) ? 1 : 0;
}
int test_small_filter_fits(int64_t n, int64_t nnz, int64_t max_row, int64_t cols, int64_t m,
                           int cx, int fp32) {
  return rcg::small_filter_fits(n, nnz, max_row, cols, m, cx != 0, fp32 != 0) ? 1 : 0;
}
}
