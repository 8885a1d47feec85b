// lz_row (rcg_lz_row.hpp) on rows at the end of an operator of INT32_MAX
// nonzeros: the arrays are address ranges of which only the last pages are
// touched.  Prints a row's product for every row length 0..20.  Used by
// tests/test_lz_row_host.py.
#include <sys/mman.h>

#include <climits>
#include <cstdio>

#include "../../rayleighchebyshevgpgpu_amd/csrc/rcg_lz_row.hpp"

template <typename T>
T* range(size_t count) {
  void* p = mmap(nullptr, count * sizeof(T), PROT_READ | PROT_WRITE,
                 MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  return p == MAP_FAILED ? nullptr : static_cast<T*>(p);
}

int main() {
  const size_t nnz = INT_MAX;
  int* col = range<int>(nnz);
  double* val = range<double>(nnz);
  if (!col || !val) return 3;
  double x[4] = {1.0, -2.0, 3.0, 0.5};
  for (int e = 1; e <= 20; ++e) {
    col[nnz - e] = e % 4;
    val[nnz - e] = e;
  }
  for (int len = 0; len <= 20; ++len) {
    const int rowptr[2] = {INT_MAX - len, INT_MAX};
    std::printf("%.17g %.17g\n", rcg::lz_row<false>(rowptr, col, val, x, 0, 1.0),
                rcg::lz_row<true>(rowptr, col, val, x, 0, 0.5));
  }
  return 0;
}
