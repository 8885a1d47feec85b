"""The rules that choose between two kernels by size, at sizes where both were timed
(host code only): the filter of a small CSR operator in one launch, and the tall
products that also form a Gram matrix."""
import ctypes as C
import os

import pytest

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "libengine_paths.so")


@pytest.mark.parametrize("n,row,cols,m,cx,fp32,want", [
    # FP64: from 2 + n / 1024 steps, whatever the columns
    (1000, 7, 512, 2, False, False, True), (3904, 5, 24, 4, False, False, False),
    (3904, 5, 24, 5, False, False, True), (3904, 5, 512, 5, False, False, True),
    (2048, 5, 24, 8, True, False, True), (2049, 5, 24, 8, True, False, False),
    # mixed: later, and much later where two workgroups share a compute unit
    (1000, 7, 256, 2, False, True, False), (1000, 7, 512, 4, False, True, True),
    (2025, 5, 272, 5, False, True, False), (2025, 5, 272, 6, False, True, True),
    (3904, 5, 256, 5, False, True, False), (3904, 5, 24, 6, False, True, True),
    (3904, 5, 272, 10, False, True, False), (4096, 7, 512, 13, False, True, False),
    (3136, 5, 64, 5, True, True, False), (3136, 5, 64, 8, True, True, True),
    # never
    (4097, 5, 24, 40, False, False, False), (1000, 13, 24, 40, False, False, False),
    (1000, 7, 513, 40, False, True, False)])
def test_small_filter(n, row, cols, m, cx, fp32, want):
    assert bool(C.CDLL(LIB).test_small_filter_fits(
        *(C.c_int64(v) for v in (n, min(row, 7) * n, row, cols, m)), int(cx), int(fp32))) == want


@pytest.mark.parametrize("n,bx,by,gram,cross", [
    (1000, 64, 64, True, True), (14000, 48, 48, True, True), (17576, 32, 32, False, False),
    (20000, 64, 16, None, True), (20000, 20, 64, None, True), (50000, 24, 24, False, False),
    (50000, 64, 64, False, False), (65536, 24, 24, False, True), (65536, 64, 64, False, False),
    (75000, 64, 64, True, True), (75000, 48, 48, True, False), (200000, 8, 8, True, True),
    (1 << 20, 24, 24, False, True), (1 << 20, 64, 64, True, True)])
def test_tall_products(n, bx, by, gram, cross):
    L = C.CDLL(LIB)
    if gram is not None:
        assert bool(L.test_tall_gram_pays(C.c_int64(n), by)) == gram
    assert bool(L.test_tall_cross_pays(C.c_int64(n), bx, by)) == cross
