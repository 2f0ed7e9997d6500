"""Which kernel a product takes, on the CPU: the lines of the dispatch that
measurements drew (the figures stand beside the rules), so that a retuned rule
cannot move a size off its kernel unseen."""

from __future__ import annotations

import ctypes as C

import pytest

from titania_amd._lib import LIB_PATH, check

SCALAR, GEMV, FEW, RAGGED, GEMM_F32, GEMM_SMALL, GEMM_LARGE, GEMM_HUGE = range(8)


def route(n, rows, cols):
    """(kernel, parts of K) of th_matmul."""
    kernel, ksplit = C.c_int(), C.c_int()
    f = C.CDLL(str(LIB_PATH)).th_test_matmul_route
    f.argtypes = [C.c_size_t] * 3 + [C.POINTER(C.c_int)] * 2
    check(f(n, rows, cols, C.byref(kernel), C.byref(ksplit)))
    return kernel.value, ksplit.value


def few_preferred(n, rows, cols, n_outs):
    few = C.c_int()
    f = C.CDLL(str(LIB_PATH)).th_test_few_preferred
    f.argtypes = [C.c_size_t] * 3 + [C.c_int, C.POINTER(C.c_int)]
    check(f(n, rows, cols, n_outs, C.byref(few)))
    return bool(few.value)


@pytest.mark.parametrize("n,rows,cols,kernel", [
    (16, 6144, 1024, FEW), (33, 6144, 1024, FEW), (64, 6144, 1024, FEW), (64, 2048, 1024, FEW), (16, 16384, 1024, FEW),
    (16, 151936, 1024, FEW), (32, 16384, 1024, GEMM_F32), (64, 32768, 512, GEMM_F32), (64, 16384, 1024, GEMM_F32),
    (16, 1024, 2048, GEMM_F32)])
def test_single_matrix_of_16_to_64_tokens(n, rows, cols, kernel):
    assert route(n, rows, cols)[0] == kernel


@pytest.mark.parametrize("n", [17, 33, 48, 64])
def test_tall_matrix_reads_its_weights_once(n):
    """An output projection's weights are not read again for every 16 tokens."""
    assert route(n, 151936, 1024)[0] >= GEMM_F32 and route(n, 65536, 512)[0] >= GEMM_F32


@pytest.mark.parametrize("n,rows,cols,few", [
    (32, 2 * 9728, 2560, True), (33, 2 * 9728, 2560, False), (64, 6144, 2560, True), (64, 6144, 1024, True),
    (64, 2 * 4096, 1024, True), (16, 2 * 16384, 1024, True), (32, 2 * 16384, 1024, False), (33, 2 * 8192, 1024, False),
    (64, 12288, 1024, False), (32, 2 * 2048, 4096, True), (33, 2 * 2048, 4096, False), (16, 2 * 8192, 4096, False),
    (33, 6144, 4096, False), (65, 64, 64, False), (15, 2 * 8192, 4096, True)])
def test_several_matrices(n, rows, cols, few):
    assert few_preferred(n, rows, cols, 2) == few and few_preferred(n, rows, cols, 3) == few


@pytest.mark.parametrize("n,rows,cols", [(5, 5003, 2968), (7, 1003, 4552), (17, 5003, 2968), (33, 5003, 2968)])
def test_odd_products_split_k(n, rows, cols):
    """An odd number of results does not keep K in one part."""
    assert n * rows % 2 and route(n, rows, cols)[1] > 1
