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


def few_together(n, rows, cols):
    few = C.c_int()
    f = C.CDLL(str(LIB_PATH)).th_test_few_together
    f.argtypes = [C.c_size_t] * 5 + [C.POINTER(C.c_int)]
    check(f(n, *rows, *[0] * (3 - len(rows)), cols, C.byref(few)))
    return bool(few.value)


@pytest.mark.parametrize("n,rows,cols,kernel", [
    (2, 1024, 1024, GEMV), (3, 9728, 2560, GEMV), (4, 1024, 1024, GEMV), (4, 9728, 2560, GEMV), (4, 5003, 2968, GEMV),
    (4, 151936, 512, GEMV), (5, 1024, 1024, FEW), (4, 16384, 1024, FEW), (4, 8192, 3072, FEW), (15, 9001, 3000, FEW),
    (3, 100, 12, SCALAR), (40, 100, 12, SCALAR)])
def test_single_matrix_of_few_tokens(n, rows, cols, kernel):
    assert route(n, rows, cols)[0] == kernel


@pytest.mark.parametrize("n,rows,cols", [(4, 8192, 3072), (8, 9001, 3000), (15, 4096, 8192), (5, 64000, 4096),
                                         (9, 40, 9736)])
def test_few_tokens_hold_their_columns(n, rows, cols):
    """K in parts of at most 2560 columns, which the registers hold."""
    kernel, ksplit = route(n, rows, cols)
    assert kernel == FEW and (cols + 31) // 32 <= 80 * ksplit


@pytest.mark.parametrize("n,rows,cols,few", [
    (2, (9728, 9728), 2560, False), (3, (9728, 9728), 2560, True), (2, (3072, 3072), 1024, True),
    (15, (1000, 1000), 520, True), (2, (8192, 8192), 4096, False), (15, (2048, 2048), 4096, False),
    (2, (4096, 1024, 1024), 4096, False), (3, (4096, 1024, 1024), 4096, True), (4, (4096, 1024, 1024), 4096, True), (8, (8192, 1024, 1024), 8192, False),
    (20, (1003, 1003), 1096, True), (700, (5003, 5003), 2968, False),
    (64, (9728, 9728), 2560, False), (1, (64, 64), 64, False)])
def test_matrices_share_a_launch(n, rows, cols, few):
    assert few_together(n, rows, cols) == few


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


@pytest.mark.parametrize("n,heads,kv_heads,pos,low,high", [
    (16, 64, 8, 1500, 8, 12), (24, 64, 8, 1000, 6, 9), (300, 4, 2, 700, 6, 8), (500, 4, 2, 500, 6, 8),  # 1024 rows or more
    (11, 32, 8, 700, 12, 12), (11, 32, 8, 4000, 20, 32), (64, 16, 8, 30000, 16, 32), (64, 16, 8, 60, 1, 1)])
def test_attention_splits(n, heads, kv_heads, pos, low, high):
    """Within a few percent of the best measured count: fewer for many (token,
    head) rows, whose combine takes longer for each."""
    splits = C.c_int()
    f = C.CDLL(str(LIB_PATH)).th_test_attention_splits
    f.argtypes = [C.c_size_t] * 4 + [C.POINTER(C.c_int)]
    check(f(n, heads, kv_heads, pos, C.byref(splits)))
    assert low <= splits.value <= high
