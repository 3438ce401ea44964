"""How the batch kernels of the bit-exact f32 matmul are launched (no GPU needed)."""
import ctypes as C

import pytest

import nncpu_amd as N

SLICE = "_ZN3nnh11batch_sliceEi"  # nnh::batch_slice(int rows)


@pytest.mark.parametrize("rows", [1, 16, 17, 1000, 65552, 262144, (1 << 26), (1 << 26) + 1, (1 << 31) - 1])
def test_a_launch_holds_less_than_2_to_the_32_threads(rows):
    f = getattr(N.lib(), SLICE)
    f.argtypes, f.restype = [C.c_int], C.c_int
    step = f(rows)
    assert step % 16 == 0
    assert (rows + 15) // 16 * (step // 16) * 512 < 1 << 32
    assert (step > 0) == (rows <= 1 << 26)


@pytest.mark.parametrize("dtype,rows,cols,n_tok,here", [
    # Slower than the one- to four-vector kernels by the factor named when they were taken here.
    (1, 20000, 1024, 3, False), (1, 37888, 3584, 3, False),   # 1.36, 1.20
    (1, 256, 4096, 2, False), (1, 2048, 12288, 2, False),     # 1.16, 1.10
    (2, 8192, 1024, 3, False), (2, 65536, 1024, 5, False),    # 1.21, 1.4
    (1, 256, 4096, 3, True), (1, 28672, 4096, 3, True), (1, 4096, 4096, 2, True), (1, 65536, 1024, 13, True),
    (2, 4096, 4096, 3, True), (2, 14336, 4096, 5, True), (2, 151936, 512, 16, True), (2, 14336, 4096, 2, False),
])
def test_few_vectors_go_where_they_are_faster(dtype, rows, cols, n_tok, here):
    f = N.lib()._ZN3nnh10batch_winsEiiiib  # nnh::batch_wins(int dtype, int rows, int nb, int n_tok, bool v2)
    f.argtypes, f.restype = [C.c_int] * 4 + [C.c_bool], C.c_bool
    assert f(dtype, rows, cols // 32, n_tok, rows >= 12288 and cols <= 16384) == here


@pytest.mark.parametrize("rows,cols,n_tok,here", [
    (257, 4096, 4, False), (14336, 2048, 4, False), (14337, 1000, 4, False),  # 1.32, 1.30, 1.19 times slower here
    (257, 1024, 4, True), (4097, 4096, 4, True), (256, 4096, 4, True), (14337, 1000, 5, True), (256, 4096, 3, False),
])
def test_few_vectors_bf16(rows, cols, n_tok, here):
    f = N.lib()._ZN3nnh15batch_wins_bf16Eiiii  # nnh::batch_wins_bf16(int path, int rows, int cols, int n_tok)
    f.argtypes, f.restype = [C.c_int] * 4, C.c_bool
    path = 1 if rows % 4 == 0 else 3 if cols % 32 == 0 else 2  # the 4-row, 1-row by 32 and 1-row by 8 kernels' chains
    assert f(path, rows, cols, n_tok) == here
