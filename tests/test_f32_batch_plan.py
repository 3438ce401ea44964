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
