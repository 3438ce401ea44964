"""The bit-exact f32 matmul of several vectors on the f32 matrix unit, against
the oracle: every output bit, at the edges of its tiles (16 rows, 16 vectors,
token tiles of up to 64), of its stages (8 blocks, steps of 4) and of Q4's
bias groups (8 blocks), with strided rows, and with signed zeros, denormals,
infinities and values whose products under- and overflow."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = pytest.importorskip("nncpu_amd")


@pytest.fixture(scope="module", autouse=True)
def device():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    N.init(0)


def run(oracle, dtype, rows, cols, n_tok, pad=0, x=None, seed=0xB47C):
    rng = oracle.Rng(seed + rows + cols + n_tok)
    m = oracle.QMatrix.from_f32(dtype, rng.normals(rows * cols, 0.02).reshape(rows, cols))
    w = N.Weight.from_split(dtype, m.buf, rows, cols)
    xs, ys = cols + pad, rows + pad
    if x is None:
        x = rng.normals(n_tok * xs, 1.0)
    y = np.full(n_tok * ys, 7.0, np.float32)
    N.gemv_batch(w, x, xs, y, ys, n_tok, N.ACT_F32)
    ref = np.full(n_tok * ys, 7.0, np.float32)
    o = oracle.gemv_batch(m, x, n_tok, xs, ys, backend="avx2")
    for t in range(n_tok):
        ref[t * ys:t * ys + rows] = o[t * ys:t * ys + rows]
    w.free()
    return y, ref


@pytest.mark.parametrize("dtype", [1, 2])
@pytest.mark.parametrize("rows,cols,n_tok,pad", [
    (1, 32, 5, 0), (15, 96, 16, 0), (16, 128, 17, 4), (17, 224, 6, 0), (33, 256, 32, 12), (40, 288, 33, 0),
    (31, 1152, 49, 0), (70, 1184, 64, 4), (129, 608, 65, 0), (257, 992, 80, 8), (4100, 2080, 7, 0), (4112, 512, 40, 0),
    (8200, 512, 81, 4), (12290, 544, 20, 0), (16400, 96, 130, 0), (100, 320, 9, 3),
])
def test_f32_batch_bit_exact(oracle, dtype, rows, cols, n_tok, pad):
    y, ref = run(oracle, dtype, rows, cols, n_tok, pad)
    assert np.array_equal(y.view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("dtype", [1, 2])
@pytest.mark.parametrize("cols", [288, 1024, 1184])
def test_f32_batch_special_values(oracle, dtype, cols):
    n_tok = 19
    rng = np.random.default_rng(cols + dtype)
    x = np.ldexp(rng.standard_normal(n_tok * cols), rng.integers(-150, 100, n_tok * cols)).astype(np.float32)
    x[rng.integers(0, x.size, x.size // 4)] = 0.0
    x[rng.integers(0, x.size, x.size // 4)] = -0.0
    x.reshape(n_tok, cols)[3] = -0.0
    x.reshape(n_tok, cols)[5, -1] = np.inf
    x.reshape(n_tok, cols)[6, 40] = 3e38
    x.reshape(n_tok, cols)[7, 5] = np.nan
    y, ref = run(oracle, dtype, 50, cols, n_tok, x=x)
    nan = np.isnan(ref)
    assert np.array_equal(np.isnan(y), nan) and nan.reshape(n_tok, 50)[7].all()
    assert np.array_equal(y[~nan].view(np.uint32), ref[~nan].view(np.uint32))


# BF16: the 4-row kernel's chains (rows % 4 == 0), the 1-row kernel's 8 (cols % 32
# != 0) and 32, around stages of 256 columns, 8- and 32-column steps.
@pytest.mark.parametrize("rows,cols,n_tok,pad", [
    (4, 8, 5, 0), (16, 264, 17, 4), (40, 520, 33, 0), (256, 1000, 64, 8), (4100, 512, 40, 0), (8208, 544, 16, 0),
    (17, 24, 6, 0), (33, 248, 16, 4), (70, 1544, 65, 0), (1030, 264, 130, 0),
    (1, 32, 4, 0), (31, 224, 18, 0), (257, 608, 49, 4), (4097, 288, 65, 0), (6, 320, 9, 3),
])
def test_bf16_batch_bit_exact(oracle, rows, cols, n_tok, pad):
    rng = np.random.default_rng(rows * 7 + cols + n_tok)
    w = oracle.f32_array_to_bf16(rng.standard_normal(rows * cols).astype(np.float32))
    xs, ys = cols + pad, rows + pad
    x = np.ldexp(rng.standard_normal(n_tok * xs), rng.integers(-30, 30, n_tok * xs)).astype(np.float32)
    x[rng.integers(0, x.size, x.size // 8)] = -0.0
    wt = N.Weight.bf16(w, rows, cols)
    y = np.full(n_tok * ys, 7.0, np.float32)
    N.gemv_batch(wt, x, xs, y, ys, n_tok)
    want = oracle.gemv_bf16(w, x, rows, cols, n_tok, xs, ys)
    for t in range(n_tok):
        got = y[t * ys:t * ys + rows]
        assert np.array_equal(got.view(np.uint32), want[t * ys:t * ys + rows].view(np.uint32)), t
    wt.free()


@pytest.mark.parametrize("rows,cols", [(48, 520), (51, 520), (51, 544)])  # the 4-row, the 8- and the 32-chain kernel's
def test_bf16_batch_special_values(oracle, rows, cols):
    n_tok = 19
    rng = np.random.default_rng(rows + cols)
    w = oracle.f32_array_to_bf16(np.ldexp(rng.standard_normal(rows * cols), rng.integers(-140, 20, rows * cols)).astype(np.float32))
    w[rng.integers(0, w.size, w.size // 8)] = 0x8000
    w[7 * cols + 3], w[9 * cols + cols - 1], w[11 * cols + 40] = 0x7F80, 0x7FC0, 1
    x = np.ldexp(rng.standard_normal(n_tok * cols), rng.integers(-150, 100, n_tok * cols)).astype(np.float32)
    x[rng.integers(0, x.size, x.size // 8)] = -0.0
    x.reshape(n_tok, cols)[3] = -0.0
    x.reshape(n_tok, cols)[5, -1] = np.inf
    x.reshape(n_tok, cols)[6, 40] = 3e38
    x.reshape(n_tok, cols)[7, 5] = np.nan
    wt = N.Weight.bf16(w, rows, cols)
    y = np.zeros(n_tok * rows, np.float32)
    N.gemv_batch(wt, x, cols, y, rows, n_tok)
    ref = oracle.gemv_bf16(w, x, rows, cols, n_tok, cols, rows)
    nan = np.isnan(ref)
    assert np.array_equal(np.isnan(y), nan) and nan.reshape(n_tok, rows)[7].all() and not nan.all()
    assert np.array_equal(y[~nan].view(np.uint32), ref[~nan].view(np.uint32))
    wt.free()


# The splits of two row groups, by the number of 16-vector groups in a token
# tile: 32 vectors at most (a full tile; tiles of two and one), 64 at most in a
# ring of two stages (tiles of three; of four and three; of four), each with
# a ragged last row tile, and stages that are whole or not.
LARGE = [(6163, 17, 2), (2470, 75, 2), (6841, 33, 3), (2934, 103, 3), (5141, 64, 3)]


def split_of(rows, n_tok):
    import torch
    f = N.lib()._ZN3nnh11batch_splitEiii  # nnh::batch_split(int rows, int n_tok, int cus)
    return f(rows, n_tok, torch.cuda.get_device_properties(0).multi_processor_count)


@pytest.mark.parametrize("dtype", [1, 2])
@pytest.mark.parametrize("cols", [96, 544, 1024, 1312])
@pytest.mark.parametrize("rows,n_tok,split", LARGE)
def test_f32_batch_large_splits(oracle, dtype, rows, cols, n_tok, split):
    assert split_of(rows, n_tok) == split
    pad = 4 * (n_tok & 1)
    rng = np.random.default_rng(rows + cols)
    x = np.ldexp(rng.standard_normal(n_tok * (cols + pad)), rng.integers(-140, 60, n_tok * (cols + pad))).astype(np.float32)
    x[rng.integers(0, x.size, x.size // 8)] = -0.0
    y, ref = run(oracle, dtype, rows, cols, n_tok, pad, x=x)
    assert np.array_equal(y.view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("path,cols", [("quad", 24), ("quad", 1304), ("quad", 512), ("row8", 264), ("row8", 1304),
                                       ("row32", 96), ("row32", 1312), ("row32", 768)])
@pytest.mark.parametrize("rows,n_tok,split", LARGE)
def test_bf16_batch_large_splits(oracle, path, rows, cols, n_tok, split):
    rows = (rows + 3) // 4 * 4 if path == "quad" else rows | 1
    assert split_of(rows, n_tok) == split
    test_bf16_batch_bit_exact(oracle, rows, cols, n_tok, 4 * (n_tok & 1))


@pytest.mark.parametrize("fmt", ["q8", "q4", "bf16"])
def test_more_vectors_than_one_launch_holds(fmt):
    """65552 rows take 16368 vectors a launch: those around the slice's end as alone."""
    import torch
    rows, cols, n_tok, edge = 65552, 32, 16400, 16368
    rng = np.random.default_rng(9)
    s = (rng.uniform(1e-2, 2e-2, (rows, 1)).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16).view(np.int16)
    if fmt == "q8":
        w = N.Weight.q8_0(rng.integers(-127, 128, (rows, cols), dtype=np.int8), s, rows, cols)
    elif fmt == "q4":
        w = N.Weight.q4(rng.integers(0, 256, (rows, cols // 2), dtype=np.uint8), s, s, rows, cols)
    else:
        w = N.Weight.bf16((rng.standard_normal((rows, cols)).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16),
                          rows, cols)
    x, y = torch.randn(n_tok, cols, device="cuda"), torch.full((n_tok, rows), 7.0, device="cuda")
    st = torch.cuda.current_stream().cuda_stream
    w.prepare(N.ACT_F32, n_tok)
    N.gemv_batch_dev(w, x.data_ptr(), cols, y.data_ptr(), rows, n_tok, N.ACT_F32, st)
    few = torch.full((16, rows), 7.0, device="cuda")
    for t in (0, edge - 16, edge, n_tok - 16):
        N.gemv_batch_dev(w, x[t:].data_ptr(), cols, few.data_ptr(), rows, 16, N.ACT_F32, st)
        assert torch.equal(y[t:t + 16], few), t
    w.free()
