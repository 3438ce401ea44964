"""The int8 GEMM's scale products, which the BF16 matrix unit forms: bit for bit
the kernel's sum with every product rounded to f32 as usual, for weight and
activation scales from zero and the smallest subnormals to infinity and NaN,
products that under- and overflow among them. Up to 8 blocks are one f32 sum in
block order (Q4: after each pair of blocks its two bias terms), 16 are two, added
in f64."""
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


def f32(bits):
    return (bits.astype(np.uint32) << 16).view(np.float32)


def fma(a, b, c):
    """f32 a * b + c rounded once: the sum with 64 bits of mantissa, and where that
    is halfway between two f32 values, a step towards the part it left out."""
    p, c = a.astype(np.longdouble) * b.astype(np.longdouble), np.broadcast_to(c, np.broadcast(a, b).shape).astype(np.longdouble)
    s = p + c
    t = s - p
    left = (p - (s - t)) + (c - t)  # exact
    f = s.astype(np.float32)
    g = np.nextafter(f, np.where(s > f, np.float32(np.inf), np.float32(-np.inf))).astype(np.longdouble)
    half = (s - f == g - s) & (left != 0) & np.isfinite(s)
    return np.where(half, np.nextafter(s, np.where(left > 0, np.longdouble(np.inf), -np.longdouble(np.inf))), s).astype(np.float32)


@pytest.mark.parametrize("dtype", [1, 2])
@pytest.mark.parametrize("nb", [1, 5, 8, 16])
def test_scales_of_every_kind(dtype, nb):
    import torch
    rows, n_tok, cols = 96, 33, 32 * nb
    rng = np.random.default_rng(100 * nb + dtype)
    special = np.array([0, 1, 2, 0x7F, 0x80, 0x7F7F, 0x7F80, 0x7FC0, 0x8001, 0x3F80], np.uint16)
    s = rng.integers(0, 0x7F80, (rows, nb)).astype(np.uint16)         # every exponent, subnormals among them
    tame = rng.random((rows, nb)) < 0.5
    s[tame] = rng.integers(0x3C00, 0x4000, int(tame.sum()))
    odd = rng.random((rows, nb)) < 0.04
    s[odd] = rng.choice(special, int(odd.sum()))
    b = rng.integers(0x3800, 0x4000, (rows, nb)).astype(np.uint16) | (rng.integers(0, 2, (rows, nb)) << 15).astype(np.uint16)
    if dtype == 1:
        q = rng.integers(-127, 128, (rows, nb, 32), dtype=np.int8)
        w = N.Weight.q8_0(q.reshape(rows, cols), s.view(np.int16), rows, cols)
        qw = q.astype(np.int64)
    else:
        p = rng.integers(0, 256, (rows, nb, 16), dtype=np.uint8)
        w = N.Weight.q4(p.reshape(rows, cols // 2), s.view(np.int16), b.view(np.int16), rows, cols)
        qw = np.concatenate([p & 15, p >> 4], 2).astype(np.int64)
    e = np.where(rng.random((n_tok, nb, 1)) < 0.5, rng.integers(-4, 4, (n_tok, nb, 1)), rng.integers(-146, 120, (n_tok, nb, 1)))
    x = np.ldexp(rng.standard_normal((n_tok, nb, 32)), e).astype(np.float32)
    x[1, 0, 3], x[2, nb - 1, 0], x[3] = np.inf, np.nan, 0
    x[4, 0] = np.ldexp(rng.standard_normal(32), -124)  # a subnormal scale
    dx, y = torch.from_numpy(x.reshape(n_tok, cols)).cuda(), torch.empty(n_tok, rows, device="cuda")
    off_s, _, size = N.act_layout_ex(N.ACT_I8, cols, n_tok)
    buf = torch.zeros(size, dtype=torch.uint8, device="cuda")
    w.prepare(N.ACT_I8, n_tok)
    torch.cuda.synchronize()
    N.quantize_act_ex_dev(N.ACT_I8, dx.data_ptr(), cols, cols, n_tok, buf.data_ptr())
    N.gemv_act_dev(w, N.ACT_I8, buf.data_ptr(), n_tok, y.data_ptr(), rows)
    N.sync()
    a = buf.cpu().numpy()
    qx = a[:n_tok * cols].view(np.int8).reshape(n_tok, nb, 32).astype(np.int64)
    sx = f32(a[off_s:off_s + 2 * n_tok * nb].view(np.uint16).reshape(n_tok, nb))
    assert (sx == 0).any() and np.isinf(sx).any() and ((sx > 0) & (sx < 2.0 ** -126)).any()
    total = np.zeros((n_tok, rows))
    with np.errstate(all="ignore"):
        for g in range(0, nb, 8):
            acc = np.zeros((n_tok, rows), np.float32)
            for j in range(g, min(g + 8, nb)):
                P = (qx[:, j] @ qw[:, j].T).astype(np.float32)  # exact: below 2^19
                acc = fma(P, sx[:, j, None] * f32(s[:, j])[None], acc)
                if dtype == 2 and (j & 1 or j == nb - 1):
                    for i in range(j & ~1, j + 1):
                        X = sx[:, i] * qx[:, i].sum(1).astype(np.float32)
                        acc = fma(f32(b[:, i])[None], X[:, None], acc)
            total += acc.astype(np.float64)
        want = total.astype(np.float32)
    got, nan = y.cpu().numpy(), np.isnan(want)
    assert nan.any() and np.isinf(want).any() and not nan.all(0).all()
    assert np.array_equal(np.isnan(got), nan)
    assert np.array_equal(got[~nan].view(np.uint32), want[~nan].view(np.uint32))
    w.free()
