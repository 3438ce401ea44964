"""The activation quantizers over several vectors, against nncpu's encoder (and
the power-of-two one) per vector: quants, scales, the f64 pairs and the
block-major copies, at the edges of their tiles (8 vectors, 4 and 16 blocks),
with strided and unaligned rows, zero blocks, denormals, infinities and NaN."""
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


@pytest.mark.parametrize("act", [1, 2])
@pytest.mark.parametrize("cols,n_tok,pad", [(32, 17, 0), (96, 16, 3), (128, 33, 1), (544, 24, 0), (1152, 3, 4),
                                            (1184, 40, 7), (4096, 65, 0)])
def test_batched_quantizer_bits(oracle, act, cols, n_tok, pad):
    import torch
    nb, xs = cols // 32, cols + pad
    rng = np.random.default_rng(cols * 131 + n_tok)
    x = np.ldexp(rng.standard_normal(n_tok * xs), rng.integers(-20, 20, n_tok * xs)).astype(np.float32)
    v = x.reshape(n_tok, xs)
    v[0, :32] = 0.0
    v[1, :32] = np.ldexp(v[1, :32], -140)
    v[2, 5] = np.inf
    v[2, 7] = np.nan
    off_s, off_sx, size = N.act_layout_ex(act, cols, n_tok)
    buf = torch.zeros(size, dtype=torch.uint8, device="cuda")
    dx = torch.from_numpy(x).cuda()
    torch.cuda.synchronize()
    N.quantize_act_ex_dev(act, dx.data_ptr(), xs, cols, n_tok, buf.data_ptr())
    N.sync()
    b = buf.cpu().numpy()
    q = b[:n_tok * cols].view(np.int8).reshape(n_tok, cols)
    s = b[off_s:off_s + 2 * n_tok * nb].view(np.uint16).reshape(n_tok, nb)
    sx = b[off_sx:off_sx + 16 * n_tok * nb].view(np.float64).reshape(n_tok, nb, 2)
    encode = oracle.quantize_act if act == 1 else oracle.quantize_act_mx
    for t in range(n_tok):
        rq, rs = encode(v[t, :cols].copy())
        assert np.array_equal(q[t], rq) and np.array_equal(s[t], np.asarray(rs).view(np.uint16))
    scale = (s.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    total = q.reshape(n_tok, nb, 32).astype(np.int64).sum(2)
    # Not the infinite value's block: its scale is infinite (Q8_0), or its scale
    # times the quant sum may pass f32's range, in which the MX one is formed.
    fin = np.isfinite(scale)
    fin[2, 0] = False
    assert np.array_equal(sx[..., 0][fin], scale[fin])
    assert np.array_equal(sx[..., 1][fin], (scale * total)[fin])
    pad_tok = (n_tok + 127) // 128 * 128
    off_t = off_sx + (16 * n_tok * nb + 255) // 256 * 256
    sxt = b[off_t:off_t + 8 * nb * pad_tok].view(np.float32).reshape(2, nb, pad_tok)[:, :, :n_tok]
    assert np.array_equal(sxt[0].T[fin], scale[fin].astype(np.float32))
    assert np.array_equal(sxt[1].T[fin], (scale * total)[fin].astype(np.float32))


@pytest.mark.parametrize("act", [1, 2])
def test_more_vectors_than_a_grid_dimension_holds(act):
    """8 * 65535 vectors and more: the last ones are quantized as they are alone."""
    import torch
    cols, n_tok = 32, 8 * 65536 + 9
    x = torch.randn(n_tok, cols, device="cuda")
    bufs = []
    for first in (0, n_tok - 20):
        off_s, off_sx, size = N.act_layout_ex(act, cols, n_tok - first)
        buf = torch.zeros(size, dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        N.quantize_act_ex_dev(act, x[first:].data_ptr(), cols, cols, n_tok - first, buf.data_ptr())
        N.sync()
        q, s = buf[:(n_tok - first) * cols], buf[off_s:off_s + 2 * (n_tok - first)]
        bufs.append((q[-20 * cols:].cpu(), s[-40:].cpu()))
    assert torch.equal(bufs[0][0], bufs[1][0]) and torch.equal(bufs[0][1], bufs[1][1])
