"""The int8 GEMM where its tiles are not whole rounds of the CUs: the last round
is split along K (one spare tile, half a round, rounds that the split does not
take), against the exact sum of the quantized product and the bits of a whole
tile; the fixed-scratch call gives the ordinary call's bits; and scratch reserved for a
batch serves smaller ones under capture."""
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


def matrix(dtype, rows, cols, seed):
    rng = np.random.default_rng(seed)
    nb = cols // 32

    def bf16(a):
        return (a.astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)

    s = bf16(rng.uniform(1e-4, 4e-4, (rows, nb)))
    if dtype == 1:
        q = rng.integers(-127, 128, (rows, cols), dtype=np.int8)
        return (q, s), N.Weight.q8_0(q, s.view(np.int16), rows, cols)
    q, b = rng.integers(0, 256, (rows, cols // 2), dtype=np.uint8), bf16(rng.uniform(-4e-3, 4e-3, (rows, nb)))
    return (q, s, b), N.Weight.q4(q, s.view(np.int16), b.view(np.int16), rows, cols)


def run(w, x, call=None):
    import torch
    n, cols = x.shape
    y = torch.empty(n, w.rows(), device="cuda")
    st = torch.cuda.current_stream().cuda_stream
    w.prepare(N.ACT_I8, n)
    (call or N.gemv_batch_dev)(w, x.data_ptr(), cols, y.data_ptr(), w.rows(), n, N.ACT_I8, st)
    torch.cuda.synchronize()
    return y


@pytest.mark.parametrize("dtype", [1, 2])
@pytest.mark.parametrize("rows,cols,n_tok", [
    (85 * 128 + 1, 2048, 300),   # 258 tiles: 2 left, 8 splits
    (97 * 128 - 5, 1504, 500),   # 388 tiles: 132 left, one split: the round stays whole
    (96 * 128, 3104, 512),       # 384 tiles: 128 left, 2 splits of 97 blocks
    (256 * 128, 1600, 100),      # a whole round
])
def test_split_tail(dtype, rows, cols, n_tok):
    import torch
    parts, w = matrix(dtype, rows, cols, rows + cols)
    nb = cols // 32
    g = torch.Generator(device="cuda")
    g.manual_seed(rows)
    x = torch.randn(n_tok, cols, generator=g, device="cuda")
    y = run(w, x)
    w.free()
    off_s, _, size = N.act_layout_ex(N.ACT_I8, cols, n_tok)
    buf = torch.zeros(size, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    N.quantize_act_ex_dev(N.ACT_I8, x.data_ptr(), cols, cols, n_tok, buf.data_ptr())
    N.sync()
    qx = buf[:n_tok * cols].view(torch.int8).view(n_tok, nb, 32).double()
    sx = buf[off_s:off_s + 2 * n_tok * nb].view(torch.bfloat16).view(n_tok, nb, 1).double()
    q, s = torch.from_numpy(parts[0]).cuda(), torch.from_numpy(parts[1].view(np.int16)).cuda().view(torch.bfloat16)
    if dtype == 2:
        q = q.view(rows, nb, 16)
        q = torch.cat([q & 15, q >> 4], 2)
    wd = q.view(rows, nb, 32).double() * s.double().unsqueeze(2)
    if dtype == 2:
        wd = wd + torch.from_numpy(parts[2].view(np.int16)).cuda().view(torch.bfloat16).double().unsqueeze(2)
    exact = (qx * sx).view(n_tok, cols) @ wd.view(rows, cols).T.contiguous()
    # Groups of 8 blocks are summed in f32 (Q4: two terms a block), everything else
    # in f64 and rounded once: 8 (16) roundings of at most the groups' magnitude.
    mag = (qx * sx).abs().view(n_tok, cols) @ wd.abs().view(rows, cols).T.contiguous()
    if dtype == 2:  # quant and bias terms one by one: |q s| + |bias| <= 0..15 s + |bias|
        up = q.view(rows, nb, 32).double() * s.double().unsqueeze(2) + torch.from_numpy(
            parts[2].view(np.int16)).cuda().view(torch.bfloat16).double().abs().unsqueeze(2)
        mag = (qx * sx).abs().view(n_tok, cols) @ up.view(rows, cols).T.contiguous()
    bound = (8 if dtype == 1 else 16) * 2.0 ** -24 * mag + 2.0 ** -24 * exact.abs()
    assert bool(((y.double() - exact).abs() <= bound).all())


@pytest.mark.parametrize("dtype", [1, 2])
@pytest.mark.parametrize("rows,cols,n_tok,roll", [
    (86 * 128, 2048, 384, 128),         # 258 tiles: 2 left, 8 splits
    (84 * 128, 3584, 512, 20 * 128),    # 336 tiles: 80 left, 3 splits of 14 groups of 8 blocks
    (96 * 128 - 9, 3200, 500, 32 * 128),  # 384 tiles: 128 left, 2 splits of 12 groups and a half
])
def test_split_tail_keeps_the_bits(dtype, rows, cols, n_tok, roll):
    """The tail's rows are computed whole when they are the matrix's first ones: the same bits."""
    import torch
    parts, w = matrix(dtype, rows, cols, rows + n_tok)
    make = N.Weight.q8_0 if dtype == 1 else N.Weight.q4
    turned = [np.roll(p.reshape(rows, -1), roll, axis=0) for p in parts]
    wt = make(*[p if i == 0 else p.view(np.int16) for i, p in enumerate(turned)], rows, cols)
    x = torch.randn(n_tok, cols, device="cuda")
    y, yt = run(w, x), run(wt, x)
    assert torch.equal(y, yt.roll(-roll, 1))
    w.free()
    wt.free()


def test_fixed_scratch_gives_the_same_bits():
    """Activations that leave no room for the tail's parts in the fixed scratch
    (64 MiB) are multiplied as by the ordinary call, also where a tail computed
    whole would round otherwise: f32 groups 1, 2^-24, then 2^-54 each add up to
    a tie in one f64 chain, and above it in the tail's parts."""
    import torch
    rows, cols, n_tok = 30 * 128, 18944, 1100  # 270 tiles, 14 split
    nb = cols // 32
    _, w = matrix(2, rows, cols, 5)
    x = torch.randn(n_tok, cols, device="cuda")
    assert torch.equal(run(w, x), run(w, x, N.gemv_batch_dev_noalloc))
    w.free()
    q = np.zeros((rows, nb, 32), np.int8)
    q[:, ::8, 1] = 1
    s = np.full(nb, 2.0 ** -54, np.float32)
    s[0], s[8] = 1, 2.0 ** -24
    s = np.tile((s.view(np.uint32) >> 16).astype(np.uint16), (rows, 1))
    w = N.Weight.q8_0(q.reshape(rows, cols), s.view(np.int16), rows, cols)
    x = torch.zeros(n_tok, nb, 32, device="cuda")
    x[..., 0], x[..., 1] = 127, 1  # scale 1, quants 127 and 1
    x = x.view(n_tok, cols)
    y = run(w, x)
    assert torch.equal(y, run(w, x, N.gemv_batch_dev_noalloc))
    assert bool((y[:, :28 * 128] == 1).all()) and bool((y[-50:, -128:] == 1 + 2.0 ** -23).all())
    # What does not fit by itself is refused as before.
    x, y = torch.zeros(2000, cols, device="cuda"), torch.empty(2000, rows, device="cuda")
    w.prepare(N.ACT_I8, 2000)
    with pytest.raises(N.InvalidArgument, match="no-alloc maximum"):
        N.gemv_batch_dev_noalloc(w, x.data_ptr(), cols, y.data_ptr(), rows, 2000, N.ACT_I8)
    w.free()


@pytest.mark.parametrize("act", [1, 2])
@pytest.mark.parametrize("rows,cols,n_tok", [
    (170 * 128, 2048, 256),  # 340 tiles, 84 left in 3 parts; 128 vectors: 170 in 2 parts
    (102 * 128, 3584, 400),  # 408 tiles, whole; 128 vectors: 102 in 3 parts
])
def test_reserved_scratch_holds_every_smaller_batch(act, rows, cols, n_tok):
    import torch
    _, w = matrix(1, rows, cols, 7)
    x, y = torch.randn(n_tok, cols, device="cuda"), torch.empty(n_tok, rows, device="cuda")
    st = torch.cuda.Stream()
    w.prepare(act, 1).prepare(act, 16).prepare(act, n_tok)
    N.stream_reserve(w, act, n_tok, st.cuda_stream)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    for n in (n_tok, 1, 5, 16, 17, 128, 129, n_tok - 1):
        N.gemv_batch_dev(w, x.data_ptr(), cols, y.data_ptr(), rows, n, act, st.cuda_stream)
        torch.cuda.synchronize()
        # A scratch that grows at least doubles (60 MiB and more here); a kernel's first launch takes 2 MiB.
        assert free - torch.cuda.mem_get_info()[0] < 16 << 20, n
    N.stream_release(st.cuda_stream)
    w.free()


def test_reserved_stream_serves_smaller_batches_under_capture():
    import torch
    rows, cols = 86 * 128, 2048
    _, w = matrix(1, rows, cols, 6)
    x = torch.randn(768, cols, device="cuda")
    eager = run(w, x[:384])  # 258 tiles, a split tail
    st = torch.cuda.Stream()
    N.stream_reserve(w, N.ACT_I8, 768, st.cuda_stream)
    y = torch.empty(384, rows, device="cuda")
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=st):
        N.gemv_batch_dev(w, x.data_ptr(), cols, y.data_ptr(), rows, 384, N.ACT_I8, st.cuda_stream)
    for _ in range(3):
        y.fill_(0)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, eager)
    del graph
    N.stream_release(st.cuda_stream)
    w.free()
