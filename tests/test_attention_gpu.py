"""The batched attention kernel (layers_gpu.hip, f32 matrix unit) against the
CPU forward, through whole layers: greedy tokens, per-layer states and K/V cache
bit for bit. Every head_dim, query rows that fill, half fill and overflow the
16-row tiles, key ranges around the 16-key tiles, the 4-key groups, the 8-key
sums and the 256-key block, with causal edges (batches of several tokens per
tile) and sliding windows (edges at both ends, whole keys shared by no token)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def N():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import nncpu_amd as N
    N.init(0)
    return N


@pytest.mark.parametrize("head_dim,n_head,n_kv,window,prompt,batch", [
    (32, 2, 2, 0, 50, 50),     # one query head: 32 tokens per tile
    (32, 10, 2, 5, 70, 33),    # 6 tokens per tile, windows shorter than a tile's spread
    (64, 3, 1, 0, 130, 64),    # 10 tokens, 30 rows
    (64, 17, 1, 20, 37, 37),   # one token per tile, a row into the second row tile
    (128, 7, 1, 0, 300, 100),  # Qwen2.5's 7 heads: 4 tokens, 28 rows; two blocks merged
    (128, 32, 1, 0, 261, 61),  # full tiles of one token
    (128, 2, 1, 257, 280, 280),  # a window a key longer than the block: partial first blocks
    (256, 4, 1, 24, 60, 31),   # 16-row tiles
    (256, 3, 3, 0, 259, 129),
])
def test_batched_attention_bit_exact(N, head_dim, n_head, n_kv, window, prompt, batch):
    from nncpu_amd.models import Model, qwen2_config
    cfg = qwen2_config(n_layer=2, n_embd=128, n_head=n_head, n_kv=n_kv, n_ff=256, n_vocab=512, n_ctx=320,
                       head_dim=head_dim)
    if window:
        cfg.window, cfg.swa_period = window, 2  # layer 0 slides
    model = Model.random(cfg, seed=head_dim + n_head + prompt)
    toks = np.random.default_rng(prompt).integers(0, cfg.n_vocab, prompt).astype(np.int32)
    tc, hc, kc, vc = model.cpu_generate(toks, 3, batch=batch)
    dev = model.device(n_batch=batch)
    try:
        tg, hg, kg, vg = dev.generate(toks, 3, batch=batch)
    finally:
        dev.free()
    assert np.array_equal(tg, tc) and np.array_equal(hg, hc)
    assert np.array_equal(kg, kc) and np.array_equal(vg, vc)
