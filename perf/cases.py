"""The work whose speed is tracked: nncpu's weight matmuls and forwards as a
serving program calls them.

A case is a dict of plain values. ``kind`` names the entry point:

* ``matmul``: one weight matrix against ``tokens`` vectors through
  ``gemv_batch_dev``: one vector in decode, 2 to 16 in speculative verify and
  in the reference's 16-token prompt batches, more in a whole prompt.
  ``act`` is the activation mode ("f32" bit-exact, "i8", "mx"), ``fmt`` the
  weight format ("q8", "q4", "bf16").
* ``head``: the vocabulary projection and its greedy token
  (``model_argmax_dev``).
* ``model``: ``DeviceForward`` over ``tokens`` tokens at position ``pos`` and
  the last token's logits: a prompt's prefill, or one decode step.
* ``load``: one matrix of a GGUF file decoded and re-encoded on the device
  (``Weight.from_gguf``) and read back in nncpu's layout.

Inputs: weights 0.02 N(0, 1) in blocks of 32 (BF16 scale, for Q4 a BF16 bias),
activations N(0, 1), norms 1 + 0.1 N(0, 1).
"""
import math

import numpy as np
import torch

import nncpu_amd as N
from nncpu_amd import models

ACTS = {"f32": N.ACT_F32, "i8": N.ACT_I8, "mx": N.ACT_MXI8}


def matmul(fmt, rows, cols, tokens, act):
    return {"kind": "matmul", "fmt": fmt, "rows": rows, "cols": cols, "tokens": tokens, "act": act}


def model(fmt, act, tokens, pos, layers, embd, heads, kv_heads, head_dim, ffn, vocab, arch):
    return {"kind": "model", "fmt": fmt, "act": act, "tokens": tokens, "pos": pos, "layers": layers, "embd": embd,
            "heads": heads, "kv_heads": kv_heads, "head_dim": head_dim, "ffn": ffn, "vocab": vocab, "arch": arch}


def listed():
    qwen = dict(embd=3584, heads=28, kv_heads=4, head_dim=128, ffn=18944, vocab=32768, layers=2, arch="qwen2")
    cases = {
        # The smallest call of a decode step: a Llama-3-8B-shaped k or v projection.
        "decode_i8_q4_small": matmul("q4", 1024, 4096, 1, "i8"),
        # Decode in the default bit-exact mode at long rows: a Llama-3-8B-shaped down projection.
        "decode_f32_q4_long": matmul("q4", 4096, 14336, 1, "f32"),
        # The greedy token of every decode step: Gemma-3's vocabulary, the tallest matrix there is.
        "head_f32_q8": {"kind": "head", "fmt": "q8", "rows": 262144, "cols": 1152},
        # Speculative verify: 8 draft tokens against a Gemma-4-E2B-like down projection.
        "verify_i8_q8": matmul("q8", 1536, 6144, 8, "i8"),
        # The reference's prompt batch (16 tokens) in its own arithmetic: Qwen2.5-7B's down projection.
        "batch_f32_q4": matmul("q4", 3584, 18944, 16, "f32"),
        # A whole prompt of an odd length in the bit-exact mode: a Llama-3-8B-shaped gate projection.
        "prompt_f32_q8": matmul("q8", 14336, 4096, 301, "f32"),
        # A whole prompt on int8 activations: Qwen2.5-7B's gate projection.
        "prompt_i8_q8": matmul("q8", 18944, 3584, 512, "i8"),
        # A prompt of an odd length on power-of-two-scaled blocks: Qwen2.5-7B's down projection.
        "prompt_mx_q4": matmul("q4", 3584, 18944, 509, "mx"),
        # A 16-token batch against a matrix kept in BF16.
        "batch_bf16": matmul("bf16", 6144, 1536, 16, "f32"),
        # Model load: one Q4_K matrix of a file into nncpu's 8-bit layout.
        "load_q4k_q8": {"kind": "load", "type": "q4_k", "fmt": "q8", "rows": 4096, "cols": 4096},
        # Prefill of a 512-token prompt through Qwen2.5-7B-shaped layers, the configuration that serves prompts.
        "prefill_model_mx": model("q8", "mx", 512, 0, **qwen),
        # One decode step of the same layers, 700 tokens into the context.
        "decode_model_i8": model("q8", "i8", 1, 700, **qwen),
    }
    return [dict(c, name=n) for n, c in cases.items()]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["matmul"] * 6 + ["bf16", "head", "prefill", "decode", "load"])
    if kind == "matmul":
        act = rng.choice(["f32", "i8", "mx"])
        tokens = rng.choice([1, _log(rng, 2, 16), _log(rng, 17, 512)])
        rows, cols = _log(rng, 256, 38000), 32 * _log(rng, 32, 592)
        # At most the work of the largest listed matmul in the mode.
        rows = max(256, min(rows, int((14336 * 4096 * 301 if act == "f32" else 18944 * 3584 * 512) / (cols * tokens))))
        return matmul(rng.choice(["q8", "q4"]), rows, cols, tokens, act)
    if kind == "bf16":
        cols = rng.choice([_log(rng, 1024, 4096), 8 * _log(rng, 128, 512), 32 * _log(rng, 32, 128)])
        return matmul("bf16", _log(rng, 256, 8192), cols, _log(rng, 1, 32), "f32")
    if kind == "head":
        return {"kind": "head", "fmt": rng.choice(["q8", "q4"]), "rows": _log(rng, 32000, 262144),
                "cols": 32 * _log(rng, 32, 64)}
    if kind == "load":
        return {"kind": "load", "type": rng.choice(["q4_k", "f16", "bf16"]), "fmt": rng.choice(["q8", "q4"]),
                "rows": _log(rng, 256, 4096), "cols": 256 * _log(rng, 4, 16)}
    head_dim, kv_heads, group = rng.choice([64, 128]), rng.choice([2, 4]), rng.choice([1, 3, 4, 7, 8])
    act = rng.choice(["f32", "i8", "mx"])
    if kind == "decode":
        tokens, pos = 1, _log(rng, 30, 3000)
    else:
        tokens, pos = _log(rng, 17, 512), rng.choice([0, _log(rng, 16, 1500)])
    if act == "f32":
        tokens = min(tokens, 64)
    return model(rng.choice(["q8", "q4"]), act, tokens, pos, 2, 32 * _log(rng, 32, 112), group * kv_heads, kv_heads,
                 head_dim, 32 * _log(rng, 64, 344), 32000, rng.choice(["qwen2", "llama"]))


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) % (1 << 62))
    return g


def _parts(fmt, rows, cols, g, std=0.02):
    """A random matrix in nncpu's split layout, on the GPU: q8 (quants, scales),
    q4 (packed nibbles, scales, biases), bf16 (values,); scales and biases BF16."""
    if fmt == "bf16":
        return (torch.randn(rows, cols, generator=g, device="cuda").mul_(std).bfloat16(),)
    w = torch.randn(rows, cols // 32, 32, generator=g, device="cuda").mul_(std)
    if fmt == "q8":
        s = (w.abs().amax(2, keepdim=True) / 127).bfloat16()
        q = (w / s.float()).round_().clamp_(-127, 127).to(torch.int8)
        return q.view(rows, cols), s.view(rows, -1)
    lo, hi = w.amin(2, keepdim=True), w.amax(2, keepdim=True)
    s, b = ((hi - lo) / 15).bfloat16(), lo.bfloat16()
    q = ((w - b.float()) / s.float()).round_().clamp_(0, 15).to(torch.uint8)
    return (q[..., :16] | (q[..., 16:] << 4)).view(rows, cols // 2), s.view(rows, -1), b.view(rows, -1)


def _host(t):
    return (t.view(torch.int16) if t.dtype == torch.bfloat16 else t).cpu().numpy()


def _weight(fmt, parts, rows, cols):
    make = {"q8": N.Weight.q8_0, "q4": N.Weight.q4, "bf16": N.Weight.bf16}[fmt]
    return make(*[_host(p) for p in parts], rows, cols)


def _dense(fmt, parts):
    """The matrix of `parts` in 64 bits."""
    if fmt == "bf16":
        return parts[0].double()
    rows, nb = parts[1].shape
    s = parts[1].double().unsqueeze(2)
    if fmt == "q8":
        return (parts[0].view(rows, nb, 32).double() * s).view(rows, -1)
    p = parts[0].view(rows, nb, 16)
    q = torch.cat([p & 15, p >> 4], 2).double()
    return (q * s + parts[2].double().unsqueeze(2)).view(rows, -1)


def _activations(x, act):
    """What mode `act` makes of the f32 vectors x, in 64 bits: blocks of 32 as
    int8 times a BF16 scale (the Q8_0 encoder) or a power of two."""
    if act == "f32":
        return x.double()
    b = x.float().reshape(x.shape[0], -1, 32)
    amax = b.abs().amax(2, keepdim=True)
    if act == "i8":
        s = (amax * np.float32(1 / 127).item()).bfloat16().float()
    else:
        s = torch.exp2(torch.ceil(torch.log2(amax.double() / 127)).clamp_(-126, 127)).float()
    inv = torch.where(s > 0, 1 / s, torch.zeros_like(s))
    q = torch.round(b * inv).clamp_(-127, 127)
    return (q.double() * s.double()).view(x.shape[0], -1)


def _mm(fmt, parts, x, act):
    """x W^T in 64 bits, by slices of rows."""
    xd = _activations(x, act)
    step = max(1, (1 << 26) // xd.shape[1])
    return torch.cat([xd @ _dense(fmt, [p[i:i + step] for p in parts]).T.contiguous()
                      for i in range(0, parts[0].shape[0], step)], 1)


def _model_parts(c, seed):
    """The weights of a ``model`` case: fused [q; k; v] and [gate; up], o,
    down per layer, the head (also the embedding table), norms, biases and
    the tokens up to and including the pass's own."""
    g = _gen(seed)
    e, f, hd = c["embd"], c["ffn"], c["head_dim"]
    qd, kvd = c["heads"] * hd, c["kv_heads"] * hd
    layers = [[_parts(c["fmt"], r, k, g) for r, k in ((qd + 2 * kvd, e), (e, qd), (2 * f, e), (e, f))]
              for _ in range(c["layers"])]
    head = _parts(c["fmt"], c["vocab"], e, g)
    rng = np.random.default_rng(seed)
    norms = (1 + 0.1 * rng.standard_normal((4 * e + 2 * hd) * c["layers"] + e)).astype(np.float32)
    biases = (0.02 * rng.standard_normal((qd + 2 * kvd) * c["layers"])).astype(np.float32)
    tokens = rng.integers(0, c["vocab"], c["pos"] + c["tokens"]).astype(np.int32)
    return layers, head, norms, biases if c["arch"] == "qwen2" else None, tokens


def _config(c):
    make = models.qwen2_config if c["arch"] == "qwen2" else models.llama_config
    return make(c["layers"], c["embd"], c["heads"], c["kv_heads"], c["ffn"], c["vocab"], 4096, c["head_dim"],
                wtype=2 if c["fmt"] == "q4" else N.Q8_0)


def _gguf_blocks(c, seed):
    rng = np.random.default_rng(seed)
    n = c["rows"] * c["cols"]
    if c["type"] == "f16":
        return 1, (0.02 * rng.standard_normal(n, np.float32)).astype(np.float16).view(np.uint8)
    if c["type"] == "bf16":
        return 30, (0.02 * rng.standard_normal(n, np.float32)).view(np.uint16)[1::2].copy().view(np.uint8)
    # Q4_K: d and dmin (f16), 12 bytes of packed 6-bit scales and mins, 128 bytes of nibbles per 256 values.
    blocks = rng.integers(0, 256, (n // 256, 144), dtype=np.uint8)
    blocks[:, :4] = rng.uniform(2e-5, 2e-4, (n // 256, 2)).astype(np.float16).view(np.uint8)
    return 12, blocks.reshape(-1)


def prepare(case, seed):
    N.init(0)
    c = case
    if c["kind"] == "load":
        ggml_type, blocks = _gguf_blocks(c, seed)
        return {"case": c, "type": ggml_type, "blocks": blocks}
    if c["kind"] == "model":
        layers, head, norms, biases, tokens = _model_parts(c, seed)
        cfg, e, f, hd = _config(c), c["embd"], c["ffn"], c["head_dim"]
        qd, kvd = c["heads"] * hd, c["kv_heads"] * hd
        ws = []
        for qkv, o, gu, down in layers:
            ws += [_weight(c["fmt"], qkv, qd + 2 * kvd, e), None, None, _weight(c["fmt"], o, e, qd),
                   _weight(c["fmt"], gu, 2 * f, e), None, _weight(c["fmt"], down, e, f)]
        ws.append(_weight(c["fmt"], head, c["vocab"], e))
        batch = max(c["tokens"], min(c["pos"], 512), 1)
        stream = torch.cuda.Stream()
        fwd = models.DeviceForward(cfg, ws, norms, biases, ws[-1], batch, ACTS[c["act"]], stream.cuda_stream)
        tok = torch.from_numpy(tokens).cuda()
        torch.cuda.synchronize()
        for p in range(0, c["pos"], batch):
            fwd.forward_dev(tok[p:].data_ptr(), min(batch, c["pos"] - p), p)
        stream.synchronize()
        logits = torch.empty(c["vocab"], device="cuda")
        return {"case": c, "fwd": fwd, "tokens": tok[c["pos"]:].clone(), "logits": logits, "stream": stream}
    g = _gen(seed)
    w = _weight(c["fmt"], _parts(c["fmt"], c["rows"], c["cols"], g), c["rows"], c["cols"])
    state = {"case": c, "w": w}
    if c["kind"] == "head":
        w.prepare(N.ACT_F32, 1)
        state["x"] = torch.randn(c["cols"], generator=g, device="cuda")
        state["y"] = torch.empty(c["rows"], device="cuda")
        state["work"] = torch.empty(N.model_argmax_work_bytes(w), dtype=torch.uint8, device="cuda")
        state["row"] = torch.zeros(1, dtype=torch.int64, device="cuda")
    else:
        w.prepare(ACTS[c["act"]], c["tokens"])
        state["x"] = torch.randn(c["tokens"], c["cols"], generator=g, device="cuda")
        state["y"] = torch.empty(c["tokens"], c["rows"], device="cuda")
    torch.cuda.synchronize()
    return state


def run(state):
    c = state["case"]
    if c["kind"] == "load":
        w = N.Weight.from_gguf(state["type"], state["blocks"], c["rows"], c["cols"],
                               N.Q8_0 if c["fmt"] == "q8" else N.Q4S)
        out = w.download()
        w.free()
        return out
    if c["kind"] == "model":
        cur = torch.cuda.current_stream()
        state["stream"].wait_stream(cur)
        state["fwd"].forward_dev(state["tokens"].data_ptr(), c["tokens"], c["pos"])
        state["fwd"].logits_last_dev(c["tokens"], state["logits"].data_ptr())
        cur.wait_stream(state["stream"])
        return state["logits"]
    st = torch.cuda.current_stream().cuda_stream
    x, y = state["x"], state["y"]
    if c["kind"] == "head":
        N.model_argmax_dev(state["w"], x.data_ptr(), y.data_ptr(), state["work"].data_ptr(), state["row"].data_ptr(),
                           st)
        return y, state["row"]
    N.gemv_batch_dev(state["w"], x.data_ptr(), c["cols"], y.data_ptr(), c["rows"], c["tokens"], ACTS[c["act"]], st)
    return y


def _weight_bytes(fmt, n):
    return {"q8": n + n // 16, "q4": n // 2 + n // 8, "bf16": 2 * n}[fmt]


def work(case):
    c = case
    if c["kind"] == "load":
        n = c["rows"] * c["cols"]
        src = n // 256 * 144 if c["type"] == "q4_k" else 2 * n
        return {"bytes": src + _weight_bytes(c["fmt"], n), "flops": 0}
    if c["kind"] == "model":
        hd, t, ctx = c["head_dim"], c["tokens"], c["pos"] + c["tokens"]
        qd, kvd = c["heads"] * hd, c["kv_heads"] * hd
        per = c["embd"] * (2 * qd + 2 * kvd + 3 * c["ffn"])
        head = c["vocab"] * c["embd"]
        attn = 4 * qd * sum(c["pos"] + i + 1 for i in range(t))
        return {"bytes": _weight_bytes(c["fmt"], c["layers"] * per + head) + c["layers"] * 4 * kvd * ctx
                + 4 * c["vocab"], "flops": c["layers"] * (2 * per * t + attn) + 2 * head}
    t = c.get("tokens", 1)
    return {"bytes": _weight_bytes(c["fmt"], c["rows"] * c["cols"]) + 4 * t * (c["rows"] + c["cols"]),
            "flops": 2 * c["rows"] * c["cols"] * t}


def tolerance(case):
    # The f32 mode and the loader promise the reference's bits.
    if case["kind"] in ("head", "load") or case["act"] == "f32":
        return "exact"
    if case["kind"] == "matmul":
        # Exact block dots; what differs is the rounding of their sum (against
        # 64 bits: 2.5e-8 up to 16 vectors, up to 6e-8 beyond).
        return {"rel": 1.5e-7 if case["tokens"] <= 16 else 3e-7}
    # One int8 quant that rounds the other way shifts later quants in turn: the
    # logits then differ by the quantization's own noise (against 64 bits 2e-2
    # to 3e-2; 2.5e-8 where no quant moved).
    return {"rel": 0.1}


def exact(case, seed):
    c = case
    if c["kind"] == "load":
        return None
    if c["kind"] != "model":
        g = _gen(seed)
        parts = _parts(c["fmt"], c["rows"], c["cols"], g)
        if c["kind"] == "head":
            return _mm(c["fmt"], parts, torch.randn(c["cols"], generator=g, device="cuda")[None], "f32")[0], None
        x = torch.randn(c["tokens"], c["cols"], generator=g, device="cuda")
        return _mm(c["fmt"], parts, x, c["act"])
    layers, head, norms, biases, tokens = _model_parts(c, seed)
    e, f, hd, hq, hk = c["embd"], c["ffn"], c["head_dim"], c["heads"], c["kv_heads"]
    qd, kvd, n = hq * hd, hk * hd, len(tokens)
    cfg = _config(c)
    norms = torch.from_numpy(norms).cuda().double()
    tok = torch.from_numpy(tokens).cuda().long()

    def norm(v, gamma):
        return v / torch.sqrt((v * v).mean(1, keepdim=True) + cfg.rms_eps) * gamma

    # The rotation angles are the reference's, stepped in f32.
    inv, ratio, angles = np.float32(1), np.float32(cfg.rope_base) ** np.float32(-2 / hd), []
    for _ in range(hd // 2):
        angles.append(np.arange(n, dtype=np.float32) * inv)
        inv = np.float32(inv * ratio)
    th = torch.from_numpy(np.stack(angles, 1)).cuda().double()
    cos, sin = th.cos().unsqueeze(1), th.sin().unsqueeze(1)

    def rope(v):
        if cfg.rope_mode == models.ROPE_NORM:
            a, b = v[..., 0::2], v[..., 1::2]
            return torch.stack([a * cos - b * sin, a * sin + b * cos], 3).view(v.shape)
        a, b = v[..., :hd // 2], v[..., hd // 2:]
        return torch.cat([a * cos - b * sin, a * sin + b * cos], 2)

    x = _dense(c["fmt"], [p[tok] for p in head])
    mask = torch.full((n, n), -math.inf, dtype=torch.float64, device="cuda").triu_(1)
    for li, (wqkv, wo, wgu, wdown) in enumerate(layers):
        nr = norms[(4 * e + 2 * hd) * li:]
        qkv = _mm(c["fmt"], wqkv, norm(x, nr[:e]), c["act"])
        if biases is not None:
            b = biases[(qd + 2 * kvd) * li:(qd + 2 * kvd) * (li + 1)]
            qkv = qkv + torch.from_numpy(b).cuda().double()
        q = rope(qkv[:, :qd].view(n, hq, hd))
        k = rope(qkv[:, qd:qd + kvd].view(n, hk, hd)).float().bfloat16().double()  # the cache is BF16
        v = qkv[:, qd + kvd:].view(n, hk, hd).float().bfloat16().double()
        out = torch.empty(n, hq, hd, dtype=torch.float64, device="cuda")
        for h in range(hq):
            kh = h // (hq // hk)
            p = torch.softmax(q[:, h] @ k[:, kh].T.contiguous() * cfg.attn_scale + mask, 1)
            out[:, h] = p @ v[:, kh].contiguous()
        x = x + _mm(c["fmt"], wo, out.view(n, qd), c["act"])
        gu = _mm(c["fmt"], wgu, norm(x, nr[2 * e + 2 * hd:3 * e + 2 * hd]), c["act"])
        gate = gu[:, :f]
        x = x + _mm(c["fmt"], wdown, gate * torch.sigmoid(gate) * gu[:, f:], c["act"])
    x = norm(x[-1:], norms[-e:])
    return _mm(c["fmt"], head, x, c["act"])[0]
