"""The work that this framework is timed on: the blocks of a quantised Qwen3 decoder and whole calls of the model.

Every case goes through the operators and the model calls of rpgbarenginecuda_amd.ops, on synthetic weights and
inputs of the Qwen3-1.7B and Qwen3-4B shapes (Q4_K_M layout: Q6_K attn_v, ffn_down and embeddings, Q4_K elsewhere):

  mlp     gate / up + SwiGLU and ffn_down on n tokens; one token takes the form with the residual + norm inside
  proj    q / k / v on n tokens, and the output projection of n attention rows
  attn    q/k norm + RoPE + K/V store of n tokens at position pos0, and attention over the cache
  ops     embedding gather, residual + norm, q/k norm + RoPE + K/V store and SwiGLU (no matrix products)
  head    logits of n tokens over the vocabulary, and a token sampled from the last row
  model   a forward of n tokens behind pos0 cached ones through a few layers and the head
"""
from __future__ import annotations

import math
import os
import struct
import tempfile

import torch

from rpgbarenginecuda_amd import ops

Q4, Q6 = ops.GGML_Q4_K, ops.GGML_Q6_K
EPS = 1e-6
THETA = 1e6
HEAD = 128
VOCAB = 151936

# hidden, intermediate, query heads, kv heads: the two models, and a tensor-parallel shard of each.
SHAPES = {
    "1.7b": (2048, 6144, 16, 8),
    "4b": (2560, 9728, 32, 8),
    "1.7b/8": (2048, 768, 2, 1),
    "4b/2": (2560, 4864, 16, 4),
}


def listed():
    return [
        # One generated token through one layer's MLP: the smallest call, all latency.
        {"name": "mlp_decode_n1", "kind": "mlp", "shape": "1.7b", "n": 1},
        # A short prompt (a greeting, a game event).
        {"name": "mlp_prompt_n21", "kind": "mlp", "shape": "1.7b", "n": 21},
        # A user's turn in the larger model, an odd number of tokens.
        {"name": "mlp_turn_4b_n333", "kind": "mlp", "shape": "4b", "n": 333},
        # A long system prompt with its lore, as a game session begins.
        {"name": "mlp_prefill_n2811", "kind": "mlp", "shape": "1.7b", "n": 2811},
        # The attention projections of a medium prompt in the larger model.
        {"name": "proj_prompt_4b_n700", "kind": "proj", "shape": "4b", "n": 700},
        # One generated token's attention in the middle of a conversation.
        {"name": "attn_decode_pos2047", "kind": "attn", "shape": "1.7b", "n": 1, "pos0": 2047, "max_seq": 4096},
        # A follow-up turn: a few tokens that look back on a long history.
        {"name": "attn_turn_n45_pos1500", "kind": "attn", "shape": "1.7b", "n": 45, "pos0": 1500, "max_seq": 4096},
        # The long prompt's attention.
        {"name": "attn_prefill_n2811", "kind": "attn", "shape": "1.7b", "n": 2811, "pos0": 0, "max_seq": 4096},
        # The long prompt's memory-bound operators.
        {"name": "ops_prefill_n2811", "kind": "ops", "shape": "1.7b", "n": 2811, "max_seq": 4096, "embd": "q4"},
        # The end of each generated token: logits, then the engine's default sampling.
        {"name": "head_sample_n1", "kind": "head", "shape": "1.7b", "n": 1, "vocab": VOCAB, "temperature": 0.7,
         "top_k": 0, "top_p": 0.95},
        # A decode step through the model's own call (8 layers stand for all of them).
        {"name": "model_step_pos300", "kind": "model", "shape": "1.7b", "n": 1, "pos0": 300, "layers": 8,
         "vocab": VOCAB},
        # A short prompt through the model's own call.
        {"name": "model_prompt_n21", "kind": "model", "shape": "1.7b", "n": 21, "pos0": 0, "layers": 8,
         "vocab": VOCAB},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    kind = rng.choice(["mlp", "mlp", "proj", "attn", "attn", "ops", "head", "model"])
    shape = rng.choice(["1.7b", "1.7b", "4b", "1.7b/8", "4b/2"])
    if kind == "mlp":
        return {"kind": kind, "shape": shape, "n": _log_int(rng, 1, 1400 if shape == "4b" else 2811)}
    if kind == "proj":
        return {"kind": kind, "shape": shape, "n": _log_int(rng, 1, 2811)}
    if kind == "attn":
        n = rng.choice([1, _log_int(rng, 2, 2811)])
        return {"kind": kind, "shape": shape, "n": n, "pos0": rng.randint(0, 4096 - n), "max_seq": 4096}
    if kind == "ops":
        return {"kind": kind, "shape": shape, "n": _log_int(rng, 1, 2811), "max_seq": 4096,
                "embd": rng.choice(["q4", "q6"])}
    if kind == "head":
        t, k, p = rng.choice([(0.7, 0, 0.95), (0.7, 40, 0.9), (1.0, 0, 1.0), (0.0, 0, 1.0)])
        return {"kind": kind, "shape": shape.split("/")[0], "n": _log_int(rng, 1, 24), "vocab": VOCAB,
                "temperature": t, "top_k": k, "top_p": p}
    return {"kind": kind, "shape": shape.split("/")[0], "n": rng.choice([1, _log_int(rng, 2, 200)]),
            "pos0": rng.randint(0, 1500), "layers": rng.choice([2, 3, 4]), "vocab": rng.choice([8191, 32000])}


# ----------------------------------------------------------------------------- inputs


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _normal(g, *shape, mean=0.0, std=1.0):
    return torch.randn(*shape, generator=g, device="cuda") * std + mean


def _norm_weight(g, n):
    return _normal(g, n, mean=1.0, std=0.1)


def _f16_bytes(x):
    return x.to(torch.float16).view(torch.uint8).reshape(x.numel(), 2)


def _table(g, ggml_type, rows, cols, std):
    """Raw blocks of a [rows, cols] matrix of zero mean and about that deviation: quants uniform, scales over the
    type's range (Q6_K: the whole int8 range with one -128 a block, as quantisers write it)."""
    nb = rows * cols // 256
    b = torch.randint(0, 256, (nb, ops.BLOCK_BYTES[ggml_type]), dtype=torch.uint8, device="cuda", generator=g)
    spread = 0.5 + torch.rand(nb, device="cuda", generator=g)
    if ggml_type == Q4:
        # d (sc q - 8 m) with m about 7.5 sc / 8 centres q = 0..15 on zero
        sc = torch.randint(8, 64, (nb, 8), device="cuda", generator=g)
        m = torch.round(7.5 * sc / 8).to(torch.int64)
        d = spread * (std / 175.0)
        b[:, 0:2] = _f16_bytes(d)
        b[:, 2:4] = _f16_bytes(d * 8)
        b[:, 4:8] = (sc[:, 0:4] | ((sc[:, 4:8] >> 4) << 6)).to(torch.uint8)
        b[:, 8:12] = (m[:, 0:4] | ((m[:, 4:8] >> 4) << 6)).to(torch.uint8)
        b[:, 12:16] = ((sc[:, 4:8] & 15) | ((m[:, 4:8] & 15) << 4)).to(torch.uint8)
    else:
        sc = torch.randint(-128, 128, (nb, 16), device="cuda", generator=g)
        sc.scatter_(1, torch.randint(0, 16, (nb, 1), device="cuda", generator=g), -128)
        b[:, 192:208] = sc.to(torch.int8).view(torch.uint8)
        b[:, 208:210] = _f16_bytes(spread * (std / 1500.0))
    return b.reshape(-1)


def _matrix(g, ggml_type, rows, cols, std=0.03):
    return ops.GpuTensor(_table(g, ggml_type, rows, cols, std), ggml_type, rows, cols)


def _rope(n_pos):
    i = torch.arange(HEAD // 2, dtype=torch.float64, device="cuda")
    a = torch.arange(n_pos, dtype=torch.float64, device="cuda")[:, None] * THETA ** (-2.0 * i / HEAD)[None, :]
    return torch.cat([a.cos(), a.sin()], 1).float()


def _cache(g, kvh, max_seq, pos0):
    """A layer's K and V with pos0 tokens in them."""
    k = torch.zeros(kvh, max_seq, HEAD, dtype=torch.float16, device="cuda")
    v = torch.zeros_like(k)
    if pos0:
        k[:, :pos0] = _normal(g, kvh, pos0, HEAD).half()
        v[:, :pos0] = _normal(g, kvh, pos0, HEAD).half()
    return k, v


def _empty(*shape):
    return torch.empty(*shape, device="cuda")


def _write_gguf(path, case, g):
    """A model file of the case's shape; returns {tensor name: (type, dims, bytes on the GPU)}."""
    hidden, inter, heads, kvh = SHAPES[case["shape"]]
    specs = [("token_embd.weight", Q6, (hidden, case["vocab"])), ("output_norm.weight", 0, (hidden,))]
    for i in range(case["layers"]):
        p = "blk.%d." % i
        specs += [(p + "attn_norm.weight", 0, (hidden,)), (p + "ffn_norm.weight", 0, (hidden,)),
                  (p + "attn_q_norm.weight", 0, (HEAD,)), (p + "attn_k_norm.weight", 0, (HEAD,)),
                  (p + "attn_q.weight", Q4, (hidden, heads * HEAD)), (p + "attn_k.weight", Q4, (hidden, kvh * HEAD)),
                  (p + "attn_v.weight", Q6, (hidden, kvh * HEAD)),
                  (p + "attn_output.weight", Q4, (heads * HEAD, hidden)),
                  (p + "ffn_gate.weight", Q4, (hidden, inter)), (p + "ffn_up.weight", Q4, (hidden, inter)),
                  (p + "ffn_down.weight", Q6, (inter, hidden))]
    tensors = {}
    for name, t, dims in specs:
        if len(dims) == 1:
            data = _norm_weight(g, dims[0]).view(torch.uint8)
        else:
            data = _table(g, t, dims[1], dims[0], 0.5 / math.sqrt(dims[0]) if name != "token_embd.weight" else 0.04)
        tensors[name] = (t, dims, data)

    def text(s):
        return struct.pack("<Q", len(s)) + s.encode()

    u32, f32, st = 4, 6, 8
    meta = [("general.architecture", st, "qwen3"), ("general.name", st, "synthetic"),
            ("qwen3.block_count", u32, case["layers"]), ("qwen3.embedding_length", u32, hidden),
            ("qwen3.attention.head_count", u32, heads), ("qwen3.attention.head_count_kv", u32, kvh),
            ("qwen3.attention.key_length", u32, HEAD), ("qwen3.attention.value_length", u32, HEAD),
            ("qwen3.feed_forward_length", u32, inter), ("qwen3.context_length", u32, 40960),
            ("qwen3.rope.freq_base", f32, THETA), ("qwen3.attention.layer_norm_rms_epsilon", f32, EPS)]
    head = b"GGUF" + struct.pack("<IQQ", 3, len(specs), len(meta))
    for key, kind, value in meta:
        head += text(key) + struct.pack("<I", kind)
        head += text(value) if kind == st else struct.pack("<I" if kind == u32 else "<f", value)
    at = 0
    for name, t, dims in specs:
        head += text(name) + struct.pack("<I", len(dims)) + struct.pack("<%dQ" % len(dims), *dims)
        head += struct.pack("<IQ", t, at)
        at += -(-tensors[name][2].numel() // 32) * 32
    with open(path, "wb") as f:
        f.write(head + b"\0" * (-len(head) % 32))
        for name, _, _ in specs:
            data = tensors[name][2].cpu().numpy()
            f.write(data.data)
            f.write(b"\0" * (-data.size % 32))
    return tensors


def _model_inputs(case, seed):
    """(tokens, cached K and V of every layer [layers, kv heads, positions, head]) of a model case."""
    kvh = SHAPES[case["shape"]][3]
    g = _gen(seed * 7 + 5)
    toks = torch.randint(0, case["vocab"], (case["n"],), generator=g, device="cuda", dtype=torch.int32)
    kv = [_cache(g, kvh, 2048, case["pos0"]) for _ in range(case["layers"])]
    return toks, kv


def prepare(case, seed):
    kind, n = case["kind"], case["n"]
    hidden, inter, heads, kvh = SHAPES[case["shape"]]
    ops.init()
    g = _gen(seed)
    s = dict(case)
    if kind == "mlp":
        s.update(gate=_matrix(g, Q4, inter, hidden), up=_matrix(g, Q4, inter, hidden),
                 down=_matrix(g, Q6, hidden, inter), x=_normal(g, n, hidden), og=_empty(n, inter), ou=_empty(n, inter),
                 out=_empty(n, hidden))
        if n == 1:  # the residual stream, the block's delta, the norm's weights
            s.update(d=_normal(g, n, hidden, std=0.5), nw=_norm_weight(g, hidden), x2=_empty(n, hidden))
    elif kind == "proj":
        s.update(q=_matrix(g, Q4, heads * HEAD, hidden), k=_matrix(g, Q4, kvh * HEAD, hidden),
                 v=_matrix(g, Q6, kvh * HEAD, hidden), o=_matrix(g, Q4, hidden, heads * HEAD),
                 x=_normal(g, n, hidden), a=_normal(g, n, heads * HEAD, std=0.3), oq=_empty(n, heads * HEAD),
                 ok=_empty(n, kvh * HEAD), ov=_empty(n, kvh * HEAD), out=_empty(n, hidden))
    elif kind in ("attn", "ops"):
        pos0 = case.get("pos0", 0)
        kc, vc = _cache(g, kvh, case["max_seq"], pos0)
        s.update(pos0=pos0, kc=kc, vc=vc, q=_normal(g, n, heads * HEAD), k=_normal(g, n, kvh * HEAD),
                 v=_normal(g, n, kvh * HEAD), qn=_norm_weight(g, HEAD), kn=_norm_weight(g, HEAD),
                 rope=_rope(case["max_seq"]))
        if kind == "attn":
            s.update(out=_empty(n, heads * HEAD))
        else:
            s.update(embd=_matrix(g, Q4 if case["embd"] == "q4" else Q6, VOCAB, hidden, std=1.0),
                     toks=torch.randint(0, VOCAB, (n,), generator=g, device="cuda", dtype=torch.int32),
                     x=_empty(n, hidden), d=_normal(g, n, hidden), nw=_norm_weight(g, hidden), h=_empty(n, hidden),
                     gate=_normal(g, n, inter, std=2.0), up=_normal(g, n, inter))
    elif kind == "head":
        ops.GpuSamplerWarmup()
        s.update(w=_matrix(g, Q6, case["vocab"], hidden, std=0.06), x=_normal(g, n, hidden),
                 logits=_empty(n, case["vocab"]), probs=torch.zeros(case["vocab"], device="cuda"),
                 token=torch.zeros(1, dtype=torch.int32, device="cuda"),
                 opt=ops.SampleOptions(case["temperature"], case["top_k"], case["top_p"]))
    else:
        with tempfile.TemporaryDirectory() as folder:
            path = os.path.join(folder, "model.gguf")
            _write_gguf(path, case, g)
            m = ops.GpuModel(path, 2048)
        toks, layers = _model_inputs(case, seed)
        kv = ops.GpuKvCache(m, 2048)
        for i, (k, v) in enumerate(layers):
            for src, dst in zip((k, v), kv.layer(i)):
                ops.GpuStreamCopy(src, dst, src.numel() * 2)
        torch.cuda.synchronize()
        s.update(m=m, kv=kv, scratch=ops.GpuScratch(), toks=toks, ids=toks.cpu().numpy(),
                 logits=_empty(case["vocab"]))
    return s


# ----------------------------------------------------------------------------- one pass


def run(s):
    kind, n = s["kind"], s["n"]
    hidden, inter, heads, kvh = SHAPES[s["shape"]]
    if kind == "mlp":
        if n == 1:
            if not ops.GpuNormMatMulQuantSwiGLU(s["x"], s["d"], s["nw"], EPS, s["x2"], s["gate"], s["up"], s["og"],
                                                s["ou"]):
                raise RuntimeError("no one-token form of this MLP")
            ops.GpuMatMulQuant(s["down"], s["og"], n, s["out"])
            return {"x": s["x2"], "act": s["og"], "out": s["out"]}
        ops.GpuMatMulQuantSwiGLU(s["gate"], s["up"], s["x"], n, s["og"], s["ou"])
        ops.GpuMatMulQuant(s["down"], s["og"], n, s["out"])
        return {"act": s["og"], "out": s["out"]}
    if kind == "proj":
        ops.GpuMatMulQuantGroup([s["q"], s["k"], s["v"]], s["x"], n, [s["oq"], s["ok"], s["ov"]])
        ops.GpuMatMulQuant(s["o"], s["a"], n, s["out"])
        return {"q": s["oq"], "k": s["ok"], "v": s["ov"], "out": s["out"]}
    if kind == "attn":
        if n > 1 or not ops.GpuQkNormRopeKvAttention(heads, kvh, HEAD, s["pos0"], s["q"], s["k"], s["v"], s["qn"],
                                                     s["kn"], s["rope"], s["max_seq"], EPS, s["kc"], s["vc"],
                                                     s["max_seq"], s["out"]):
            ops.GpuQkNormRopeKv(s["q"], s["k"], s["v"], s["qn"], s["kn"], heads, kvh, HEAD, s["rope"], s["max_seq"],
                                s["pos0"], n, EPS, s["kc"], s["vc"], s["max_seq"])
            ops.GpuAttentionFromCache(heads, kvh, HEAD, s["pos0"], s["q"], n, s["kc"], s["vc"], s["max_seq"],
                                      s["out"])
        return {"out": s["out"], "k": s["kc"], "v": s["vc"]}
    if kind == "ops":
        ops.GpuEmbeddingLookup(s["embd"], s["toks"], n, s["x"])
        ops.GpuAddRmsNorm(s["x"], s["d"], s["nw"], n, hidden, EPS, s["h"])
        ops.GpuQkNormRopeKv(s["q"], s["k"], s["v"], s["qn"], s["kn"], heads, kvh, HEAD, s["rope"], s["max_seq"],
                            s["pos0"], n, EPS, s["kc"], s["vc"], s["max_seq"])
        ops.GpuSiluMulInPlace(s["gate"], s["up"], n * inter)
        return {"x": s["x"], "h": s["h"], "q": s["q"], "k": s["kc"], "v": s["vc"], "act": s["gate"]}
    if kind == "head":
        ops.GpuMatMulQuant(s["w"], s["x"], n, s["logits"])
        last = s["logits"][n - 1]
        if s["temperature"] == 0.0:
            ops.GpuArgMax(last, s["vocab"], s["token"])
            return {"logits": s["logits"], "token": s["token"]}
        ops.GpuSampleToken(last, s["vocab"], s["opt"], 2026, n, s["probs"], s["token"])
        return {"logits": s["logits"], "probs": s["probs"], "token": s["token"]}
    s["kv"].set_len(s["pos0"])  # the turn is taken again from the same history
    if n == 1:
        ops.GpuForwardStepDev(s["m"], s["toks"], s["pos0"], s["kv"], s["scratch"])
    else:
        ops.GpuForwardFull(s["m"], s["ids"], s["scratch"], want_logits=False, kv=s["kv"])
    row = 4 * s["vocab"]
    ops.GpuStreamCopy(s["scratch"].logits_dev() + (n - 1) * row, s["logits"], row)
    return {"logits": s["logits"]}


# ----------------------------------------------------------------------------- cost and tolerance


def _table_bytes(ggml_type, rows, cols):
    return rows * (cols // 256) * ops.BLOCK_BYTES[ggml_type]


def _mlp_work(n, hidden, inter):
    b = 2 * _table_bytes(Q4, inter, hidden) + _table_bytes(Q6, hidden, inter) + 4 * n * (2 * hidden + inter)
    return b, 2 * n * 3 * hidden * inter


def _proj_work(n, hidden, heads, kvh):
    b = _table_bytes(Q4, heads * HEAD, hidden) * 2 + _table_bytes(Q4, kvh * HEAD, hidden)
    b += _table_bytes(Q6, kvh * HEAD, hidden) + 4 * n * HEAD * (2 * heads + 2 * kvh) + 8 * n * hidden
    return b, 2 * n * hidden * HEAD * (2 * heads + 2 * kvh)


def _attn_work(n, pos0, heads, kvh):
    pairs = n * pos0 + n * (n + 1) // 2
    b = n * HEAD * (8 * heads + 12 * kvh + 4) + 4 * pos0 * kvh * HEAD
    return b, 4 * pairs * heads * HEAD


def work(case):
    kind, n = case["kind"], case["n"]
    hidden, inter, heads, kvh = SHAPES[case["shape"]]
    if kind == "mlp":
        b, f = _mlp_work(n, hidden, inter)
    elif kind == "proj":
        b, f = _proj_work(n, hidden, heads, kvh)
    elif kind == "attn":
        b, f = _attn_work(n, case["pos0"], heads, kvh)
    elif kind == "ops":
        b = n * (hidden // 256) * ops.BLOCK_BYTES[Q4 if case["embd"] == "q4" else Q6] + 12 * n * hidden
        b, f = b + n * HEAD * (8 * heads + 12 * kvh + 4) + 12 * n * inter, n * (6 * hidden + 20 * inter)
    elif kind == "head":
        b = _table_bytes(Q6, case["vocab"], hidden) + 4 * n * (hidden + case["vocab"]) + 8 * case["vocab"]
        f = 2 * n * hidden * case["vocab"]
    else:
        parts = [_mlp_work(n, hidden, inter), _proj_work(n, hidden, heads, kvh), _attn_work(n, case["pos0"], heads, kvh)]
        b = case["layers"] * sum(p[0] for p in parts) + _table_bytes(Q6, case["vocab"], hidden)
        b += 4 * n * case["vocab"]
        f = case["layers"] * sum(p[1] for p in parts) + 2 * n * hidden * case["vocab"]
    return {"bytes": float(b), "flops": float(f)}


def tolerance(case):
    """About four times what the outputs were seen to be off their 64-bit values: matrix products 5e-7, cache rows
    4.6e-6 (a value next to a rounding boundary of fp16 may fall to either side, 1e-3 of it), a model's logits 5e-5
    (those roundings, through the layers that follow)."""
    return {"mlp": {"rel": 3e-6}, "proj": {"rel": 3e-6}, "attn": {"rel": 2e-5, "max": 2e-3},
            "ops": {"rel": 2e-5, "max": 2e-3}, "head": {"rel": 3e-6}, "model": {"rel": 3e-4}}[case["kind"]]


# ----------------------------------------------------------------------------- in 64 bits


def _f16(b):
    return b.contiguous().view(torch.float16).double().reshape(-1)


def _dequant(raw, ggml_type, rows, cols):
    b = raw.reshape(-1, ops.BLOCK_BYTES[ggml_type])
    nb = b.shape[0]
    if ggml_type == Q4:
        d, dmin = _f16(b[:, 0:2]), _f16(b[:, 2:4])
        p = b[:, 4:16].to(torch.int32)
        sc = torch.cat([p[:, 0:4] & 63, (p[:, 8:12] & 15) | ((p[:, 0:4] >> 6) << 4)], 1)
        m = torch.cat([p[:, 4:8] & 63, (p[:, 8:12] >> 4) | ((p[:, 4:8] >> 6) << 4)], 1)
        qs = b[:, 16:144].reshape(nb, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).reshape(nb, 8, 32)
        w = (d[:, None] * sc)[:, :, None] * q.double() - (dmin[:, None] * m)[:, :, None]
    else:
        d = _f16(b[:, 208:210])
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        ql = b[:, 0:128].to(torch.int32).reshape(nb, 2, 2, 32)
        qh = b[:, 128:192].to(torch.int32).reshape(nb, 2, 32)
        q = torch.stack([(ql[:, :, 0] & 15) | ((qh & 3) << 4), (ql[:, :, 1] & 15) | (((qh >> 2) & 3) << 4),
                         (ql[:, :, 0] >> 4) | (((qh >> 4) & 3) << 4), (ql[:, :, 1] >> 4) | (((qh >> 6) & 3) << 4)], 2)
        w = (d[:, None] * sc)[:, :, None] * (q.reshape(nb, 16, 16).double() - 32.0)
    return w.reshape(rows, cols)


def _product(x, t):
    """x . W^T, a slice of W's rows at a time."""
    raw = t.buf.reshape(t.rows, -1)
    return torch.cat([x @ _dequant(raw[r:r + 16384].reshape(-1), t.type, min(16384, t.rows - r), t.cols).t()
                      for r in range(0, t.rows, 16384)], 1)


def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _silu_mul(g, u):
    return g * torch.sigmoid(g) * u


def _norm_rope(x, n_heads, w, rope):
    """The head norm and the rotation of rows [n, heads * 128] with the table's rows [n, 128]."""
    x = _rms(x.double().reshape(x.shape[0], n_heads, HEAD), w)
    c, sn = rope[:, None, :HEAD // 2].double(), rope[:, None, HEAD // 2:].double()
    a, b = x[..., :HEAD // 2], x[..., HEAD // 2:]
    return torch.cat([a * c - b * sn, b * c + a * sn], -1)


def _attention(q, kc, vc, pos0):
    """q [n, heads, 128] over the caches [kv heads, positions, 128] (fp16 values), causal from pos0."""
    n, heads = q.shape[0], q.shape[1]
    total, group = pos0 + n, heads // kc.shape[0]
    mask = torch.arange(total, device="cuda")[None, :] > pos0 + torch.arange(n, device="cuda")[:, None]
    out = torch.empty(n, heads, HEAD, dtype=torch.float64, device="cuda")
    for h in range(heads):
        k, v = kc[h // group, :total].double(), vc[h // group, :total].double()
        p = (q[:, h] @ k.t()) / math.sqrt(HEAD)
        out[:, h] = torch.softmax(p.masked_fill(mask, -math.inf), -1) @ v
    return out.reshape(n, heads * HEAD)


def _attend(q, k, v, qn, kn, rope, kc, vc, pos0):
    """(attention output, K cache, V cache, rotated q) of raw projections, the cache's rows stored in fp16."""
    n, kvh = q.shape[0], kc.shape[0]
    rows = rope[pos0:pos0 + n]
    kc, vc = kc.clone(), vc.clone()
    kc[:, pos0:pos0 + n] = _norm_rope(k, kvh, kn, rows).transpose(0, 1).half()
    vc[:, pos0:pos0 + n] = v.reshape(n, kvh, HEAD).transpose(0, 1).half()
    qr = _norm_rope(q, q.shape[1] // HEAD, qn, rows)
    return qr, kc, vc


def _filtered(logits, temperature, top_k, top_p):
    """The sampler's distribution over one row."""
    v = logits / temperature
    if 0 < top_k < v.numel():
        v = v.masked_fill(v < torch.topk(v, top_k).values[-1], -math.inf)
    p = torch.softmax(v, 0)
    if top_p < 1.0:
        order = torch.argsort(p)
        drop = torch.cumsum(p[order], 0) <= 1.0 - top_p
        drop[-1] = False
        p[order[drop]] = 0.0
        p = p / p.sum()
    return p


def _exact_model(case, seed):
    hidden, inter, heads, kvh = SHAPES[case["shape"]]
    with tempfile.TemporaryDirectory() as folder:
        tensors = _write_gguf(os.path.join(folder, "model.gguf"), case, _gen(seed))
    toks, kv = _model_inputs(case, seed)

    def mat(name):
        t, dims, raw = tensors[name]
        return ops.GpuTensor(raw, t, dims[1], dims[0])

    def vec(name):
        return tensors[name][2].view(torch.float32)

    embd, rope, pos0 = mat("token_embd.weight"), _rope(2048), case["pos0"]
    raw = embd.buf.reshape(embd.rows, -1)[toks.long()]
    x = _dequant(raw.reshape(-1), embd.type, case["n"], hidden)
    for i in range(case["layers"]):
        p = "blk.%d." % i
        h = _rms(x, vec(p + "attn_norm.weight"))
        q, k, v = (_product(h, mat(p + "attn_%s.weight" % c)) for c in "qkv")
        qr, kc, vc = _attend(q, k, v, vec(p + "attn_q_norm.weight"), vec(p + "attn_k_norm.weight"), rope, *kv[i], pos0)
        x = x + _product(_attention(qr, kc, vc, pos0), mat(p + "attn_output.weight"))
        h = _rms(x, vec(p + "ffn_norm.weight"))
        act = _silu_mul(_product(h, mat(p + "ffn_gate.weight")), _product(h, mat(p + "ffn_up.weight")))
        x = x + _product(act, mat(p + "ffn_down.weight"))
    return {"logits": _product(_rms(x[-1:], vec("output_norm.weight")), embd)[0]}


def exact(case, seed):
    kind, n = case["kind"], case["n"]
    if kind == "model":
        return _exact_model(case, seed)
    s = prepare(case, seed)
    hidden, inter, heads, kvh = SHAPES[case["shape"]]
    if kind == "mlp":
        x, out = s["x"].double(), {}
        if n == 1:
            x = x + s["d"].double()
            out["x"] = x
            x = _rms(x, s["nw"])
        out["act"] = _silu_mul(_product(x, s["gate"]), _product(x, s["up"]))
        out["out"] = _product(out["act"], s["down"])
        return out
    if kind == "proj":
        x = s["x"].double()
        return {"q": _product(x, s["q"]), "k": _product(x, s["k"]), "v": _product(x, s["v"]),
                "out": _product(s["a"].double(), s["o"])}
    if kind in ("attn", "ops"):
        qr, kc, vc = _attend(s["q"], s["k"], s["v"], s["qn"], s["kn"], s["rope"], s["kc"], s["vc"], s["pos0"])
        if kind == "attn":
            return {"out": _attention(qr, kc, vc, s["pos0"]), "k": kc.double(), "v": vc.double()}
        raw = s["embd"].buf.reshape(VOCAB, -1)[s["toks"].long()]
        x = _dequant(raw.reshape(-1), s["embd"].type, n, hidden) + s["d"].double()
        return {"x": x, "h": _rms(x, s["nw"]), "q": qr.reshape(n, heads * HEAD), "k": kc.double(), "v": vc.double(),
                "act": _silu_mul(s["gate"].double(), s["up"].double())}
    logits = _product(s["x"].double(), s["w"])
    if case["temperature"] == 0.0:
        return {"logits": logits, "token": None}
    probs = _filtered(logits[n - 1], case["temperature"], case["top_k"], case["top_p"])
    return {"logits": logits, "probs": probs, "token": None}
