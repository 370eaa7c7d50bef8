"""Short turns over a long cache (the matrix-core kernel for 2 to 63 tokens): its
tiles' and blocks' edges against the float64 oracle, within the bound of
tests/test_gpu_attention.py; an infinite value reaches only the tokens that see it;
a capture laid out for a larger budget; values outside the tile's keys don't matter."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_attention import check, dev, host, make

pytestmark = pytest.mark.gpu

CASES = [
    # (n_heads, n_kv_heads, max_seq, pos0, seq)
    (16, 8, 4096, 1500, 45),
    (16, 8, 4096, 1504, 64 - 1),   # the first token's keys end in the middle of a block
    (32, 8, 2048, 1503, 32),       # a full tile
    (32, 8, 2048, 2048 - 33, 33),  # one token in the second tile, full cache
    (32, 8, 4200, 4096, 22),       # a last block of one key for some tokens
    (8, 8, 8192, 6001, 63),        # MHA
]


def takes_it(gpu, call):
    gpu.profile_start(4)
    call()
    gpu.profile_stop()
    return set(gpu.profile_report()) == {"AttnTurnKernel"}


# (n_heads, n_kv_heads, pos0, seq, whether the matrix-core kernel was measured to be the faster one)
ROUTES = [
    (8, 8, 3000, 32, False), (8, 8, 4000, 32, False), (16, 16, 2200, 16, False), (32, 32, 4000, 8, False),
    (8, 8, 4000, 33, False), (16, 8, 3000, 32, False), (16, 8, 1500, 21, False),
    (16, 8, 1500, 45, True), (32, 8, 1500, 21, True), (16, 4, 1500, 45, True), (8, 8, 1500, 40, True),
    (16, 16, 3000, 31, True), (64, 16, 1500, 12, True),
]


@pytest.mark.parametrize("nh,nkv,pos0,seq,turn", ROUTES)
def test_turn_route_is_the_faster_kernel(gpu, nh, nkv, pos0, seq, turn):
    import torch

    q = torch.zeros((seq, nh, 128), device="cuda")
    kv = torch.zeros(nkv * 4200 * 128, dtype=torch.int16, device="cuda")
    assert takes_it(gpu, lambda: gpu.GpuAttentionFromCache(nh, nkv, 128, pos0, q, seq, kv, kv, 4200, torch.empty_like(q))) == turn


@pytest.mark.parametrize("nh,nkv,max_seq,pos0,seq", CASES)
def test_turn_vs_f64(gpu, ora, nh, nkv, max_seq, pos0, seq):
    import torch

    rng = np.random.default_rng(pos0 + seq + nh)
    q, kc, vc = make(rng, nh, nkv, max_seq, seq, qscale=0.5)
    q[seq // 2] *= 1e-42 if seq % 2 else 1e-3  # a subnormal row: every key counts alike
    kc = kc.copy().reshape(nkv, max_seq, 128)
    vc = vc.copy().reshape(nkv, max_seq, 128)
    ref, smag, vmax = ora.attention_f64(q, kc.reshape(-1), vc.reshape(-1), max_seq, nh, nkv, 128, pos0, seq)
    kc[:, pos0 + seq:] = np.float16(np.inf).view(np.uint16)
    vc[:, pos0 + seq:] = np.float16(np.nan).view(np.uint16)
    out = torch.full((seq + 1, nh, 128), np.nan, dtype=torch.float32, device="cuda")
    args = (nh, nkv, 128, pos0, dev(q), seq, dev(kc.reshape(-1)), dev(vc.reshape(-1)), max_seq)
    assert takes_it(gpu, lambda: gpu.GpuAttentionFromCache(*args, out))
    check(host(out)[:seq], ref, smag, vmax, pos0)
    assert torch.isnan(out[seq]).all(), "wrote past the last token"


def test_turn_infinite_value(gpu, ora):
    """Token 20's value row holds an infinity: tokens 0 to 19 keep their results bit for
    bit, and from token 20 on that element is the infinity and the others are as before."""
    import torch

    nh, nkv, max_seq, pos0, seq = 16, 8, 2048, 1500, 45
    rng = np.random.default_rng(7)
    q, kc, vc = make(rng, nh, nkv, max_seq, seq)
    outs = []
    for bad in (False, True):
        v = vc.copy().reshape(nkv, max_seq, 128)
        v[:, pos0 + 20, 77] = np.float16(-np.inf if bad else 0.0).view(np.uint16)
        out = torch.empty((seq, nh, 128), dtype=torch.float32, device="cuda")
        gpu.GpuAttentionFromCache(nh, nkv, 128, pos0, dev(q), seq, dev(kc), dev(v.reshape(-1)), max_seq, out)
        outs.append(host(out))
    plain, got = outs
    assert np.array_equal(plain[:20], got[:20])
    assert np.all(got[20:, :, 77] == -np.inf)
    assert np.array_equal(np.delete(plain, 77, axis=2), np.delete(got, 77, axis=2))


def test_turn_captured(gpu, ora):
    """Captured for a budget of 4096 positions and replayed at others, with eager work
    and synchronisations in between."""
    import torch

    nh, nkv, max_seq, seq = 16, 8, 4096, 45
    rng = np.random.default_rng(11)
    q, kc, vc = make(rng, nh, nkv, max_seq, seq, qscale=0.5)
    qd, kd, vd = dev(q), dev(kc), dev(vc)
    out = torch.empty((seq, nh, 128), dtype=torch.float32, device="cuda")
    gpu.init()
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        with gpu.ScopedEngineStream(stream):
            graph.capture_begin()
            gpu.GpuAttentionFromCache(nh, nkv, 128, 0, qd, seq, kd, vd, max_seq, out, max_seq)
            graph.capture_end()
    torch.cuda.synchronize()
    for pos in (0, 31, 1500, 4096 - seq, 1200):
        gpu.stage_pos0(pos)
        torch.cuda.synchronize()
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        ref, smag, vmax = ora.attention_f64(q, kc, vc, max_seq, nh, nkv, 128, pos, seq)
        check(host(out), ref, smag, vmax, pos)


@pytest.mark.parametrize("seq", [64, 130])
def test_prefill_unaligned_values(gpu, seq):
    """The prefill kernel with the value rows at an address that is only a multiple of 4
    bytes gives the bits of the aligned call."""
    import torch

    nh, nkv, max_seq, pos0 = 4, 2, 512, 77
    rng = np.random.default_rng(seq)
    q, kc, vc = make(rng, nh, nkv, max_seq, seq)
    moved = torch.zeros(vc.size + 8, dtype=torch.int16, device="cuda")
    moved[2:2 + vc.size] = dev(vc.reshape(-1).view(np.int16))
    outs = [torch.empty((seq, nh, 128), device="cuda") for _ in range(2)]
    for v, out in ((dev(vc), outs[0]), (moved[2:2 + vc.size], outs[1])):
        gpu.GpuAttentionFromCache(nh, nkv, 128, pos0, dev(q), seq, dev(kc), v, max_seq, out)
    assert torch.equal(*outs)


@pytest.mark.parametrize("max_seq,seq", [(2048, 45), (2048, 64), (700, 200), (4001, 300)])
def test_staged_past_the_cache(gpu, ora, max_seq, seq):
    """A turn or a prefill: a replay whose staged position puts tokens past the cache's end: they see the whole
    cache, and nothing behind it is read (as the decode kernel does)."""
    import torch

    nh, nkv = 16, 8
    rng = np.random.default_rng(max_seq + seq)
    q, kc, vc = make(rng, nh, nkv, max_seq, seq, qscale=0.5)
    qd, kd, vd = dev(q), dev(kc), dev(vc)
    out = torch.empty((seq, nh, 128), dtype=torch.float32, device="cuda")
    gpu.init()
    gpu.GpuAttentionFromCache(nh, nkv, 128, 0, qd, seq, kd, vd, max_seq, out, max_seq)  # the library's buffers
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        with gpu.ScopedEngineStream(stream):
            graph.capture_begin()
            gpu.GpuAttentionFromCache(nh, nkv, 128, 0, qd, seq, kd, vd, max_seq, out, max_seq)
            graph.capture_end()
    torch.cuda.synchronize()
    for pos in (max_seq - 20, max_seq + 7):
        gpu.stage_pos0(pos)
        torch.cuda.synchronize()
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        got = host(out)
        for t in (0, 19, 20, 33, seq - 1):
            at = min(pos + t, max_seq - 1)
            ref, smag, vmax = ora.attention_f64(q[t:t + 1], kc, vc, max_seq, nh, nkv, 128, at, 1)
            check(got[t:t + 1], ref, smag, vmax, at)


def test_turn_refuses_what_the_decode_kernel_refuses(gpu):
    """A cache of more rows than the decode kernel's 32-bit indexing reaches is refused on the
    host for a turn too (nothing is launched, so the buffers may be small)."""
    import torch

    nh, nkv, seq = 16, 4, 45
    q = torch.zeros((seq, nh, 128), device="cuda")
    kv = torch.zeros(4096, dtype=torch.int16, device="cuda")
    with pytest.raises(gpu.RpgError, match="32-bit"):
        gpu.GpuAttentionFromCache(nh, nkv, 128, 3000, q, seq, kv.data_ptr(), kv.data_ptr(), (2 ** 31 - 1) // 256 + 1, torch.empty_like(q))


def reference(q, kc, vc, max_seq, nkv, pos0):
    """Causal attention in float64 with its infinities: [seq, heads, 128]."""
    seq, nh = q.shape[:2]
    k = kc.reshape(nkv, max_seq, 128).view(np.float16).astype(np.float64)
    v = vc.reshape(nkv, max_seq, 128).view(np.float16).astype(np.float64)
    out = np.empty((seq, nh, 128))
    with np.errstate(invalid="ignore"):
        for t in range(seq):
            n = pos0 + t + 1
            for h in range(nh):
                j = h // (nh // nkv)
                s = (k[j, :n] * q[t, h].astype(np.float64)).sum(1) / np.sqrt(128)
                p = np.exp(s - s.max())
                out[t, h] = (p[:, None] * v[j, :n]).sum(0) / p.sum()
    return out


@pytest.mark.parametrize("key", [0, 100, 1499, 1500, 1503])
def test_turn_infinities_in_the_history(gpu, key):
    """An infinite value of a token that the whole tile sees is that infinity in its dim (and
    other dims and kv heads keep their bits); an infinite key leaves its token out where the
    score is -inf and gives NaN where it is +inf. As the decode kernel does."""
    import torch

    nh, nkv, max_seq, pos0, seq = 16, 8, 2048, 1500, 45
    rng = np.random.default_rng(key)
    q, kc, vc = make(rng, nh, nkv, max_seq, seq, qscale=0.5)
    q[:, :, 5] = np.abs(q[:, :, 5]) + np.float32(0.1)

    def run(k, v):
        out = torch.empty((seq, nh, 128), dtype=torch.float32, device="cuda")
        args = (nh, nkv, 128, pos0, dev(q), seq, dev(k.reshape(-1)), dev(v.reshape(-1)), max_seq, out)
        assert takes_it(gpu, lambda: gpu.GpuAttentionFromCache(*args))
        return host(out)

    plain = run(kc, vc)
    first = max(key - pos0, 0)  # the first token that sees it
    v = vc.copy().reshape(nkv, max_seq, 128)
    v[3, key, 77] = np.float16(-np.inf).view(np.uint16)
    got = run(kc, v)
    assert np.all(got[first:, 6:8, 77] == -np.inf)
    rest = np.ones(plain.shape, bool)
    rest[first:, 6:8, 77] = False
    assert np.array_equal(got[rest], plain[rest])
    v[3, key - 1 if key else 1, 77] = np.float16(np.inf).view(np.uint16)
    assert np.all(np.isnan(run(kc, v)[max(key - pos0, 1):, 6:8, 77]))

    k = kc.copy().reshape(nkv, max_seq, 128)
    k[3, key, 5] = np.float16(-np.inf).view(np.uint16)
    got = run(k, vc)
    rest = np.ones(plain.shape, bool)
    rest[first:, 6:8] = False
    assert np.array_equal(got[rest], plain[rest])
    # scores and values of size 1: 1e-5 is 80 roundings of 2^-23
    assert np.allclose(got, reference(q, k, vc, max_seq, nkv, pos0), rtol=0, atol=1e-5)
    k[3, key, 5] = np.float16(np.inf).view(np.uint16)
    got = run(k, vc)
    assert np.all(np.isnan(got[first:, 6:8])) and np.array_equal(got[rest], plain[rest])


@pytest.mark.parametrize("nh,nkv,pos0,seq,decode", [(32, 8, 1500, 21, 1.891e-7), (16, 4, 1024, 63, 1.891e-7),
                                                       (16, 8, 1500, 45, 2.2e-7)])
def test_turn_error_is_below_the_decode_kernels(gpu, ora, nh, nkv, pos0, seq, decode):
    """Queries, probabilities and sums as two fp16 terms lose nothing against the fp32 kernel
    that took these calls: `decode` is that kernel's error (2-norm, relative) on these inputs."""
    import torch

    max_seq = 2048
    rng = np.random.default_rng(pos0 + seq)
    q, kc, vc = make(rng, nh, nkv, max_seq, seq)
    out = torch.empty((seq, nh, 128), dtype=torch.float32, device="cuda")
    gpu.GpuAttentionFromCache(nh, nkv, 128, pos0, dev(q), seq, dev(kc), dev(vc), max_seq, out)
    ref = ora.attention_f64(q, kc, vc, max_seq, nh, nkv, 128, pos0, seq)[0]
    err = float(np.linalg.norm(host(out).astype(np.float64) - ref) / np.linalg.norm(ref))
    assert err <= decode
