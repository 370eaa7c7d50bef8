"""The small-batch quantised matmul (2 tokens to a medium prompt): every workgroup shape
at the edges of its tiles, against the float64 oracle within the fp32 summation
bound of tests/test_gpu_matmul.py, and against itself where the bits must agree. The
sizes are ones that the rule sends to the kernel; each test checks that it ran."""
from __future__ import annotations

import numpy as np
import pytest

import synth
from test_gpu_matmul import check, dev, host

pytestmark = pytest.mark.gpu

Q4, Q6 = 12, 14

def launches(gpu, call):
    gpu.profile_start(16)
    call()
    gpu.profile_stop()
    return set(gpu.profile_report())


def small(gpu, t, call):
    """The call's launches are the kernel of that type, and perhaps its reduce."""
    return launches(gpu, call) - {"MatMulSmallReduceKernel"} == {"MatMulSmallQ%dKKernel" % (4 if t == Q4 else 6)}


def centred_magnitude(ora, t, w, rows, cols, x):
    """Q4_K only: sum_e (|d1 (q_e - 8)| + |8 d1 - m1|) |x_e|, the terms that the kernel sums:
    it multiplies by the centred quants and adds what the centring took by the runs' sums.
    (A column a thousand times the others with quant 0 and a small m1 rounds by 8 d1 of it,
    which the weight itself does not bound.) A copy of the matrix with every quant 8
    dequantises to 8 d1 - m1."""
    if t != Q4:
        return 0.0
    z = np.array(w, copy=True).reshape(-1, 144)
    z[:, 16:] = 0x88
    n = rows * cols
    wd = ora.dequantize_row(t, np.ascontiguousarray(w), n).reshape(rows, cols).astype(np.float64)
    w8 = ora.dequantize_row(t, z.reshape(-1), n).reshape(rows, cols).astype(np.float64)
    return np.abs(np.asarray(x, np.float64).reshape(-1, cols)) @ (np.abs(wd - w8) + np.abs(w8)).T


SHAPES = [
    # (type, rows, cols, tokens)
    (Q4, 1, 256, 33), (Q6, 1, 256, 40),            # one row, one block
    (Q4, 17, 768, 36), (Q6, 15, 768, 49),          # ragged row tile, odd blocks, one token over a tile
    (Q4, 2049, 2048, 9), (Q4, 700, 2048, 31), (Q4, 300, 2048, 33),  # up to the slices' limit and over it
    (Q6, 7001, 1280, 25),                          # 5 blocks: waves with nothing to do
    (Q4, 2049, 2048, 65), (Q6, 2049, 2048, 97),    # ragged rows and token tiles, several tiles per workgroup
    (Q6, 20001, 2048, 17), (Q4, 20000, 512, 21),   # many tiles
    (Q4, 9001, 768, 16), (Q6, 9003, 512, 21), (Q4, 30001, 256, 9),  # short rows
    (Q6, 3003, 2304, 10), (Q4, 3001, 2560, 19),    # 9 and 10 blocks
    (Q6, 5001, 2560, 100), (Q4, 5001, 2560, 150),  # 10 blocks in two slices
    (Q6, 2001, 2816, 30), (Q6, 1000, 2816, 40),    # 11 blocks: walked by a workgroup, in slices of unequal length
    (Q4, 2501, 9728, 18), (Q6, 500, 9728, 30), (Q4, 500, 9728, 36),  # 38 blocks likewise
]


@pytest.mark.parametrize("t,rows,cols,n", SHAPES)
def test_small_matmul_vs_f64(gpu, ora, t, rows, cols, n):
    import torch

    rng = np.random.default_rng(rows + cols + n + t)
    w = synth.quant_table(rng, t, rows, cols)
    x = rng.normal(0, 1, (n, cols)).astype(np.float32)
    x[n // 2] *= 1e-20  # tokens of very different size keep their own scale
    x[:, cols // 2] *= 1e3
    out = torch.full((n + 1, rows), np.nan, dtype=torch.float32, device="cuda")
    assert small(gpu, t, lambda: gpu.GpuMatMulQuant(gpu.GpuTensor(dev(w), t, rows, cols), dev(x), n, out[:n]))
    exact, absdot = ora.matmul_quant_f64(t, w, rows, cols, x)
    check(host(out[:n]), exact, absdot, cols, centred_magnitude(ora, t, w, rows, cols, x))
    assert torch.isnan(out[n]).all(), "wrote past the last token"


@pytest.mark.parametrize("off", [2, 6, 14])
@pytest.mark.parametrize("rows,cols,n", [(2501, 2560, 21), (2001, 2816, 30), (131, 2560, 40)])
def test_small_matmul_unaligned_q6k(gpu, rows, cols, n, off):
    """A Q6_K matrix at any even address gives the bits of the aligned one."""
    import torch

    rng = np.random.default_rng(off)
    w = dev(synth.quant_table(rng, Q6, rows, cols))
    moved = torch.zeros(w.numel() + 64, dtype=torch.uint8, device="cuda")
    moved[off:off + w.numel()] = w
    x = dev(rng.normal(0, 1, (n, cols)).astype(np.float32))
    outs = [torch.empty((n, rows), device="cuda") for _ in range(2)]
    for buf, out in zip((w, moved[off:off + w.numel()]), outs):
        assert small(gpu, Q6, lambda: gpu.GpuMatMulQuant(gpu.GpuTensor(buf, Q6, rows, cols), x, n, out))
    assert torch.equal(*outs)


@pytest.mark.parametrize("cols,n", [(256, 30), (512, 100), (768, 40), (2048, 21), (2048, 40), (2048, 200), (2560, 21), (2560, 70), (6144, 20), (6144, 50)])
def test_small_group_and_swiglu_equal_separate_calls(gpu, cols, n):
    """Matrices of both types and of sizes that prefer different shapes, each bit-identical to its own call;
    gate / up likewise to the two products followed by SwiGLU."""
    import torch

    rng = np.random.default_rng(cols + n)
    x = dev(rng.normal(0, 1, (n, cols)).astype(np.float32))
    ws = [gpu.GpuTensor(dev(synth.quant_table(rng, t, r, cols)), t, r, cols)
          for t, r in ((Q4, 2048), (Q4, 129), (Q6, 1024), (Q4, 9728), (Q4, 9728))]
    alone = [torch.empty((n, w.rows), device="cuda") for w in ws]
    for w, o in zip(ws, alone):
        gpu.GpuMatMulQuant(w, x, n, o)
    outs = [torch.empty_like(o) for o in alone]
    gpu.GpuMatMulQuantGroup(ws, x, n, outs)
    for w, a, o in zip(ws, alone, outs):
        assert torch.equal(a, o), (w.type, w.rows)
    gate, up = torch.empty_like(alone[3]), torch.empty_like(alone[4])
    gpu.GpuMatMulQuantSwiGLU(ws[3], ws[4], x, n, gate, up)
    gpu.GpuSiluMulInPlace(alone[3], alone[4], n * 9728)
    assert torch.equal(gate, alone[3])
    assert torch.equal(up, alone[4]), "up holds its own product after a call of several tokens"


@pytest.mark.parametrize("t", [Q4, Q6])
@pytest.mark.parametrize("rows,cols,n", [(40, 2048, 40), (1500, 6144, 24), (40, 6144, 48)])
def test_small_one_hot_selects_columns(gpu, ora, t, rows, cols, n):
    """A single activation 1 gives the dequantised weight, bit for bit."""
    import torch

    rng = np.random.default_rng(t + cols + n)
    w = synth.quant_table(rng, t, rows, cols)
    picks = rng.permutation(cols)[:n]
    x = np.zeros((n, cols), np.float32)
    x[np.arange(n), picks] = 1.0
    out = torch.empty((n, rows), device="cuda")
    assert small(gpu, t, lambda: gpu.GpuMatMulQuant(gpu.GpuTensor(dev(w), t, rows, cols), dev(x), n, out))
    want = ora.dequantize_row(t, w, rows * cols).reshape(rows, cols)[:, picks].T
    assert np.array_equal(host(out), want)


def test_small_matmul_captures_without_a_first_run(gpu):
    """Below 32 tokens a call needs no buffer of the library, also for a long K."""
    import torch

    rows, cols, n = 3000, 16384, 7
    rng = np.random.default_rng(5)
    w = gpu.GpuTensor(dev(synth.quant_table(rng, Q4, rows, cols)), Q4, rows, cols)
    x = dev(rng.normal(0, 1, (n, cols)).astype(np.float32))
    out, eager = torch.empty((n, rows), device="cuda"), torch.empty((n, rows), device="cuda")
    st, g = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    st.wait_stream(torch.cuda.current_stream())
    with gpu.ScopedEngineStream(st), torch.cuda.graph(g, stream=st):
        gpu.GpuMatMulQuant(w, x, n, out)
    for scale in (1.0, -2.0):
        x *= scale
        out.fill_(float("nan"))
        g.replay()
        assert launches(gpu, lambda: gpu.GpuMatMulQuant(w, x, n, eager)) == {"MatMulSmallQ4KKernel"}
        torch.cuda.synchronize()
        assert torch.equal(out, eager)


@pytest.mark.parametrize("t,rows,cols,n", [(Q4, 6144, 2048, 21), (Q6, 6144, 2048, 12), (Q6, 2048, 6144, 21),
                                           (Q4, 4000, 2560, 21)])
def test_small_infinite_activation(gpu, ora, t, rows, cols, n):
    """Below 32 tokens an infinite or NaN activation gives what the sum of the dequantised
    weights' products gives (an infinity of the weight's sign, NaN where the weight is 0),
    as the tiled kernel does; the other tokens keep their bits. Alone, in a group and
    under SwiGLU."""
    import torch

    rng = np.random.default_rng(t + rows + cols + n)
    raw = [synth.quant_table(rng, t, rows, cols) for _ in range(2)]
    ws = [gpu.GpuTensor(dev(w), t, rows, cols) for w in raw]
    x = rng.normal(0, 1, (n, cols)).astype(np.float32)
    plain = torch.empty((n, rows), device="cuda")
    gpu.GpuMatMulQuant(ws[0], dev(x), n, plain)
    bad = [0, n // 2, n - 1]
    x[bad[0], cols // 3] = -np.inf
    x[bad[1], cols - 1] = np.inf
    x[bad[2], 0] = np.nan
    xd = dev(x)
    outs = [torch.empty((n, rows), device="cuda") for _ in range(3)]
    assert small(gpu, t, lambda: gpu.GpuMatMulQuant(ws[0], xd, n, outs[0]))
    gpu.GpuMatMulQuantGroup(ws, xd, n, outs[1:])
    gate, up = torch.empty((n, rows), device="cuda"), torch.empty((n, rows), device="cuda")
    gpu.GpuMatMulQuantSwiGLU(ws[0], ws[1], xd, n, gate, up)
    wants = []
    for w in raw:
        w = ora.dequantize_row(t, w, rows * cols).reshape(rows, cols).astype(np.float64)
        with np.errstate(invalid="ignore"):
            wants.append(np.stack([(w * x[b].astype(np.float64)).sum(1) for b in bad]))
    assert np.isinf(wants[0][:2]).any() and not np.isfinite(wants[0]).any()
    good = [i for i in range(n) if i not in bad]
    for out, want in ((outs[0], wants[0]), (outs[1], wants[0]), (outs[2], wants[1]), (up, wants[1])):
        assert np.array_equal(host(out)[bad].astype(np.float64), want, equal_nan=True)
    assert np.array_equal(host(outs[0])[good], host(plain)[good])
    gpu.GpuSiluMulInPlace(outs[1], outs[2], n * rows)
    assert np.array_equal(host(gate), host(outs[1]), equal_nan=True)


@pytest.mark.parametrize("n", [33, 48, 64])
def test_small_short_prompt_of_a_shard_is_one_launch(gpu, n):
    """q / k / v of a tensor-parallel shard (512 rows of 2048 columns): K fits the workgroups, so
    there are no slices to sum."""
    import torch

    rng = np.random.default_rng(n)
    ws = [gpu.GpuTensor(dev(synth.quant_table(rng, t, r, 2048)), t, r, 2048) for t, r in ((Q4, 256), (Q4, 128), (Q6, 128))]
    x = dev(rng.normal(0, 1, (n, 2048)).astype(np.float32))
    outs = [torch.empty((n, w.rows), device="cuda") for w in ws]
    assert launches(gpu, lambda: gpu.GpuMatMulQuantGroup(ws, x, n, outs)) == {"MatMulSmallQ4KQ6KKernel"}
    assert launches(gpu, lambda: gpu.GpuMatMulQuant(ws[0], x, n, outs[0])) == {"MatMulSmallQ4KKernel"}


@pytest.mark.parametrize("n", [1, 8, 21, 64, 600])
def test_group_refuses_null_activations(gpu, n):
    """On the host, whatever kernel the group would take (nothing is launched)."""
    import torch

    rng = np.random.default_rng(n)
    ws = [gpu.GpuTensor(dev(synth.quant_table(rng, t, 2048, 2048)), t, 2048, 2048) for t in (Q4, Q6)]
    outs = [torch.empty((n, 2048), device="cuda") for _ in ws]
    with pytest.raises(gpu.RpgError, match="null pointer"):
        gpu.GpuMatMulQuantGroup(ws, None, n, outs)


@pytest.mark.parametrize("t,rows,cols,n,kernel", [
    # measured there and here, us: 74 and 103, 84 and 120, 94 and 106, 99 and 108; 12.4 and 14.3
    (Q4, 9728, 2560, 300, "MatMulMfmaQ4KKernel"), (Q4, 5120, 5120, 333, "MatMulMfmaQ4KKernel"),
    (Q4, 2560, 9728, 333, "MatMulMfmaQ4KKernel"), (Q6, 9728, 2560, 300, "MatMulMfmaQ6KKernel"),
    (Q4, 2048, 6144, 3, "MatMulQ4KKernel"),
    # 55 and 43, 123 and 104, 141 and 128, 36 and 22, 35 and 26
    (Q4, 6144, 2048, 300, "MatMulSmallQ4KKernel"), (Q6, 2560, 9728, 333, "MatMulSmallQ6KKernel"),
    (Q6, 32000, 2048, 200, "MatMulSmallQ6KKernel"), (Q4, 6144, 2048, 128, "MatMulSmallQ4KKernel"),
    (Q4, 12000, 512, 224, "MatMulSmallQ4KKernel")])
def test_small_route_is_the_faster_kernel(gpu, t, rows, cols, n, kernel):
    import torch

    w = torch.zeros(rows * cols // 256 * (144 if t == Q4 else 210), dtype=torch.uint8, device="cuda")
    x, out = torch.zeros((n, cols), device="cuda"), torch.empty((n, rows), device="cuda")
    assert kernel in launches(gpu, lambda: gpu.GpuMatMulQuant(gpu.GpuTensor(w, t, rows, cols), x, n, out))
