"""The matmul on decoded weight planes (512 tokens and more, and fewer on large
matrices): ragged row groups, row and token tiles, one block to several, against the
float64 oracle within the bound of tests/test_gpu_matmul.py."""
from __future__ import annotations

import os
import subprocess
import sys

import numpy as np
import pytest

import synth
from test_gpu_matmul import check, dev, factored_magnitude, host

pytestmark = pytest.mark.gpu

Q4, Q6 = 12, 14


@pytest.mark.parametrize("t", [Q4, Q6])
@pytest.mark.parametrize("rows,cols,n", [(1, 256, 512), (31, 768, 513), (33, 512, 640), (129, 1280, 700), (257, 2048, 641),
                                         (300, 2560, 1025), (9700, 2560, 385), (2560, 9728, 448)])
def test_planes_matmul_vs_f64(gpu, ora, t, rows, cols, n):
    import torch

    rng = np.random.default_rng(rows + cols + n + t)
    w = synth.quant_table(rng, t, rows, cols)
    x = rng.normal(0, 1, (n, cols)).astype(np.float32)
    x[n // 2] *= 1e-20  # tokens of very different size keep their own scale
    out = torch.full((n + 1, rows), np.nan, dtype=torch.float32, device="cuda")
    gpu.profile_start(16)
    gpu.GpuMatMulQuant(gpu.GpuTensor(dev(w), t, rows, cols), dev(x), n, out[:n])
    gpu.profile_stop()
    assert "MatMulMfmaQ%dKPlanesKernel" % (4 if t == Q4 else 6) in gpu.profile_report()
    exact, absdot = ora.matmul_quant_f64(t, w, rows, cols, x)
    check(host(out[:n]), exact, absdot, cols, factored_magnitude(ora, t, w, rows, cols, x))
    assert torch.isnan(out[n]).all(), "wrote past the last token"


CAPTURE = """
import torch
from rpgbarenginecuda_amd import ops

ops.init()
gen = torch.Generator(device="cuda")
gen.manual_seed(1)


def matrix(rows, cols):
    b = torch.randint(0, 256, (rows * cols // 256, 144), generator=gen, device="cuda", dtype=torch.uint8)
    b[:, 0:4] = 20  # the fp16 scales: 0x1414
    return ops.GpuTensor(b.reshape(-1), 12, rows, cols)


def capture(w, x, out, refused):
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    stream.wait_stream(torch.cuda.current_stream())
    with ops.ScopedEngineStream(stream), torch.cuda.stream(stream):
        graph.capture_begin()
        try:
            ops.GpuMatMulQuant(w, x, len(x), out)
            assert not refused, "captured without its buffers"
        except ops.RpgError as e:
            assert refused and "run the same shape once before capturing" in str(e), e
        finally:
            graph.capture_end()
    torch.cuda.synchronize()
    return graph


def kernels(call):
    ops.profile_start(16)
    call()
    ops.profile_stop()
    return set(ops.profile_report())


w, other = matrix(9728, 2560), matrix(9728, 3072)
x = torch.randn(448, 2560, generator=gen, device="cuda")
out, eager = (torch.empty(448, 9728, device="cuda") for _ in range(2))
# the activations' buffer, from a call on the GEMM that decodes as it goes
x3 = torch.randn(384, 3072, generator=gen, device="cuda")
assert "MatMulMfmaQ4KKernel" in kernels(lambda: ops.GpuMatMulQuant(other, x3, 384, eager))
capture(w, x, out, True)
assert "MatMulMfmaQ4KPlanesKernel" in kernels(lambda: ops.GpuMatMulQuant(w, x, 448, eager))
graph = capture(w, x, out, False)
for scale in (1.0, -2.0, 0.5):
    x *= scale
    out.fill_(float("nan"))
    graph.replay()
    ops.GpuMatMulQuant(w, x, 448, eager)
    torch.cuda.synchronize()
    assert torch.equal(out, eager)
print("done", flush=True)
"""


def test_planes_capture_takes_the_eager_route():
    """448 tokens on a matrix that runs on the planes, in a process of its own (the library's
    buffers only grow): captured before the shape has run, with the activations' buffer
    there from another call, it is refused and not sent to another kernel; after a run,
    replays give the eager bits."""
    repo = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    run = subprocess.run([sys.executable, "-c", CAPTURE], cwd=repo, timeout=100, capture_output=True, text=True)
    assert run.returncode == 0 and "done" in run.stdout, run.stderr[-2000:]
