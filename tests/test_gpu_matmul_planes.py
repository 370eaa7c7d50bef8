"""The matmul on decoded weight planes (512 tokens and more, and fewer on large
matrices): ragged row groups, row and
token tiles, one block to several, against the float64 oracle within the bound of
tests/test_gpu_matmul.py."""
from __future__ import annotations

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
    gpu.GpuMatMulQuant(gpu.GpuTensor(dev(w), t, rows, cols), dev(x), n, out[:n])
    exact, absdot = ora.matmul_quant_f64(t, w, rows, cols, x)
    check(host(out[:n]), exact, absdot, cols, factored_magnitude(ora, t, w, rows, cols, x))
    assert torch.isnan(out[n]).all(), "wrote past the last token"
