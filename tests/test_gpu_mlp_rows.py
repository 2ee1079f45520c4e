"""The network's row kernels at the edges of their ranges: 16 rows per workgroup up to 4096 rows, 32 up to
8192, 64 above, and gradients whose last split of 256 rows is short.

A row's output does not depend on which kernel or workgroup computed it (the same products in the same
order), so calls of different sizes agree bit for bit; the largest is held against the oracle at the bars of
test_gpu_mlp.py.
"""
import numpy as np
import pytest

import mlp_oracle as mo
from crime_amd.emulator import Mlp

pytestmark = pytest.mark.gpu


def data(n, seed):
    rng = np.random.default_rng(seed)
    x = rng.normal(size=(n, 8)).astype(np.float32)
    return x, (np.sin(x[:, 0]) + 0.5 * x[:, 1] * x[:, 2]).astype(np.float32)


@pytest.mark.parametrize("n", [1, 15, 17, 4096, 4097, 8192, 8193, 8255])
def test_forward_does_not_depend_on_the_call_size(n):
    p = mo.init_params(7)
    x, _ = data(8255, 8)
    x[3] *= 40.0      # activations far into both tails of the SiLU
    with Mlp(max_batch=16384) as net:
        net.set_params(p)
        y = net.forward(x[:n])
        parts = np.concatenate([net.forward(x[i:min(n, i + 1000)]) for i in range(0, n, 1000)])
    assert np.array_equal(y, parts)
    if n < len(x):      # the oracle's bars are quantiles over many rows
        return
    ref, _, _ = mo.forward(p, x[:n], bf16=True)
    err = np.abs(y - ref) / np.sqrt(np.mean(ref ** 2))
    assert np.percentile(err, 90) < 1e-6 and err.max() < 5e-2


@pytest.mark.parametrize("n", [64, 320, 2112])
def test_gradient_with_a_short_last_split(n):
    """n rows end in a split of 64; 4 n rows whose others weigh nothing fill every split.  The loss's 1/n scales
    every row's gradient by the power of two, which no rounding sees, and the others add zeros."""
    p = mo.init_params(9)
    x, t = data(4 * n, 10)
    w = np.exp(np.random.default_rng(11).normal(size=4 * n)).astype(np.float32)
    w[n:] = 0
    with Mlp(max_batch=64 * 133) as net:
        net.set_params(p)
        loss, g = net.loss_grad(x[:n], t[:n], w[:n])
        loss4, g4 = net.loss_grad(x, t, w)
    assert abs(loss - 4 * loss4) <= 1e-5 * loss     # FP32 atomics, in any order
    assert np.abs(g).max() > 0
    assert np.array_equal(g, 4 * g4)
