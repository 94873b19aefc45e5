"""The network's forward pass and gradient at the row counts where the
kernels' blocks end: 16 rows a wave, 64 a workgroup, 8192 where a chunk of
the weight gradients takes more than one workgroup's rows; against the numpy
restatement.  Both round the same operands to bfloat16 and sum in single
precision in another order, so an operand at a rounding boundary may fall to
the other side (2^-8 of itself): 1e-2 of the largest output at one row, 1e-4
of a gradient's norm where many rows are summed, 1e-2 for a few."""
import ctypes
import importlib
import os
import sys

import numpy as np
import pytest

from conftest import ROOT, load_pkg

sys.path.insert(0, os.path.join(ROOT, "oracle"))
import mlp_oracle as mo  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 15, 16, 17, 63, 64, 65, 1024, 8191, 8192, 8193, 20001])
def test_rows(rows):
    sps = load_pkg()
    sur = importlib.import_module("stress-particle-sph_amd.surrogate")
    net = sur.Network(ctypes.CDLL(sps.PRODUCT_LIB), seed=4, batch_rows=rows)
    print(f"[network] {rows} rows", flush=True)
    theta = net.params()
    rng = np.random.default_rng(rows)
    x = rng.standard_normal((rows, 10)).astype(np.float32)
    t = rng.standard_normal((rows, 4)).astype(np.float32)
    y, yo = net.forward(x), mo.forward(theta, x)[0]
    assert np.abs(y - yo).max() <= 1e-2 * np.abs(yo).max()
    lo, go = mo.loss_and_grad(theta, x, t)
    for _ in range(2):          # the second in the buffers of the first
        loss, g = net.gradient(x, t)
        assert abs(loss - lo) <= 1e-3 * lo
        assert np.linalg.norm(g - go) <= (1e-4 if rows >= 1000 else 1e-2) * np.linalg.norm(go)
