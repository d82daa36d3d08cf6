"""The network kernels at the edges of their tiles: gradients over tile counts around the
four quarters in which the per-tile slots are summed (fewer tiles than quarters, uneven
quarters, more than sixteen slots per quarter) and around the ranges of points of the hidden
matrices' gradients (fewer steps than waves, one, two and eight ranges, uneven), predictions of one point, around a tile of 64,
and with more than eight tiles per workgroup (two rounds of features read ahead).

Tolerances: as tests/test_gpu_mlp.py -- outputs 5e-3 and gradients 1e-2 relative (FP32
summation order flips single BF16 roundings), loss 1e-4.
"""
import sys

import numpy as np
import pytest

from boundaryvaluediffeq_amd import _lib
import mlp_oracle as MO
from test_gpu_mlp import _net

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 65, 3 * 64, 5 * 64, 33 * 64 + 5, 35 * 64, 130 * 64 + 1])
def test_gradient_slots(n):
    print("mlp gradient slots", n, flush=True)
    sys.stdout.flush()
    net, w, norm = _net(_lib.context(0), seed=6)
    rng = np.random.default_rng(n)
    x = rng.uniform(-1, 1, (n, 4)).astype(np.float32)
    y = rng.normal(0, 1, (n, 2)).astype(np.float32)
    loss, g = net.gradient(x, y)
    lr, gr = MO.loss_and_grad(w, x, y, norm, emulate=True)
    assert abs(loss - lr) <= 1e-4 * lr
    assert np.linalg.norm(g - gr) <= 1e-2 * np.linalg.norm(gr)
    assert np.array_equal(net.gradient(x, y)[1], g)  # the sums have a fixed order


@pytest.mark.parametrize("n", [1, 63, 64, 65, 511, 513, 64 * 256 + 1, 64 * 256 * 9 + 7])
def test_predict_tiles(n):
    print("mlp predict tiles", n, flush=True)
    sys.stdout.flush()
    net, w, norm = _net(_lib.context(0), seed=7)
    x = np.random.default_rng(n).uniform(-1.5, 1.5, (n, 4)).astype(np.float32)
    got = net.predict(x)
    ref, _ = MO.forward(w, x, norm, emulate=True)
    scale = np.asarray(norm[3], np.float32)
    assert np.all(np.abs(got - ref) <= 5e-3 * (np.abs(ref) + scale)), np.max(np.abs(got - ref))
