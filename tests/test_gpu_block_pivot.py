"""Pivots of the FP64 block elimination where only FP64 can tell the candidates apart: with
A = [[0, X], [Y, 0]] of size 1e60 and diag(XY) = diag(YX) = 0, the diagonals of the block rows
(A^2 up to rounding) are some 1e16 times smaller than the entries around them, and all of them are
larger than FP32 holds.  A comparison in FP32 takes the first of these infinities, a diagonal
entry, and the elimination loses every digit.

Tolerance: 1e-9 relative to the largest entry, as tests/test_gpu_block.py; the blocks' rows
are all of one size and the system's condition that of X and Y (about 10).
"""
import sys

import numpy as np
import pytest

from boundaryvaluediffeq_amd import _abi, _lib
import pyoracle as O
import cases

pytestmark = pytest.mark.gpu


def _trap(rng, M, scale):
    h = M // 2
    X, Y = (rng.uniform(0.5, 2, (h, h)) * rng.choice([-1, 1], (h, h)) for _ in range(2))
    C = np.zeros((2 * h, h * h))  # diag(XY) and diag(YX) as linear functions of Y
    for i in range(h):
        C[i, i::h] = X[i]
        C[h + i, i * h:(i + 1) * h] = X[:, i]
    Y = Y - np.linalg.lstsq(C, C @ Y.reshape(-1), rcond=None)[0].reshape(h, h)
    A = np.zeros((M, M))
    A[:h, h:], A[h:, :h] = X, Y
    return A * scale


@pytest.mark.parametrize("method", [4, 6])
@pytest.mark.parametrize("M", [8, 16])
def test_pivots_are_compared_in_fp64(M, method):
    print("block pivots", M, method, flush=True)
    sys.stdout.flush()
    specs = []
    for seed in range(3):
        for N in (1, 2, 8, 9, 17):
            rng = np.random.default_rng(seed)
            bc = ([(k, rng.standard_normal()) for k in range(M // 2)],
                  [(k, rng.standard_normal()) for k in range(M // 2, M)])
            # MIRK6 multiplies A three times: 1e180, and pivot products stay finite
            s = cases.linear(_trap(rng, M, 1e60 if method == 4 else 1e45), c=0.1, tspan=(0.0, 1.0), bc=bc, dt=1.0 / N)
            specs.append(cases.random_state(s, rng, 0.3))
    got = _lib.newton_step(_lib.context(0), method, specs, precision=_abi.PREC_FP64)
    for s, d in zip(specs, got):
        ref = O.newton_step(method, s)
        assert np.all(np.isfinite(ref))
        assert np.max(np.abs(d - ref)) <= 1e-9 * max(1.0, np.max(np.abs(ref))), s.N
