"""The equidistribution walk and the transfer's chained base values at their block edges: both
take 64 intervals (nodes) at a time, so old and new meshes lie around multiples of 64, with
meshes that shrink, stay about the same (long chains within a block) and grow.

The states are Bratu solutions with noise of 1e-5 at the nodes: every defect is far above
rounding, so the new nodes are determined to about 1e-13 / (smallest defect) (the noise of a
defect, times 100 as in tests/test_gpu_parity.py) and the values by the slope times that."""
import sys

import numpy as np
import pytest

from boundaryvaluediffeq_amd import _abi, _lib
import pyoracle as O
import cases

pytestmark = pytest.mark.gpu

SIZES = (1, 2, 3, 31, 32, 33, 58, 59, 63, 64, 65, 116, 127, 128, 129, 200)


def _specs(method):
    out = []
    for n in SIZES:
        s = cases.bratu(2.0, N=4).with_state(np.linspace(0.0, 1.0, n + 1), np.zeros(2 * (n + 1)))
        st = O.solve(O.opts(method, adaptive=0, newton_abstol=1e-12), s)
        noise = 1e-5 * np.random.default_rng(n).standard_normal(st.u.size)
        out.append(s.with_state(st.t, st.u.reshape(-1) + noise))
    return out


@pytest.mark.parametrize("mode", [_abi.TRANSFER_REFERENCE, _abi.TRANSFER_CLEAN])
@pytest.mark.parametrize("abstol", [0.3, 1e-5, 1e-8])
@pytest.mark.parametrize("method", [4, 6])
def test_walk_and_chain(method, abstol, mode):
    print("mesh walk", method, abstol, mode, flush=True)
    sys.stdout.flush()
    specs = _specs(method)
    o = _abi.default_opts(method)
    o.abstol = abstol
    o.transfer_mode = mode
    moved = 0
    for s, (info, n, t, y) in zip(specs, _lib.mesh_select(_lib.context(0), o, specs)):
        ri, rn, rt, ry = O.mesh_select(O.opts(method, abstol=abstol, transfer_mode=mode), s)
        assert (info, n) == (int(ri), int(rn)), s.N
        if info != 0:
            continue
        moved += 1
        e, _ = O.defect(method, s)
        tol_t = max(1e-10, 1e-13 / np.min(np.max(np.abs(e), axis=1)))
        assert np.max(np.abs(t - rt)) <= tol_t, s.N
        assert np.max(np.abs(y - ry)) <= (1e-9 + 10 * tol_t) * max(1.0, np.max(np.abs(ry))), s.N
    assert moved >= len(SIZES) - 3
