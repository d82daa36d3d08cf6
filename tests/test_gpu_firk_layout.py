"""The FIRK kernels' lane-interleaved areas and row-exchange pass at the sizes where they can
go wrong: fewer intervals than lanes, one per lane, one lane with one more, chunks of two
and three, in one launch; with local systems of 2, 4, 6, 10 unknowns and 14 (rolled), that
need no row exchange (Bratu) or need one in every interval (u'' = k^2 u with h k^2 > 10).

Tolerances: as tests/test_gpu_firk.py -- residual 1e-12, Newton correction and solves 1e-9
relative; the nested form's residual 1e-11 (an inner solve may stop one iteration apart).
"""
import sys

import numpy as np
import pytest

from boundaryvaluediffeq_amd import _abi, _lib
import pyoracle as O
import cases
from test_gpu_firk import _opts, _oopts

pytestmark = pytest.mark.gpu

SIZES = (1, 2, 3, 63, 64, 65, 127, 128, 129, 191, 193)


def _stiff(N, k2=4000.0):
    return cases.linear([[0, 1], [k2, 0]], tspan=(0.0, 1.0), bc=([(0, 1.0)], [(0, 0.0)]), dt=1.0 / N)


@pytest.mark.parametrize("nested", [False, True], ids=["expanded", "nested"])
@pytest.mark.parametrize("code", [101, 102, 103, 105, 107, 303])
def test_firk_layout(code, nested):
    print("firk layout", code, nested, flush=True)
    sys.stdout.flush()
    ctx = _lib.context(0)
    nc = code + (_abi.FIRK_NESTED if nested else 0)
    rng = np.random.default_rng(code)
    specs = [cases.random_state(cases.bratu(1.0, N=n), rng, 0.2) for n in SIZES]
    for s, g in zip(specs, _lib.firk_residual(ctx, nc, specs)):
        ref = O.firk_residual(nc, s)
        assert np.max(np.abs(g - ref)) <= (1e-11 if nested else 1e-12) * max(1.0, np.max(np.abs(ref))), s.N
    for s, g in zip(specs, _lib.firk_newton_step(ctx, nc, specs)):
        ref = O.firk_newton_step(nc, s)
        assert np.max(np.abs(g - ref)) <= 1e-9 * max(1.0, np.max(np.abs(ref))), s.N
    kw = dict(adaptive=0, newton_abstol=1e-11)
    specs = [cases.bratu(1.0 + 0.1 * i, N=n) for i, n in enumerate(SIZES)]
    specs += [_stiff(n) for n in SIZES if n > 3]
    ref = [O.solve(_oopts(nc, **kw), s) for s in specs]
    for s, g, r in zip(specs, _lib.solve_batch(ctx, _opts(nc, **kw), specs), ref):
        assert g.retcode == r.retcode and g.N == r.N == s.N, (g.retcode, r.retcode, s.N)
        if r.retcode == 0:
            assert np.max(np.abs(g.u - r.u) / np.maximum(1.0, np.abs(r.u))) <= 1e-9, s.N
            assert np.max(np.abs(g.stages - r.stages) / np.maximum(1.0, np.abs(r.stages))) <= 1e-9, s.N
    assert sum(r.retcode == 0 for r in ref) >= len(SIZES), [r.retcode for r in ref]
