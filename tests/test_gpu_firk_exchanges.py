"""FIRK local systems that need row exchanges, where they have to succeed: stiff linear problems
of every FIRK state dimension (all of them, and among Bratu problems that need none, so that
one launch takes both passes), in the kernels with and without the trust-region stage, and
the nested form's dense output where neighbouring threads hold instances of different families.

Tolerances: nodes 1e-9 relative, dense output 1e-11, as tests/test_gpu_firk.py.  Stages 1e-9
relative to the instance's largest: a stage equation K = f(y + h A K) multiplies K by
h k2 (up to 12,000 here), so its evaluation alone rounds by eps h k2 |K| < 3e-12 |K|, in every
entry alike, and the two sides stop at max|F| <= 1e-9 in an iterate of their own.
"""
import sys

import numpy as np
import pytest

import boundaryvaluediffeq_amd as bvp
from boundaryvaluediffeq_amd import _abi, _lib
import pyoracle as O
import cases

pytestmark = pytest.mark.gpu

SIZES = (4, 63, 64, 65, 130)


def _stiff(M, N, k2):
    """Pairs u'' = k2 u with u(0) = 1, u(1) = 0, coupled weakly; a last odd component decays."""
    A = np.zeros((M, M))
    bca, bcb = [], []
    for p in range(M // 2):
        A[2 * p, 2 * p + 1], A[2 * p + 1, 2 * p] = 1.0, k2 * (1 + p)
        bca.append((2 * p, 1.0))
        bcb.append((2 * p, 0.0))
    if M % 2:
        A[M - 1, M - 1] = -k2 if M == 1 else -5.0
        if M > 1:
            A[M - 1, 0] = 0.3
        bca.append((M - 1, 1.0))
    return cases.linear(A, c=0.0, tspan=(0.0, 1.0), bc=(bca, bcb), dt=1.0 / N)


def _check(code, specs, stages, want_ok):
    kw = dict(adaptive=0, newton_abstol=1e-9, nlsolve_stages=stages, nest_abstol=1e-9)
    o = _abi.default_opts(code)
    for k, v in kw.items():
        setattr(o, k, v)
    ref = [O.solve(O.opts(code, **kw), s) for s in specs]
    assert all(r.retcode == 0 for r, w in zip(ref, want_ok) if w), [r.retcode for r in ref]
    for s, g, r in zip(specs, _lib.solve_batch(_lib.context(0), o, specs), ref):
        assert g.retcode == r.retcode and g.newton_iters == r.newton_iters, (g.retcode, r.retcode, s.N)
        if r.retcode == 0:
            assert np.max(np.abs(g.u - r.u) / np.maximum(1.0, np.abs(r.u))) <= 1e-9, s.N
            assert np.max(np.abs(g.stages - r.stages)) <= 1e-9 * max(1.0, np.max(np.abs(r.stages))), s.N


@pytest.mark.parametrize("stages", [3, 7], ids=["plain", "general"])
@pytest.mark.parametrize("M,code", [(1, 103), (1, 107), (2, 102), (2, 103), (2, 105), (2, 204), (2, 303), (2, 107),
                                    (3, 103), (3, 204), (4, 102), (4, 103), (6, 102), (6, 103)])
def test_stiff_expanded(M, code, stages):
    print("firk exchanges", M, code, stages, flush=True)
    sys.stdout.flush()
    specs = [_stiff(M, n, k2) for n in SIZES for k2 in (40.0, 4000.0)]
    if M == 2:
        specs += [cases.bratu(1.0, N=n) for n in SIZES]
    _check(code, specs, stages, [True] * len(specs))


@pytest.mark.parametrize("M,code", [(1, 1103), (2, 1102), (2, 1103), (2, 1105), (2, 1107), (3, 1103), (4, 1103),
                                    (6, 1102), (6, 1103)])
def test_stiff_nested(M, code):
    print("firk exchanges nested", M, code, flush=True)
    specs = [_stiff(M, n, k2) for n in SIZES for k2 in (40.0, 4000.0)]
    if M == 2:
        specs += [cases.bratu(1.0, N=n) for n in SIZES]
    _check(code, specs, 3, [True] * len(specs))


@pytest.mark.parametrize("code", [1103, 1105, 1107])
def test_nested_dense_output_of_mixed_families(code):
    print("firk nested dense output, mixed", code, flush=True)
    rng = np.random.default_rng(code)
    pen = bvp.extract(bvp.TwoPointBVProblem(bvp.PendulumFunction(), ([(0, 0.2)], [(0, -0.1)]), [0.0, 0.0], (0.0, 1.0),
                                            [9.81]), dt=0.1)
    specs = [cases.random_state(s, rng, 0.2) for s in
             (cases.bratu(1.0, N=5), pen, cases.singpert(0.1, N=6), cases.linear([[0, 1], [-2, 0.1]], c=0.2, bc=(
                 [(0, 1.0)], [(0, 0.0)]), tspan=(0.0, 1.0), dt=0.2), cases.bratu(2.0, N=9))]
    ts = [rng.uniform(s.t0, s.t1, 5) for s in specs]
    got = _lib.firk_interpolate(_lib.context(0), code, specs, ts)
    for s, t, (u, du) in zip(specs, ts, got):
        ru, rdu = O.firk_interpolate(code, s, t)
        assert np.max(np.abs(u - ru)) <= 1e-11 * max(1.0, np.max(np.abs(ru)))
        assert np.max(np.abs(du - rdu)) <= 1e-9 * max(1.0, np.max(np.abs(rdu)))
