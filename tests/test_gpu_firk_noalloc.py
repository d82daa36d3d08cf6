"""FIRK batches that nearly fill the no-allocation scratch: the lines that their areas round up to
(csrc/firk_layout.h) must not refuse what packed areas of the same waves hold, and fewer waves give the
same bits as bvp_mirk_solve_batch.  Small capacities, where a line is many times an instance's
intervals, on both sides of the 32 intervals up to which instances share lines."""
import sys

import numpy as np
import pytest

from boundaryvaluediffeq_amd import _abi, _lib
import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("code,n,cap", [(105, 560, 16), (105, 500, 33), (105, 20, 63), (103, 640, 8), (1105, 560, 16),
                                        (107, 500, 12)])
def test_nearly_full(code, n, cap):
    print("firk no-alloc", code, n, cap, flush=True)
    sys.stdout.flush()
    ctx = _lib.context(0)
    o = _abi.default_opts(code)
    o.adaptive = 0
    o.nlsolve_stages = 3
    o.max_num_subintervals = cap
    o.newton_abstol = 1e-10
    specs = [cases.bratu(0.5 + 2.0 * i / n, N=1 + (i * 7) % cap) for i in range(n)]
    want = _lib.solve_batch(ctx, o, specs)
    for _ in range(2):
        got = _lib.solve_batch_noalloc(ctx, o, specs)
        for g, w, s in zip(got, want, specs):
            assert g.retcode == w.retcode == 0 and g.N == w.N == s.N
            assert np.array_equal(g.u, w.u) and np.array_equal(g.stages, w.stages), s.N
