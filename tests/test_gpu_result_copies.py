"""Results on their way to the host: batches whose solutions fit the small staging area, exceed
it, and span several chunks (with instances cut by a chunk's end), FIRK stages with them, and
rows that are too small; each against the same instance solved alone, bit for bit.  Every
batch runs twice and in a second context, so that it also meets memory that an earlier call
left."""
import ctypes as C
import sys

import numpy as np
import pytest

from boundaryvaluediffeq_amd import _abi, _lib
import cases

pytestmark = pytest.mark.gpu


def _specs(n, N):
    return [cases.bratu(0.5 + 2.0 * (i % 97) / 97, N=N + i % 5) for i in range(n)]


def _opts(method):
    o = _abi.default_opts(method)
    o.adaptive = 0
    return o


@pytest.mark.parametrize("method,n,N", [(4, 1, 5), (4, 9, 40), (4, 300, 220), (4, 2000, 560), (6, 700, 1100),
                                        (103, 9, 40), (103, 900, 400)])
def test_batch_equals_single(method, n, N):
    print("result copies", method, n, N, flush=True)
    sys.stdout.flush()
    specs, o = _specs(n, N), _opts(method)
    pick = sorted({0, 1 % n, n // 3, n // 2, n - 1})
    for ctx in (_lib.context(0), _lib.Context(0)):
        one = {i: _lib.solve_batch(ctx, o, [specs[i]])[0] for i in pick}
        for _ in range(2):
            got = _lib.solve_batch(ctx, o, specs)
            for i in pick:
                g, r = got[i], one[i]
                assert g.retcode == r.retcode == 0 and g.N == r.N == specs[i].N
                assert np.array_equal(g.t, r.t) and np.array_equal(g.u, r.u), i
                if method >= 100:
                    assert np.array_equal(g.stages, r.stages), i
            for g, s in zip(got, specs):
                assert g.u.shape == (s.N + 1, 2) and g.t[0] == 0.0 and g.t[-1] == 1.0


@pytest.mark.parametrize("n,N", [(9, 40), (2000, 560)])
def test_row_too_small(n, N):
    print("result rows too small", n, N, flush=True)
    ctx = _lib.context(0)
    specs, o = _specs(n, N), _opts(4)
    want = _lib.solve_batch(ctx, o, specs)
    from boundaryvaluediffeq_amd.problems import instance_array
    cap = max(s.N for s in specs) + 1
    res, bufs = _lib._result_array(specs, cap)
    res[n // 2].capacity = 3
    rc = _lib.lib().bvp_mirk_solve_batch(ctx.handle, C.byref(o), n, instance_array(specs), res)
    assert rc == _abi.EINVAL
    for i in (0, n // 2 - 1, n // 2 + 1, n - 1):
        assert np.array_equal(bufs[1][i][:2 * (specs[i].N + 1)].reshape(-1, 2), want[i].u)
    assert not bufs[1][n // 2].any() and res[n // 2].N_final == specs[n // 2].N
