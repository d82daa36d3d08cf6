"""Plans, networks and contexts that are not each other's: a network of one context attached to a
plan of another and destroyed while the plan runs, and a plan run on another context's stream
and destroyed there.  Memory that the contexts keep between calls must not be handed on while
the other stream still reads it: results bit for bit those of one context."""
import sys

import numpy as np
import pytest

from boundaryvaluediffeq_amd import _abi, _lib, synthetic

pytestmark = pytest.mark.gpu


def _specs(n, seed):
    return synthetic.bratu_ab_batch(n, seed=seed, ab=(-0.3, 0.3), lam=(0.1, 2.0), Nrange=(64, 300))[0]


def _opts():
    o = _abi.default_opts(4)
    o.adaptive = 0
    o.max_num_subintervals = 300
    return o


def _solve(ctx, specs, net=None):
    b = _lib.Batch(ctx, _opts(), specs)
    b.set_graph(False)
    if net is not None:
        b.set_warm_start(net)
    b.run()
    b.sync()
    r = b.results()
    b.close()
    return r


def _same(got, want):
    for g, w in zip(got, want):
        assert g.retcode == w.retcode and np.array_equal(g.t, w.t) and np.array_equal(g.u, w.u)


@pytest.mark.parametrize("n", [3, 2000])
def test_network_of_another_context(n):
    print("network of another context", n, flush=True)
    sys.stdout.flush()
    a, b = _lib.Context(0), _lib.Context(0)
    specs = _specs(n, 5)
    own = _lib.MLP(a, seed=4)
    want = _solve(a, specs, own)
    plan = _lib.Batch(a, _opts(), specs)
    plan.set_graph(False)
    for _ in range(3):
        net = _lib.MLP(b, seed=4)
        plan.set_warm_start(net)
        plan.run()
        plan.set_warm_start(None)
        net.close()
        other = _lib.MLP(b, seed=77)  # would take the network's memory from a pool
        other.predict(np.ones((100, 4)))
        plan.sync()
        _same(plan.results(), want)
        other.close()
    plan.close()


@pytest.mark.parametrize("warm", [False, True])
def test_plan_on_another_stream(warm):
    print("plan on another stream", warm, flush=True)
    a, b = _lib.Context(0), _lib.Context(0)
    specs, others = _specs(3000, 6), _specs(3000, 7)
    net = _lib.MLP(a, seed=3) if warm else None
    want, want_others = _solve(a, specs, net), _solve(a, others)
    for _ in range(3):
        plan = _lib.Batch(a, _opts(), specs)
        plan.set_graph(False)
        if warm:
            plan.set_warm_start(net)
        b.call("bvp_batch_run", b.handle, plan._h)
        b.call("bvp_batch_sync", b.handle, plan._h, _lib.C.byref(_lib.C.c_float()))
        _same(plan.results(), want)
        b.call("bvp_batch_run", b.handle, plan._h)
        plan.close()  # with the run in flight
        _same(_solve(a, others), want_others)
