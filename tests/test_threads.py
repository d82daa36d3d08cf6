"""Several Python threads on one context: its calls take turns.  A C context serves one host
thread at a time (include/bvp_mirk.h), and the Python layer hands the same default context to
every caller."""
import ctypes as C
import sys
import threading
import time

import numpy as np
import pytest

from boundaryvaluediffeq_amd import _abi, _lib
import cases


class FakeLib:
    """Stands in for the library: every entry notes how many calls are inside at once."""

    def __init__(self):
        self.inside = self.most = self.calls = 0
        self.mu = threading.Lock()

    def __getattr__(self, name):
        def entry(*args):
            if name.endswith("_create"):
                args[-1]._obj.value = 1
            if name in ("bvp_ctx_create", "bvp_ctx_destroy"):
                return 0
            with self.mu:
                self.inside += 1
                self.calls += 1
                self.most = max(self.most, self.inside)
            time.sleep(0.002)  # the interpreter lock is free in a library call
            with self.mu:
                self.inside -= 1
            return None if name.endswith("_destroy") else 0
        return entry


def _in_threads(fns):
    errors = []

    def guard(fn):
        try:
            fn()
        except BaseException as e:  # reported in the main thread
            errors.append(e)
    threads = [threading.Thread(target=guard, args=(f,)) for f in fns]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors


def test_calls_of_a_context_take_turns(monkeypatch):
    fake = FakeLib()
    monkeypatch.setattr(_lib, "_lib", fake)
    ctx = _lib.Context(0)
    o = _abi.default_opts(4)
    o.max_num_subintervals = 16
    specs = [cases.bratu(1.0, N=8)]

    def work():
        b = _lib.Batch(ctx, o, specs)
        net = _lib.MLP(ctx)
        for _ in range(3):
            _lib.solve_batch(ctx, o, specs)
            _lib.interpolate(ctx, 4, specs, [[0.5]])
            b.run()
            b.sync()
            b.results()
            net.predict(np.zeros((2, 4)))
        net.close()
        b.close()
    _in_threads([work] * 4)
    assert fake.most == 1 and fake.calls == 4 * (4 + 3 * 6)
    ctx.close()


def test_contexts_do_not_wait_for_each_other(monkeypatch):
    fake = FakeLib()
    monkeypatch.setattr(_lib, "_lib", fake)
    meet = threading.Barrier(2, timeout=30)
    fake.bvp_mirk_residual = lambda *a: meet.wait() * 0  # passes only with both threads inside
    _in_threads([lambda c=_lib.Context(0): c.call("bvp_mirk_residual", c.handle) for _ in range(2)])


def test_one_default_context_per_device(monkeypatch):
    fake = FakeLib()
    monkeypatch.setattr(_lib, "_lib", fake)
    monkeypatch.setattr(_lib, "_ctx", {})
    fake.bvp_ctx_create = lambda *a: time.sleep(0.01) or 0
    got = []
    _in_threads([lambda: got.append(_lib.context(0))] * 8)
    assert all(c is got[0] for c in got)


def test_an_error_raises_with_its_text(monkeypatch):
    fake = FakeLib()
    fake.bvp_batch_run = lambda *a: _abi.EINVAL
    fake.bvp_last_error = lambda h: b"the text"
    monkeypatch.setattr(_lib, "_lib", fake)
    ctx = _lib.Context(0)
    with pytest.raises(_lib.BVPError, match=r"batch_run failed \(-?\d+\): the text"):
        ctx.call("bvp_batch_run", ctx.handle, C.c_void_p())


@pytest.mark.gpu
def test_threads_get_their_own_solutions():
    """Different batches (results that fit the staging area and results that span several
    chunks, MIRK and FIRK, dense output) solved by four threads on the default context: bit
    for bit what one thread gets."""
    print("threads", flush=True)
    sys.stdout.flush()
    ctx = _lib.context(0)
    jobs = []
    for k, (method, n, N) in enumerate([(4, 40, 60), (4, 1500, 500), (103, 300, 130), (6, 3, 200)]):
        o = _abi.default_opts(method)
        o.adaptive = 0
        specs = [cases.bratu(0.5 + 0.3 * k + 1.0 * i / n, N=N + i % 3) for i in range(n)]
        jobs.append((o, specs, _lib.solve_batch(ctx, o, specs)))
    ts = [np.linspace(0, 1, 11)]

    def work(o, specs, want):
        for _ in range(6):
            got = _lib.solve_batch(_lib.context(0), o, specs)
            for g, w in zip(got, want):
                assert g.retcode == w.retcode == 0
                assert np.array_equal(g.t, w.t) and np.array_equal(g.u, w.u)
            if o.method < 100:
                s = specs[0].with_state(got[0].t, got[0].u)
                (u, _), = _lib.interpolate(_lib.context(0), o.method, [s], ts)
                assert abs(u[0][0]) <= 1e-9 and u[5][0] > 0.05
    _in_threads([lambda j=j: work(*j) for j in jobs])
