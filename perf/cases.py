"""Workloads of the solver library as a user's program calls it, for timing and comparison.

Each case is a dict of plain values; ``prepare`` builds what a program has in hand before
the call (problems, plans, networks, result buffers), ``run`` makes one pass through the
public entry points and returns its whole output, ``exact`` gives the same output in
64 bits without the library: the discrete collocation solution on the same mesh (Newton's
method on the collocation equations, written here for each family), the problem's own
solution where the mesh is the solver's choice, or the network in float64.
"""
import ctypes
from fractions import Fraction
import math

import numpy as np
import torch

from __graft_entry__ import load_package

bvp = load_package()
from boundaryvaluediffeq_amd import _abi, _lib  # noqa: E402
from boundaryvaluediffeq_amd.problems import InstanceSpec, uniform_mesh  # noqa: E402

_dp = ctypes.POINTER(ctypes.c_double)


def listed():
    return [
        # one small problem: the README's pendulum, solved and evaluated at 33 times
        dict(name="pendulum", kind="pendulum", g=9.81, dt=0.05),
        # a parameter study through EnsembleProblem: 64 trajectories of a 4-component system
        dict(name="ensemble_m4_mirk6", kind="ensemble", M=4, method=6, n=64, N=150),
        # the batched headline: uneven uniform meshes, learned guess, FP32 records, one plan
        dict(name="bratu_plan", kind="bratu", n=8192, lo=96, hi=1024, warm=True, mixed=True),
        # adaptive refinement of boundary and interior layers from a coarse mesh, dense output
        dict(name="singpert_adaptive", kind="singpert", n=512, N0=32, eps_lo=1e-3, eps_hi=1e-1),
        # the reference's Swirling Flow III system (six components) over a range of viscosities
        dict(name="swirl_m6", kind="swirl", n=48, method=4, dt=0.01),
        # one large system, where only one problem's own parallelism is there
        dict(name="lintanh32_one", kind="lintanh", M=32, method=6, n=1, lo=301, hi=301, mixed=True),
        # a batch of large systems with uneven meshes
        dict(name="lintanh32_batch", kind="lintanh", M=32, method=6, n=64, lo=272, hi=720, mixed=True),
        # mid-size systems with FP64 factors
        dict(name="lintanh16_fp64", kind="lintanh", M=16, method=4, n=200, lo=200, hi=600, mixed=False),
        # fully implicit collocation, expanded system, five stages
        dict(name="radau5_batch", kind="firk", family="radau", s=5, nested=False, n=2048, lo=96, hi=1024),
        # fully implicit collocation with inner stage solves, three stages
        dict(name="radau3_nested", kind="firk", family="radau", s=3, nested=True, n=4096, lo=192, hi=1024),
        # the warm-start network: training from given weights
        dict(name="mlp_train", kind="mlp_train", n=65536, batch=8192, epochs=4),
        # the warm-start network: evaluation of many points
        dict(name="mlp_predict", kind="mlp_predict", n=262144),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["pendulum", "ensemble", "bratu", "singpert", "swirl", "lintanh", "lintanh", "firk", "firk",
                       "mlp_train", "mlp_predict"])
    if kind == "pendulum":
        return dict(kind=kind, g=round(rng.uniform(5.0, 12.0), 3), dt=round(rng.uniform(0.02, 0.06), 4))
    if kind == "ensemble":
        return dict(kind=kind, M=rng.choice([1, 2, 3, 4]), method=rng.choice([4, 6]), n=_log(rng, 1, 64),
                    N=rng.randint(100, 170))
    if kind == "bratu":
        lo = rng.randint(96, 400)
        return dict(kind=kind, n=_log(rng, 64, 8192), lo=lo, hi=rng.randint(lo, 1024), warm=rng.random() < 0.5,
                    mixed=rng.random() < 0.5)
    if kind == "singpert":
        return dict(kind=kind, n=_log(rng, 16, 512), N0=rng.randint(24, 64), eps_lo=1e-3, eps_hi=1e-1)
    if kind == "swirl":
        return dict(kind=kind, n=_log(rng, 1, 48), method=rng.choice([4, 6]), dt=round(rng.uniform(0.008, 0.015), 4))
    if kind == "lintanh":
        M = rng.choice([8, 16, 32])
        lo = rng.randint(272, 400)
        return dict(kind=kind, M=M, method=6 if M == 32 else rng.choice([4, 6]), n=_log(rng, 1, 64 if M == 32 else 200),
                    lo=lo, hi=rng.randint(lo, 700), mixed=M == 32 or rng.random() < 0.5)
    if kind == "firk":
        fam = rng.choice(["radau", "lobatto_a"])
        s = rng.choice([3, 5]) if fam == "radau" else rng.choice([4, 5])
        lo = rng.randint(192, 400)
        return dict(kind=kind, family=fam, s=s, nested=rng.random() < 0.5, n=_log(rng, 16, 2048), lo=lo,
                    hi=rng.randint(lo, 1024))
    if kind == "mlp_train":
        batch = 64 * _log(rng, 4, 128)
        return dict(kind=kind, n=batch * rng.randint(2, 8) + rng.randint(0, 63), batch=batch, epochs=rng.randint(1, 4))
    return dict(kind=kind, n=_log(rng, 1, 262144))


# ------------------------------------------------------------------ problems of each kind
def _rng(seed, salt):
    return np.random.default_rng([int(seed) & 0x7FFFFFFF, salt])


def _pendulum(case):
    return bvp.BVProblem(bvp.PendulumFunction(), [(math.pi / 4, 0, -math.pi / 2), (math.pi / 2, 0, math.pi / 2)],
                         [math.pi / 2, math.pi / 2], (0.0, math.pi / 2), [case["g"]])


def _pendulum_times(seed):
    return np.sort(_rng(seed, 1).uniform(0.0, math.pi / 2, 33))


def _linear_system(rng, M, spread):
    """A = Q diag(mu) Q^T with half of the rates decaying and half growing, and M boundary values."""
    Q, R = np.linalg.qr(rng.standard_normal((M, M)))
    Q = Q * np.sign(np.diag(R))
    half = M // 2
    mags = np.logspace(math.log10(spread[0]), math.log10(spread[1]), max(half, M - half))
    mu = np.concatenate([-mags[:M - half], mags[:half]])
    return Q, mu, (Q * mu) @ Q.T, rng.standard_normal(M)


def _spread(M):
    return (0.5, 50.0) if M == 32 else ((0.5, 20.0) if M >= 8 else (0.5, 5.0))


def _sizes(case):
    """Intervals per instance, uniform on lo..hi: part of the case, the same for every seed."""
    return _rng(case["lo"] * 4099 + case["hi"], 2).integers(case["lo"], case["hi"] + 1, case["n"])


def _lintanh_data(case, seed):
    M = case["M"]
    return [_linear_system(np.random.default_rng([int(seed) & 0x7FFFFFFF, 3, i]), M, _spread(M))
            for i in range(case["n"])]


def _lintanh_specs(case, seed):
    M = case["M"]
    La = M - M // 2
    bc_t = np.concatenate([np.zeros(La), np.ones(M - La)])
    specs = []
    for (Q, mu, A, bcv), N in zip(_lintanh_data(case, seed), _sizes(case)):
        specs.append(InstanceSpec(_abi.FAMILY_LINEAR_TANH, M, 0.0, 1.0, np.concatenate([[0.1], A.reshape(-1)]),
                                  _abi.BC_TWO_POINT, bc_t, np.arange(M, dtype=np.int32), bcv, int(N), None, None,
                                  np.zeros(M)))
    return specs


def _bratu_data(case, seed):
    return _rng(seed, 4).uniform(0.1, 3.4, case["n"]), _sizes(case)


def _bratu_specs(case, seed):
    lam, N = _bratu_data(case, seed)
    return [InstanceSpec(_abi.FAMILY_BRATU, 2, 0.0, 1.0, [l], _abi.BC_TWO_POINT, [0.0, 1.0], [0, 0], [0.0, 0.0],
                         int(k), None, None, np.zeros(2)) for l, k in zip(lam, N)]


def _singpert_eps(case, seed):
    r = _rng(seed, 5)
    return np.exp(r.uniform(math.log(case["eps_lo"]), math.log(case["eps_hi"]), case["n"]))


_SINGPERT_T = np.linspace(-1.0, 1.0, 33)


def _swirl_eps(case, seed):
    return np.exp(_rng(seed, 6).uniform(math.log(2e-2), math.log(2e-1), case["n"]))


def _swirl_problem(eps):
    bc = [(0.0, 0, -1.0), (0.0, 2, 0.0), (0.0, 3, 0.0), (1.0, 0, 1.0), (1.0, 2, 0.0), (1.0, 3, 0.0)]
    return bvp.BVProblem(bvp.SwirlFunction(), bc, [0.0] * 6, (0.0, 1.0), [eps])


def _firk_code(case):
    code = (_abi.RADAU_IIA if case["family"] == "radau" else _abi.LOBATTO_IIIA)(case["s"])
    return code + (_abi.FIRK_NESTED if case["nested"] else 0)


# ------------------------------------------------------------------ the warm-start network
_SHAPES = [(4, 256), (256,), (256, 256), (256,), (256, 256), (256,), (256, 2), (2,)]
_MLP_PARAMS = sum(int(np.prod(s)) for s in _SHAPES)


def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _unpack(w):
    out, o = [], 0
    for s in _SHAPES:
        k = int(np.prod(s))
        out.append(w[o:o + k].reshape(s))
        o += k
    return out


def _init_params(r):
    parts = []
    for s in _SHAPES:
        if len(s) == 2:
            b = math.sqrt(6.0 / (s[0] + s[1]))
            parts.append(r.uniform(-b, b, s).reshape(-1))
        else:
            parts.append(np.zeros(s))
    return np.concatenate(parts).astype(np.float32)


def _bratu_samples(r, n):
    """Points (lambda, a = 0, b = 0, t) and the lower-branch solution (u, u') there (float32)."""
    lam, t = r.uniform(0.1, 3.4, n), r.uniform(0.0, 1.0, n)
    th = np.sqrt(2 * lam)
    for _ in range(300):
        th = np.sqrt(2 * lam) * np.cosh(th / 4)
    u = -2 * np.log(np.cosh((t - 0.5) * th / 2) / np.cosh(th / 4))
    du = -th * np.tanh((t - 0.5) * th / 2)
    z = np.zeros(n)
    return np.stack([lam, z, z, t], 1).astype(np.float32), np.stack([u, du], 1).astype(np.float32)


def _norms(x, y):
    sx = x.std(0).astype(np.float64)
    sx[sx == 0] = 1.0
    sy = y.std(0).astype(np.float64)
    return (x.mean(0).astype(np.float32), (1.0 / sx).astype(np.float32), y.mean(0).astype(np.float32),
            sy.astype(np.float32))


def _forward(P, x):
    h = torch.tanh(x @ P[0] + P[1])
    h = torch.tanh(h @ P[2] + P[3])
    h = torch.tanh(h @ P[4] + P[5])
    return h @ P[6] + P[7]


def _fitted_net(seed):
    """(weights, normalisation) of a network fitted to the Bratu family with torch, as a program
    keeps them from an earlier training."""
    r = _rng(seed, 7)
    x, y = _bratu_samples(r, 16384)
    nrm = _norms(x, y)
    d = _dev()
    w = torch.tensor(_init_params(r), device=d, requires_grad=True)
    xt = (torch.tensor(x, device=d) - torch.tensor(nrm[0], device=d)) * torch.tensor(nrm[1], device=d)
    yt = (torch.tensor(y, device=d) - torch.tensor(nrm[2], device=d)) / torch.tensor(nrm[3], device=d)
    opt = torch.optim.Adam([w], lr=2e-3)
    steps = 300
    sched = torch.optim.lr_scheduler.CosineAnnealingLR(opt, steps, 2e-5)
    for k in range(steps):
        s = slice((k % 8) * 2048, (k % 8 + 1) * 2048)
        loss = (_forward(_unpack(w), xt[s]) - yt[s]).square().mean()
        opt.zero_grad()
        loss.backward()
        opt.step()
        sched.step()
    return w.detach().cpu().numpy(), nrm


# ------------------------------------------------------------------ prepare and run
def _result_buffers(specs, stages=0):
    """bvp_result rows whose mesh, solution and stage arrays lie back to back in caller buffers
    with room for twice the initial mesh."""
    res = (_abi.Result * len(specs))()
    cap = np.array([2 * s.N + 1 for s in specs], dtype=np.int64)
    off = np.concatenate([[0], np.cumsum(cap)])
    M = specs[0].M
    t, u = np.zeros(off[-1]), np.zeros(off[-1] * M)
    k = np.zeros(off[-1] * stages * M) if stages else None
    for i in range(len(specs)):
        res[i].capacity = int(cap[i])
        res[i].mesh = ctypes.cast(t.ctypes.data + int(off[i]) * 8, _dp)
        res[i].u = ctypes.cast(u.ctypes.data + int(off[i]) * M * 8, _dp)
        if stages:
            res[i].stages = ctypes.cast(k.ctypes.data + int(off[i]) * stages * M * 8, _dp)
    return dict(res=res, t=t, u=u, k=k, off=off)


def _plan(specs, opts, stages=0):
    ctx = _lib.context(0)
    st = dict(ctx=ctx, plan=_lib.Batch(ctx, opts, specs), specs=specs)
    st.update(_result_buffers(specs, stages))
    return st


def _run_plan(st):
    """One pass of a plan: solve, wait, results into the caller's buffers (C ABI)."""
    st["plan"].run()
    st["plan"].sync()
    st["ctx"].check(_lib.lib().bvp_batch_results(st["ctx"].handle, st["plan"]._h, st["res"]), "batch_results")
    out = dict(retcode=np.array([r.retcode for r in st["res"]], dtype=np.int32),
               N=np.array([r.N_final for r in st["res"]], dtype=np.int32), t=st["t"], u=st["u"])
    if st["k"] is not None:
        out["stages"] = st["k"]
    return out


def prepare(case, seed):
    kind = case["kind"]
    if kind == "pendulum":
        return dict(kind=kind, prob=_pendulum(case), alg=bvp.MIRK4(), dt=case["dt"], ts=_pendulum_times(seed))
    if kind == "ensemble":
        M, n = case["M"], case["n"]
        La = M - M // 2
        data = [_linear_system(np.random.default_rng([int(seed) & 0x7FFFFFFF, 8, i]), M, _spread(M)) for i in range(n)]
        probs = [bvp.TwoPointBVProblem(bvp.LinearTanhFunction(M), ([(c, b[c]) for c in range(La)],
                                                                   [(c, b[c]) for c in range(La, M)]),
                                       [0.0] * M, (0.0, 1.0), np.concatenate([[0.1], A.reshape(-1)]))
                 for _, _, A, b in data]
        ens = bvp.EnsembleProblem(probs[0], prob_func=lambda p, i, rep: probs[i - 1])
        return dict(kind=kind, ens=ens, alg=bvp.MIRK6() if case["method"] == 6 else bvp.MIRK4(), n=n,
                    dt=1.0 / case["N"])
    if kind == "bratu":
        o = _abi.default_opts(4)
        o.abstol, o.newton_abstol = 1e-8, 1e-12
        if case["mixed"]:
            o.precision = _abi.PREC_FP32_REFINE64
        st = _plan(_bratu_specs(case, seed), o)
        if case["warm"]:
            w, nrm = _fitted_net(seed)
            net = _lib.MLP(st["ctx"], seed=1)
            net.set_normalization(*nrm)
            net.set_params(w)
            st["plan"].set_warm_start(net, _abi.FEAT_PARAM, anchors=4)
        return dict(st, kind=kind)
    if kind == "singpert":
        o = _abi.default_opts(4)
        o.newton_abstol = 1e-9
        specs = [InstanceSpec(_abi.FAMILY_SINGPERT, 2, -1.0, 1.0, [e], _abi.BC_TWO_POINT, [-1.0, 1.0], [0, 0],
                              [1.0, 2.0], case["N0"], None, None, np.zeros(2)) for e in _singpert_eps(case, seed)]
        return dict(kind=kind, ctx=_lib.context(0), opts=o, specs=specs)
    if kind == "swirl":
        o = _abi.default_opts(case["method"])
        o.abstol, o.newton_abstol = 1e-4, 1e-10
        specs = [bvp.extract(_swirl_problem(e), dt=case["dt"]) for e in _swirl_eps(case, seed)]
        return dict(kind=kind, ctx=_lib.context(0), opts=o, specs=specs)
    if kind == "lintanh":
        o = _abi.default_opts(case["method"])
        o.abstol = 1e-6 if case["method"] == 6 else 1e-4
        o.newton_abstol = 1e-11
        if case["mixed"]:
            o.precision, o.refine_iters = _abi.PREC_FP32_REFINE64, 2
        return dict(_plan(_lintanh_specs(case, seed), o), kind=kind)
    if kind == "firk":
        o = _abi.default_opts(_firk_code(case))
        o.abstol, o.newton_abstol = 1e-6, 1e-12
        o.nlsolve_stages = _abi.STAGE_NEWTON | _abi.STAGE_BACKTRACKING
        # the expanded form's dense output needs the stages of the solution, the nested one's does not
        return dict(_plan(_bratu_specs(case, seed), o, 0 if case["nested"] else case["s"]), kind=kind)
    r = _rng(seed, 9)
    if kind == "mlp_train":
        x, y = _bratu_samples(r, case["n"])
        net = _lib.MLP(_lib.context(0), seed=1)
        net.set_normalization(*_norms(x, y))
        return dict(kind=kind, net=net, w0=_init_params(r), x=x, y=y, epochs=case["epochs"], batch=case["batch"])
    x, y = _bratu_samples(r, max(case["n"], 2))
    net = _lib.MLP(_lib.context(0), seed=1)
    net.set_normalization(*_norms(*_bratu_samples(r, 4096)))
    net.set_params(_init_params(r))
    return dict(kind=kind, net=net, x=x[:case["n"]])


def run(st):
    kind = st["kind"]
    if kind == "pendulum":
        sol = bvp.solve(st["prob"], st["alg"], dt=st["dt"], abstol=1e-6)
        return dict(u=sol(st["ts"]), nodes=np.asarray(sol.u), t=sol.t)
    if kind == "ensemble":
        sols = bvp.solve(st["ens"], st["alg"], dt=st["dt"], abstol=1e-6, trajectories=st["n"],
                         nlsolve_kwargs={"abstol": 1e-11})
        return dict(t=np.concatenate([s.t for s in sols]), u=np.concatenate([np.asarray(s.u) for s in sols]))
    if kind == "singpert":
        sols = _lib.solve_batch(st["ctx"], st["opts"], st["specs"])
        at = [s.with_state(r.t, r.u) for s, r in zip(st["specs"], sols)]
        vals = _lib.interpolate(st["ctx"], st["opts"].method, at, [_SINGPERT_T] * len(at), derivative=False)
        return dict(u=np.stack([v for v, _ in vals]))
    if kind == "swirl":
        sols = _lib.solve_batch(st["ctx"], st["opts"], st["specs"])
        return dict(t=np.concatenate([r.t for r in sols]), u=np.concatenate([r.u for r in sols]))
    if kind in ("bratu", "lintanh", "firk"):
        return _run_plan(st)
    if kind == "mlp_train":
        st["net"].set_params(st["w0"])
        loss, _ = st["net"].train(st["x"], st["y"], epochs=st["epochs"], batch=st["batch"], lr=1e-3, lr_min=2e-5,
                                  warmup=8, seed=7)
        return dict(params=st["net"].params(), loss=loss)
    return dict(y=st["net"].predict(st["x"]))


# ------------------------------------------------------------------ work and tolerances
def _mean_n(case):
    return (case["lo"] + case["hi"]) / 2.0


def work(case):
    """Bytes a pass must read and write (inputs once, solution once) and the operations of two
    Newton steps (residual, blocks, elimination) where the path is an elimination."""
    kind = case["kind"]
    if kind == "pendulum":
        N, M, n = math.pi / 2 / case["dt"], 2, 1
    elif kind == "ensemble":
        N, M, n = case["N"], case["M"], case["n"]
    elif kind == "singpert":
        N, M, n = 4.0 * case["N0"], 2, case["n"]
    elif kind == "swirl":
        N, M, n = 1.0 / case["dt"], 6, case["n"]
    elif kind in ("bratu", "lintanh", "firk"):
        N, M, n = _mean_n(case), case.get("M", 2), case["n"]
    elif kind == "mlp_train":
        return dict(bytes=24.0 * case["n"] + 8.0 * _MLP_PARAMS,
                    flops=6.0 * _MLP_PARAMS * case["epochs"] * (case["n"] // case["batch"]) * case["batch"])
    else:
        return dict(bytes=24.0 * case["n"] + 4.0 * _MLP_PARAMS, flops=2.0 * _MLP_PARAMS * case["n"])
    s = case["s"] if kind == "firk" else (5 if case.get("method") == 6 else 3)
    nodes = n * N
    per = 2.0 * (2 * s * M * M + 8.0 / 3 * M ** 3 + 8 * M * M + 2 * s * M ** 3)
    if kind == "firk":
        per = 2.0 * (2.0 / 3 * (s * M) ** 3 + 2 * (s * M) ** 2 * (M + 1) + 8 * M ** 3)
    size = 8.0 * (2 * M + 1 + (s * M if kind == "firk" and not case["nested"] else 0))
    return dict(bytes=nodes * size, flops=nodes * per)


def tolerance(case):
    kind = case["kind"]
    if kind == "singpert":
        # the redistributed nodes follow the rounding of the defects: one unit in the last place
        # of abstol moves the values by up to 2.5e-10 (24 problems)
        return {"rel": 4e-9, "max": 4e-8}
    if kind == "pendulum":
        return {"rel": 1e-8, "max": 1e-7}
    if kind == "mlp_train":
        # BF16 weights and activations: 4.2e-4 from the unrounded schedule after 32 steps
        return {"rel": 2e-3}
    if kind == "mlp_predict":
        # BF16 weights and activations: 1.7e-3 to 3.9e-3 from the unrounded network
        return {"rel": 1e-2}
    # Newton stops within 2e-10 (M = 2, 6) or 4e-12 of the discrete solution, and two correct
    # solves stop at different corrections
    return {"rel": 1e-9, "max": 1e-8}


# ------------------------------------------------------------------ 64-bit solutions without the library
def _mirk_tableau(method):
    if method == 4:
        v = [0.0, 1.0, 0.5]
        b = [1 / 6, 1 / 6, 2 / 3]
        x = [[0, 0, 0], [0, 0, 0], [1 / 8, -1 / 8, 0]]
        return [0.0, 1.0, 0.5], v, b, x
    c = [0.0, 1.0, 0.25, 0.75, 0.5]
    v = [0.0, 1.0, 5 / 32, 27 / 32, 0.5]
    b = [7 / 90, 7 / 90, 16 / 45, 16 / 45, 2 / 15]
    x = [[0] * 5, [0] * 5, [9 / 64, -3 / 64, 0, 0, 0], [3 / 64, -9 / 64, 0, 0, 0], [-5 / 24, 5 / 24, 2 / 3, -2 / 3, 0]]
    return c, v, b, x


def _intervals(dt):
    """Intervals of a uniform mesh of [0, 1] for a step dt: the exact quotient, rounded up."""
    return math.ceil(Fraction(1.0) / Fraction(dt))


def _mm(A, B):
    return (A.unsqueeze(-1) * B.unsqueeze(-3)).sum(-2)


def _mirk_blocks(f, jac, method, h, ya, yb):
    """Phi, S = dPhi/dya, R = dPhi/dyb of every interval; h [...], ya, yb [..., M]."""
    _, v, b, x = _mirk_tableau(method)
    h1, h2 = h.unsqueeze(-1), h.unsqueeze(-1).unsqueeze(-1)
    eye = torch.eye(ya.shape[-1], dtype=ya.dtype, device=ya.device)
    K, Da, Db = [], [], []
    for r in range(len(b)):
        y = (1 - v[r]) * ya + v[r] * yb
        a_, b_ = (1 - v[r]) * eye, v[r] * eye
        for j in range(r):
            if x[r][j]:
                y = y + h1 * x[r][j] * K[j]
                a_ = a_ + h2 * x[r][j] * Da[j]
                b_ = b_ + h2 * x[r][j] * Db[j]
        J = jac(y)
        K.append(f(y))
        Da.append(_mm(J, a_.expand_as(J)))
        Db.append(_mm(J, b_.expand_as(J)))
    phi = yb - ya - h1 * sum(b[r] * K[r] for r in range(len(b)))
    S = -eye - h2 * sum(b[r] * Da[r] for r in range(len(b)))
    R = eye - h2 * sum(b[r] * Db[r] for r in range(len(b)))
    return phi, S, R


def _meshes(Ns, device):
    """Padded uniform meshes [n, max N + 1]; the padding continues past the end with the same step."""
    n, m = len(Ns), int(max(Ns))
    t = np.zeros((n, m + 1))
    for i, N in enumerate(Ns):
        t[i, :N + 1] = uniform_mesh(0.0, 1.0, int(N))
        t[i, N + 1:] = 1.0 + np.arange(1, m - N + 1) / N
    return t, torch.tensor(t, device=device)


def _shoot(T, r, y, Ns):
    """Newton correction d_{k+1} = T_k d_k + r_k with d_0[0] and d_N[0] removing the boundary
    residuals (values 0 at both ends), by superposition; T [n, N, 2, 2]."""
    n, m = T.shape[:2]
    idx = torch.tensor(np.asarray(Ns), device=T.device)
    p = torch.zeros(n, 2, dtype=T.dtype, device=T.device)
    p[:, 0] = -y[:, 0, 0]
    q = torch.zeros_like(p)
    q[:, 1] = 1.0
    ps, qs = [p], [q]
    for k in range(m):
        p = _mm(T[:, k], p.unsqueeze(-1)).squeeze(-1) + r[:, k]
        q = _mm(T[:, k], q.unsqueeze(-1)).squeeze(-1)
        ps.append(p)
        qs.append(q)
    P, Q = torch.stack(ps, 1), torch.stack(qs, 1)
    rows = torch.arange(n, device=T.device)
    a = (-y[rows, idx, 0] - P[rows, idx, 0]) / Q[rows, idx, 0]
    return P + a[:, None, None] * Q


def _pack_exact(Ns, t, u, M, stages=None):
    cap = 2 * np.asarray(Ns, dtype=np.int64) + 1
    off = np.concatenate([[0], np.cumsum(cap)])
    T, U = np.zeros(off[-1]), np.zeros(off[-1] * M)
    K = np.zeros(off[-1] * stages.shape[2] * M) if stages is not None else None
    for i, N in enumerate(Ns):
        T[off[i]:off[i] + N + 1] = t[i, :N + 1]
        U[off[i] * M:(off[i] + N + 1) * M] = u[i, :N + 1].reshape(-1)
        if K is not None:
            w = stages.shape[2] * M
            K[off[i] * w:(off[i] + N) * w] = stages[i, :N].reshape(-1)
    out = dict(retcode=np.zeros(len(Ns), dtype=np.int32), N=np.asarray(Ns, dtype=np.int32), t=T, u=U)
    if K is not None:
        out["stages"] = K
    return out


def _exact_bratu(case, seed):
    lam_, Ns = _bratu_data(case, seed)
    d = _dev()
    t, tt = _meshes(Ns, d)
    h = tt[:, 1:] - tt[:, :-1]
    lam = torch.tensor(lam_, device=d)[:, None]

    def f(y):
        return torch.stack([y[..., 1], -lam * torch.exp(y[..., 0])], -1)

    def jac(y):
        z = torch.zeros_like(y[..., 0])
        return torch.stack([torch.stack([z, z + 1], -1), torch.stack([-lam * torch.exp(y[..., 0]), z], -1)], -2)

    y = torch.zeros(*tt.shape, 2, dtype=torch.float64, device=d)
    for _ in range(9):
        phi, S, R = _mirk_blocks(f, jac, 4, h, y[:, :-1], y[:, 1:])
        Ri = torch.linalg.inv_ex(R)[0] if R.shape[-1] > 2 else _inv2(R)
        y = y + _shoot(-_mm(Ri, S), -_mm(Ri, phi.unsqueeze(-1)).squeeze(-1), y, Ns)
    return _pack_exact(Ns, t, y.cpu().numpy(), 2)


def _inv2(A):
    det = A[..., 0, 0] * A[..., 1, 1] - A[..., 0, 1] * A[..., 1, 0]
    a = torch.stack([torch.stack([A[..., 1, 1], -A[..., 0, 1]], -1),
                     torch.stack([-A[..., 1, 0], A[..., 0, 0]], -1)], -2)
    return a / det[..., None, None]


def _collocation(family, s):
    """Nodes, A and b of Radau IIA or Lobatto IIIA with s stages (integrals of the Lagrange basis)."""
    L = np.polynomial.legendre
    if family == "radau":
        c = (L.legroots([0.0] * (s - 1) + [-1.0, 1.0]) + 1) / 2
    else:
        c = (np.concatenate([[-1.0], np.sort(L.legroots(L.legder([0.0] * (s - 1) + [1.0]))), [1.0]]) + 1) / 2
    c = np.sort(c)
    A, b = np.zeros((s, s)), np.zeros(s)
    for j in range(s):
        p = np.array([1.0])
        for m in range(s):
            if m != j:
                p = np.polymul(p, np.array([1.0, -c[m]]) / (c[j] - c[m]))
        q = np.polyint(p)
        A[:, j] = np.polyval(q, c)
        b[j] = np.polyval(q, 1.0)
    return A, b


def _exact_firk(case, seed):
    lam_, Ns = _bratu_data(case, seed)
    d, s = _dev(), case["s"]
    A_, b_ = _collocation(case["family"], s)
    A, b = torch.tensor(A_, device=d), torch.tensor(b_, device=d)
    t, tt = _meshes(Ns, d)
    h = tt[:, 1:] - tt[:, :-1]
    lam = torch.tensor(lam_, device=d)[:, None, None]
    n, m = h.shape
    y = torch.zeros(n, m + 1, 2, dtype=torch.float64, device=d)
    K = torch.zeros(n, m, s, 2, dtype=torch.float64, device=d)
    hh = h[..., None]
    for _ in range(9):
        # stage unknowns (K1, K2) of an interval: K1 = Y2, K2 = -lam e^{Y1}, Y = y + h A K
        Y1 = y[:, :-1, None, 0] + hh * (K[..., 0] @ A.T)
        Y2 = y[:, :-1, None, 1] + hh * (K[..., 1] @ A.T)
        e = -lam * torch.exp(Y1)
        W = torch.zeros(n, m, 2 * s, 2 * s + 3, dtype=torch.float64, device=d)
        for r in range(s):
            W[..., r, r] = 1.0
            W[..., s + r, s + r] = 1.0
            W[..., r, s:2 * s] -= h[..., None] * A[r]
            W[..., s + r, :s] -= (h * e[..., r])[..., None] * A[r]
            W[..., r, 2 * s] = Y2[..., r] - K[..., r, 0]
            W[..., s + r, 2 * s] = e[..., r] - K[..., r, 1]
            W[..., r, 2 * s + 2] = 1.0
            W[..., s + r, 2 * s + 1] = e[..., r]
        for j in range(2 * s):  # Gauss-Jordan; the pivots stay near 1 (W = I + O(h))
            W[..., j, j + 1:] = W[..., j, j + 1:] / W[..., j, j:j + 1]
            f = W[..., :, j].clone()
            f[..., j] = 0.0
            W[..., :, j + 1:] -= f.unsqueeze(-1) * W[..., j, j + 1:].unsqueeze(-2)
        X = W[..., 2 * s:].reshape(n, m, 2, s, 3)  # component, stage, (rhs, d/dy1, d/dy2)
        cond = (X * b[:, None]).sum(-2)            # component, (rhs, d/dy1, d/dy2)
        T = h[..., None, None] * cond[..., 1:] + torch.eye(2, dtype=torch.float64, device=d)
        phi = y[:, 1:] - y[:, :-1] - hh * (K * b[:, None]).sum(-2)
        dy = _shoot(T, -phi + hh * cond[..., 0], y, Ns)
        K = K + (X[..., 0] + X[..., 1] * dy[:, :-1, None, None, 0] + X[..., 2] * dy[:, :-1, None, None, 1]).transpose(-1, -2)
        y = y + dy
    return _pack_exact(Ns, t, y.cpu().numpy(), 2, None if case["nested"] else K.cpu().numpy())


def _linear_tanh_solution(Q, mu, A, bcv, N, method, c=0.1):
    """The MIRK solution of u' = A u + c tanh(u) on N uniform intervals: fixed-point iteration
    with the modes of u' = A u solved exactly (decaying ones forwards, growing ones backwards)."""
    M = len(mu)
    La = M - M // 2
    _, v, b, x = _mirk_tableau(method)
    t = uniform_mesh(0.0, 1.0, N)
    h = (t[1:] - t[:-1])[:, None]
    mc = mu + c  # tanh'(0) belongs to the linear part

    def blocks(z):  # S and R of the scalar problem u' = mc u
        Ka, Kb = [], []
        for r in range(len(b)):
            a_, b_ = (1 - v[r]) + 0 * z, v[r] + 0 * z
            for j in range(r):
                a_, b_ = a_ + x[r][j] * Ka[j], b_ + x[r][j] * Kb[j]
            Ka.append(z * a_)
            Kb.append(z * b_)
        return -1 - sum(b[r] * Ka[r] for r in range(len(b))), 1 - sum(b[r] * Kb[r] for r in range(len(b)))

    S, R = blocks(h * mc)
    up = mc < 0  # modes carried forwards
    F, G = -S / R, -R / S
    fwd = np.cumprod(np.vstack([np.ones(M), np.where(up, F, 1.0)]), 0)
    bwd = np.cumprod(np.vstack([np.ones(M), np.where(up, 1.0, G)[::-1]]), 0)[::-1]
    hom = np.where(up, fwd, bwd)
    B = np.vstack([Q[:La] * hom[0], Q[La:] * hom[-1]])
    u = np.zeros((N + 1, M))
    last = np.inf
    for it in range(400):
        K = []
        for r in range(len(b)):
            y = (1 - v[r]) * u[:-1] + v[r] * u[1:]
            for j in range(r):
                if x[r][j]:
                    y = y + h * x[r][j] * K[j]
            K.append(y @ A.T + c * np.tanh(y))
        phi = (u[1:] - u[:-1] - h * sum(b[r] * K[r] for r in range(len(b)))) @ Q
        p = np.zeros((N + 1, M))
        for k in range(N):
            p[k + 1, up] = ((-phi[k] - S[k] * p[k]) / R[k])[up]
        for k in range(N - 1, -1, -1):
            p[k, ~up] = ((-phi[k] - R[k] * p[k + 1]) / S[k])[~up]
        res = np.concatenate([bcv[:La] - u[0, :La], bcv[La:] - u[-1, La:]])
        a = np.linalg.solve(B, res - np.concatenate([Q[:La] @ p[0], Q[La:] @ p[-1]]))
        d = (p + hom * a) @ Q.T
        u += d
        size = np.abs(d).max()
        if size < 1e-15 * max(1.0, np.abs(u).max()) or (size < 1e-12 and size >= last):
            break
        last = size
    return t, u


def _exact_swirl(case, seed):
    ts, us = [], []
    for eps in _swirl_eps(case, seed):
        N = _intervals(case["dt"])
        t = uniform_mesh(0.0, 1.0, N)
        h = torch.tensor(t[1:] - t[:-1])

        def f(y):
            return torch.stack([y[..., 1], (y[..., 0] * y[..., 3] - y[..., 2] * y[..., 1]) / eps, y[..., 3], y[..., 4],
                                y[..., 5], (-y[..., 2] * y[..., 5] - y[..., 0] * y[..., 1]) / eps], -1)

        def jac(y):
            J = torch.zeros(*y.shape, 6, dtype=y.dtype)
            J[..., 0, 1] = J[..., 2, 3] = J[..., 3, 4] = J[..., 4, 5] = 1.0
            J[..., 1, 0], J[..., 1, 1] = y[..., 3] / eps, -y[..., 2] / eps
            J[..., 1, 2], J[..., 1, 3] = -y[..., 1] / eps, y[..., 0] / eps
            J[..., 5, 0], J[..., 5, 1] = -y[..., 1] / eps, -y[..., 0] / eps
            J[..., 5, 2], J[..., 5, 5] = -y[..., 5] / eps, -y[..., 2] / eps
            return J

        y = torch.zeros(N + 1, 6, dtype=torch.float64)
        rows, vals = [0, 2, 3, 6 * N, 6 * N + 2, 6 * N + 3], [-1.0, 0.0, 0.0, 1.0, 0.0, 0.0]
        for _ in range(40):
            phi, S, R = _mirk_blocks(f, jac, case["method"], h, y[:-1], y[1:])
            J = np.zeros((6 * (N + 1), 6 * (N + 1)))
            for i, k in enumerate(rows):
                J[i, k] = 1.0
            for k in range(N):
                J[6 + 6 * k:12 + 6 * k, 6 * k:6 * k + 6] = S[k]
                J[6 + 6 * k:12 + 6 * k, 6 * k + 6:6 * k + 12] = R[k]
            F = np.concatenate([y.reshape(-1).numpy()[rows] - vals, phi.reshape(-1).numpy()])
            d = np.linalg.solve(J, -F)
            y = y + torch.tensor(d).reshape(N + 1, 6)
            if np.abs(d).max() < 1e-14:
                break
        ts.append(t)
        us.append(y.numpy())
    return dict(t=np.concatenate(ts), u=np.concatenate(us))


def _exact_pendulum(case, seed):
    """The boundary value problem by shooting from t = pi/4 with classical Runge-Kutta steps."""
    g, ts = case["g"], _pendulum_times(seed)
    mid, end = math.pi / 4, math.pi / 2

    def f(y):
        return np.array([y[1], -g * math.sin(y[0])])

    def go(y, a, b):
        n = max(1, int(math.ceil(abs(b - a) / 2e-3)))
        h = (b - a) / n
        y = np.array(y)
        for _ in range(n):
            k1 = f(y)
            k2 = f(y + h / 2 * k1)
            k3 = f(y + h / 2 * k2)
            k4 = f(y + h * k3)
            y = y + h / 6 * (k1 + 2 * k2 + 2 * k3 + k4)
        return y

    # candidates for the speed at the midpoint; the solution is the one the solver's start leads to
    def miss(w):
        return go([-math.pi / 2, w], mid, end)[0] - math.pi / 2

    ws = np.linspace(-12, 12, 241)
    ms = [miss(w) for w in ws]
    roots = []
    for a, b, fa, fb in zip(ws[:-1], ws[1:], ms[:-1], ms[1:]):
        if fa * fb < 0 and abs(fa - fb) < 4:
            for _ in range(80):
                c = (a + b) / 2
                fc = miss(c)
                if fa * fc <= 0:
                    b = c
                else:
                    a, fa = c, fc
            roots.append((a + b) / 2)
    if len(roots) != 1:
        return None
    w = roots[0]
    out = np.zeros((len(ts), 2))
    y, at = np.array([-math.pi / 2, w]), mid
    for i in np.where(ts >= mid)[0]:
        y = go(y, at, ts[i])
        at = ts[i]
        out[i] = y
    y, at = np.array([-math.pi / 2, w]), mid
    for i in np.where(ts < mid)[0][::-1]:
        y = go(y, at, ts[i])
        at = ts[i]
        out[i] = y
    return dict(u=out, nodes=None, t=None)


def _exact_train(case, seed):
    """The same schedule of Adam steps in float64 without any rounding of weights or activations."""
    r = _rng(seed, 9)
    x, y = _bratu_samples(r, case["n"])
    nrm = [torch.tensor(v, dtype=torch.float64, device=_dev()) for v in _norms(x, y)]
    w = torch.tensor(_init_params(r), dtype=torch.float64, device=_dev(), requires_grad=True)
    xt = (torch.tensor(x, dtype=torch.float64, device=_dev()) - nrm[0]) * nrm[1]
    yt = (torch.tensor(y, dtype=torch.float64, device=_dev()) - nrm[2]) / nrm[3]
    n, batch, mask64 = case["n"], case["batch"], (1 << 64) - 1
    spe = n // batch
    total, warm, lr0, lr1 = spe * case["epochs"], 8, 1e-3, 2e-5
    m = torch.zeros_like(w)
    v = torch.zeros_like(w)
    loss_all = []
    for e in range(case["epochs"]):
        s = 7 ^ 0x6A09E667F3BCC909 ^ ((e + 1) * 0xD1B54A32D192ED03 & mask64)

        def unit():
            nonlocal s
            s = (s + 0x9E3779B97F4A7C15) & mask64
            z = s
            z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & mask64
            z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask64
            z ^= z >> 31
            return (z >> 11) / 9007199254740992.0

        while True:
            a = 1 + int(unit() * float(n - 1))
            if a < n and math.gcd(a, n) == 1:
                break
        c = int(unit() * float(n)) % n
        for k in range(spe):
            i = (a * torch.arange(k * batch, (k + 1) * batch, device=w.device) + c) % n
            loss = 0.5 * (_forward(_unpack(w), xt[i]) - yt[i]).square().sum() / batch
            g, = torch.autograd.grad(loss, w)
            step = e * spe + k
            if step < warm:
                lr = lr0 * (step + 1) / warm
            else:
                lr = lr1 + 0.5 * (lr0 - lr1) * (1 + math.cos(math.pi * min(1.0, (step - warm) / max(1, total - warm))))
            with torch.no_grad():
                m.mul_(0.9).add_(0.1 * g)
                v.mul_(0.999).add_(0.001 * g * g)
                w -= lr * (m / (1 - 0.9 ** (step + 1))) / ((v / (1 - 0.999 ** (step + 1))).sqrt() + 1e-8)
            loss_all.append(float(loss))
    return dict(params=w.detach().cpu().numpy(), loss=np.array(loss_all))


def exact(case, seed):
    kind = case["kind"]
    if kind == "pendulum":
        return _exact_pendulum(case, seed)
    if kind == "ensemble":
        data = [_linear_system(np.random.default_rng([int(seed) & 0x7FFFFFFF, 8, i]), case["M"], _spread(case["M"]))
                for i in range(case["n"])]
        N = _intervals(1.0 / case["N"])
        sols = [_linear_tanh_solution(Q, mu, A, b, N, case["method"]) for Q, mu, A, b in data]
        return dict(t=np.concatenate([t for t, _ in sols]), u=np.concatenate([u for _, u in sols]))
    if kind == "bratu":
        return _exact_bratu(case, seed)
    if kind == "singpert":
        eps = torch.tensor(_singpert_eps(case, seed))[:, None]
        t = torch.tensor(_SINGPERT_T)[None, :]
        root = torch.sqrt(math.pi / (2 * eps))

        def g(t):
            return torch.exp(-t * t / (2 * eps)) + t * root * torch.erf(t / torch.sqrt(2 * eps))

        b = 1.5 / g(torch.ones_like(eps))
        return dict(u=torch.stack([0.5 * t + b * g(t), 0.5 + b * root * torch.erf(t / torch.sqrt(2 * eps))], -1).numpy())
    if kind == "swirl":
        return _exact_swirl(case, seed)
    if kind == "lintanh":
        Ns = _sizes(case)
        if float(np.sum(Ns)) * case["M"] > 1.5e6:
            return None  # the fixed-point iterations would take over 20 seconds
        sols = [_linear_tanh_solution(Q, mu, A, b, int(N), case["method"])
                for (Q, mu, A, b), N in zip(_lintanh_data(case, seed), Ns)]
        m = int(max(Ns))
        t, u = np.zeros((len(Ns), m + 1)), np.zeros((len(Ns), m + 1, case["M"]))
        for i, (ti, ui) in enumerate(sols):
            t[i, :len(ti)], u[i, :len(ti)] = ti, ui
        return _pack_exact(Ns, t, u, case["M"])
    if kind == "firk":
        return _exact_firk(case, seed)
    if kind == "mlp_train":
        return _exact_train(case, seed)
    r = _rng(seed, 9)
    x, _ = _bratu_samples(r, max(case["n"], 2))
    nrm = [torch.tensor(v, dtype=torch.float64) for v in _norms(*_bratu_samples(r, 4096))]
    P = [p.double() for p in _unpack(torch.tensor(_init_params(r)))]
    xn = (torch.tensor(x[:case["n"]], dtype=torch.float64) - nrm[0]) * nrm[1]
    return dict(y=(_forward(P, xn) * nrm[3] + nrm[2]).numpy())
