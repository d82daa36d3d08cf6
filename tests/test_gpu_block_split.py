"""The block kernels' split of an instance over the waves of its workgroup: meshes around
the wave count (fewer intervals than waves, one per wave, one wave with one more, chunks
merged over an odd number of waves) and around the 64 / M intervals a wave holds in the
FP64 stage passes.

Tolerances: as tests/test_gpu_block.py -- residual 1e-12 and Newton correction 1e-9
relative to the largest entry (FP64 factors, or FP32 factors whose three refinement steps
each gain the FP32 factorisation's 3 to 4 digits), defect 1e-9.
"""
import sys

import numpy as np
import pytest

from boundaryvaluediffeq_amd import _abi, _lib
import pyoracle as O
import cases

pytestmark = pytest.mark.gpu

SIZES = (1, 2, 3, 7, 8, 9, 15, 16, 17, 31, 33, 65)


def _specs(M):
    out = []
    for n in SIZES:
        rng = np.random.default_rng(100 * M + n)
        s = cases.linear_tanh_c3(rng, M=M, N=n, spread=(0.5, 20.0))
        s = cases.random_state(s, rng, 0.3)
        out.append(cases.random_mesh(s, rng) if n % 2 else s)
    return out


@pytest.mark.parametrize("M", [8, 16, 32])
@pytest.mark.parametrize("method", [4, 6])
def test_block_split(M, method):
    print("block split", M, method, flush=True)
    sys.stdout.flush()
    ctx = _lib.context(0)
    specs = _specs(M)
    for s, g in zip(specs, _lib.residual(ctx, method, specs)):
        ref = O.residual(method, s)
        assert np.max(np.abs(g - ref)) <= 1e-12 * max(1.0, np.max(np.abs(ref))), s.N
    for s, (err, dn) in zip(specs, _lib.defect(ctx, method, specs)):
        er, dr = O.defect(method, s)
        assert np.max(np.abs(err - er)) <= 1e-9 * max(1.0, np.max(np.abs(er))), s.N
        assert abs(dn - dr) <= 1e-9 * max(1.0, dr), s.N
    modes = [(_abi.PREC_FP32_REFINE64, 3)] + ([(_abi.PREC_FP64, 0)] if M < 32 else [])
    for prec, refine in modes:
        got = _lib.newton_step(ctx, method, specs, precision=prec, refine_iters=refine)
        for s, d in zip(specs, got):
            ref = O.newton_step(method, s)
            err = np.max(np.abs(d - ref)) / max(1.0, np.max(np.abs(ref)))
            assert err <= 1e-9, (s.N, prec, err)


@pytest.mark.parametrize("M,prec,refine", [(8, _abi.PREC_FP64, 0), (16, _abi.PREC_FP64, 0),
                                           (32, _abi.PREC_FP32_REFINE64, 2)])
def test_block_mesh_select_and_transfer(M, prec, refine):
    """Mesh selection and both transfer modes (the in-place chain of the reference mode
    included) against the oracle on meshes that are redistributed."""
    print("block mesh select", M, flush=True)
    ctx = _lib.context(0)
    for mode in (_abi.TRANSFER_REFERENCE, _abi.TRANSFER_CLEAN):
        for n in (5, 24, 40):
            rng = np.random.default_rng(n + M)
            s = cases.linear_tanh_c3(rng, M=M, N=n, spread=(0.5, 20.0))
            st = O.solve(O.opts(4, adaptive=0, newton_abstol=1e-11), s)
            s = s.with_state(st.t, st.u.reshape(-1))
            o = _abi.default_opts(4)
            o.abstol = 1e-5
            o.precision = prec
            o.refine_iters = refine
            o.transfer_mode = mode
            (info, N, t, y), = _lib.mesh_select(ctx, o, [s])
            ref = O.mesh_select(O.opts(4, abstol=1e-5, transfer_mode=mode), s)
            assert (info, N) == (int(ref[0]), int(ref[1]))
            if info == 0:
                # the defect is a difference of O(1) quantities: relative rounding noise
                # ~1e-15 / defect, and the nodes move by up to ~100x that; the solution's
                # slope is up to 20 (the largest rate) times its size
                e, _ = O.defect(4, s)
                tol_t = max(1e-10, 1e-13 / np.min(np.max(np.abs(e), axis=1)))
                assert np.max(np.abs(t - ref[2])) <= tol_t
                assert np.max(np.abs(y - ref[3])) <= (1e-9 + 40 * tol_t) * max(1.0, np.max(np.abs(ref[3])))
