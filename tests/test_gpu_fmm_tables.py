"""The FMM's operator tables are built once per order and basis.

Mixed steps with an SFS model translate in another basis of the M2L than the
other evaluations, so a field may use both in turn.  Tables that were rebuilt on
every change had a size of their own each (311,469 rows of 112 or 176 doubles at
p = 8): device memory in use then differs between the two calls by 160 MB, and
does not once both are kept.  The core-spreading re-fit walks the near lists
only and needs no table at all: on a fresh context it takes its vectors, tree and
lists (20,000 particles: tens of MB), not the 279 MB of operator rows.
"""
import ctypes

import numpy as np
import pytest
import torch

from flowunsteady_amd import _native as N
from flowunsteady_amd import vpm
from helpers import make_field

pytestmark = pytest.mark.gpu

MB = 1 << 20
STEP = 32 * MB


def field(n, **kw):
    rng = np.random.default_rng(n)
    X, G = rng.uniform(-1, 1, (n, 3)), rng.normal(0, 1e-3, (n, 3))
    s = np.full(n, 3.0 / n ** (1.0 / 3.0))
    return make_field(X, G, s, precision="mixed", SFS=vpm.DynamicSFS(), UJ=vpm.UJ_fmm_gpu,
                      fmm=vpm.FMM(p=8, ncrit=50, theta=0.4), **kw)


def used():
    torch.cuda.synchronize()
    free, total = torch.cuda.mem_get_info(0)
    return total - free


def test_alternating_bases_keep_their_tables():
    pf = field(5000)
    ctx = vpm._context(0)

    def evaluate(sfs):
        P = pf._uj_params(sfs=sfs, fmm=True)
        ctx.check(N.lib().vpmx_uj(ctx.ptr, pf._ptr(), pf.np, ctypes.byref(pf.layout),
                                  ctypes.byref(P)))
        return vpm.get_U(pf).copy(), vpm.get_J(pf).copy(), used()

    first = [evaluate(sfs) for sfs in (False, True)]
    for _ in range(2):
        for sfs in (False, True):
            U, J, held = evaluate(sfs)
            assert abs(held - first[1][2]) < STEP, (sfs, held, first[1][2])
            assert np.array_equal(U, first[sfs][0]) and np.array_equal(J, first[sfs][1])
    # another order: its own tables and results, and back
    pf.fmm = vpm.FMM(p=4, ncrit=50, theta=0.4)
    evaluate(False), evaluate(True)
    pf.fmm = vpm.FMM(p=8, ncrit=50, theta=0.4)
    for sfs in (True, False):
        U, J, _ = evaluate(sfs)
        assert np.array_equal(U, first[sfs][0]) and np.array_equal(J, first[sfs][1])


def test_refit_builds_no_tables():
    pf = field(20000, viscous=vpm.CoreSpreading(1e-4, 3.0 / 20000 ** (1.0 / 3.0), vpm.zeta_fmm,
                                                itmax=2, tol=1e-1))
    ctx, L = N.Context(0), N.lib()
    ctx.check(L.vpmx_upload(ctx.ptr, pf._ptr(), pf.np, ctypes.byref(pf.layout)))
    base = used()
    P, S = pf._uj_params(fmm=True), pf._step_params()
    ctx.check(L.vpmx_core_spreading_reset(ctx.ptr, ctypes.byref(P), ctypes.byref(S), 1, None, None,
                                          None))
    held = used() - base
    ctx.close()
    assert held < 128 * MB, held
