"""The matrix-core M2L's two bases (the independent harmonic coefficients; every
Cartesian coefficient, kept for mixed-precision evaluations that feed the SFS
stretching pass) give the same truncated far field: the same mixed evaluation
with and without Estr differs by FP64 rounding only (the near field is the same
code), asked here to 1e-13, at every order, with level gaps between the cells and
separations inside and outside the operator table."""
import ctypes

import numpy as np
import pytest

from flowunsteady_amd import _native as N
from flowunsteady_amd import vpm, workloads
from helpers import make_field, normwise

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p", range(1, 11))
def test_harmonic_and_full_basis_agree(p):
    X, G, s, _ = workloads.gaussian_blob(n=6000, seed=6)
    rng = np.random.default_rng(7)
    d = rng.standard_normal((200, 3))
    X = np.vstack([X, 40.0 * d / np.linalg.norm(d, axis=1, keepdims=True)])   # sparse distant shell
    G = np.vstack([G, 1e-3 * rng.standard_normal((200, 3))])
    s = np.concatenate([s, np.full(200, 0.05)])
    out = []
    for sfs in (False, True):
        pf = make_field(X, G, s, precision="mixed", fmm=vpm.FMM(p=p, ncrit=20, theta=0.5))
        P = pf._uj_params(sfs=sfs, fmm=True)
        ctx = vpm._context(0)
        ctx.check(N.lib().vpmx_uj(ctx.ptr, pf._ptr(), pf.np, ctypes.byref(pf.layout),
                                  ctypes.byref(P)))
        out.append((vpm.get_U(pf).copy(), vpm.get_J(pf).copy()))
    eu, ej = normwise(out[0][0], out[1][0]), normwise(out[0][1], out[1][1])
    print(p, eu, ej)
    assert eu[0] < 1e-13 and ej[0] < 1e-13
