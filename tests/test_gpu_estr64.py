"""FP64 SFS stretching at the edges of its tiles: sizes around the 64-target
workgroups and runs, the 256-source tiles and the segment splits (all pairs),
and every kind of lane packing of one leaf (FMM lists), both schemes, against
the oracle's sums on the same J.  A sum of n <= 4,100 products carries at most
~n 2^-53 = 5e-13 of its terms' size: <= 1e-12 of max |E|.  Isolated particles
have E = 0 exactly (no rounding of their own stretching)."""
import ctypes

import numpy as np
import pytest

from flowunsteady_amd import _native as N
from flowunsteady_amd import vpm
from helpers import make_field, normwise
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def estr(X, G, s, kernel, transposed, fmm=None):
    pf = make_field(X, G, s, kernel=kernel, transposed=transposed, **({"fmm": fmm} if fmm else {}))
    P = pf._uj_params(sfs=True, fmm=fmm is not None)
    ctx = vpm._context(0)
    ctx.check(N.lib().vpmx_uj(ctx.ptr, pf._ptr(), pf.np, ctypes.byref(pf.layout), ctypes.byref(P)))
    return vpm.get_SFS(pf).copy(), vpm.get_J(pf).copy()


def check(X, G, s, kernel, transposed, fmm=None):
    E, J = estr(X, G, s, kernel, transposed, fmm)
    ref = O.estr_direct(kernel, transposed, X, J, X, G, s, J)
    assert normwise(E, ref)[0] < 1e-12


def field(n, seed):
    rng = np.random.default_rng(seed)
    L = max(1.0, (n / 60.0) ** (1.0 / 3.0))
    return rng.uniform(-L, L, (n, 3)), rng.normal(0, 1e-2, (n, 3)), rng.uniform(0.2, 0.6, n)


@pytest.mark.parametrize("n", [2, 63, 64, 65, 257, 1000, 4097])
@pytest.mark.parametrize("kernel,transposed", [("gaussianerf", True), ("gaussianerf", False),
                                               ("gaussian", True), ("winckelmans", False)])
def test_direct(kernel, transposed, n):
    check(*field(n, n), kernel, transposed)


@pytest.mark.parametrize("n", [2, 4, 5, 20, 32, 33, 64, 65, 130])
@pytest.mark.parametrize("kernel,transposed", [("gaussianerf", True), ("winckelmans", False)])
def test_one_leaf(kernel, transposed, n):
    check(*field(n, 50 + n), kernel, transposed, vpm.FMM(p=2, ncrit=200, theta=0.4))


@pytest.mark.parametrize("fmm", [None, vpm.FMM(p=2, ncrit=200, theta=0.4)])
@pytest.mark.parametrize("n", [1, 3, 70])
def test_isolated_particles(n, fmm):
    rng = np.random.default_rng(n)
    X = np.stack([np.arange(n) * 50.0, rng.uniform(0, 1, n), rng.uniform(0, 1, n)], axis=1)
    E, _ = estr(X, rng.normal(0, 1.0, (n, 3)), np.full(n, 0.5), "gaussianerf", True, fmm)
    assert not E.any()
