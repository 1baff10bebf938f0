"""SFS stretching of a weak cluster whose workgroup (leaf) also holds a far stronger
vortex.  J at the strong cluster is 1e7 times that at the weak one, 500 cores
away; the stretching of the weak particles may round with the J and Gamma of
the pairs that zeta joins, not with the strong ones:
  |E_i - ref_i| <= c 2^-53 sum_j zeta_ij (|J_i| + |J_j|) |Gamma_j|
against the per-pair sums on the same J.  c: n = 40 additions and below 32
roundings of a term (zeta with x <= 60, the products, the difference), in each
of two parts of at most twice the size: 4 (n + 32).
The dynamic coefficient's averages at the weak cluster, against the oracle's
own J: J carries (n + 16) 2^-53 of 13 there and varies by 0.1, 1e-12 of
the differences, and enters each product twice or more: 1e-10 of the largest."""
import ctypes

import numpy as np
import pytest

from flowunsteady_amd import _native as N
from flowunsteady_amd import vpm
from helpers import make_field
from oracle import oracle as O

pytestmark = pytest.mark.gpu

M = 20            # particles of each cluster
LEAF = vpm.FMM(p=2, ncrit=200, theta=0.4)


def clusters(seed, strong_first):
    """Strong and weak cluster; the Morton order starts at the low corner."""
    rng = np.random.default_rng(seed)
    a, b = rng.uniform(0.0, 0.2, (2, M, 3))
    far = 30.0 * np.ones(3)
    X = np.concatenate([a, b + far]) if strong_first else np.concatenate([a + far, b])
    G = rng.normal(0, 1, (2 * M, 3)) * np.repeat([1e6, 1e-3], M)[:, None]
    return X, G, rng.uniform(0.08, 0.12, 2 * M)


def zeta(kernel, rho):
    if kernel == "gaussianerf":
        return (2 * np.pi) ** -1.5 * np.exp(-rho ** 2 / 2)
    if kernel == "gaussian":
        return 3 / (4 * np.pi) * np.exp(-rho ** 3)
    return 15 / (8 * np.pi) * (1 + rho ** 2) ** -3.5


@pytest.mark.parametrize("strong_first", [True, False])
@pytest.mark.parametrize("fmm", [None, LEAF])
@pytest.mark.parametrize("kernel,transposed", [("gaussianerf", True), ("gaussianerf", False),
                                               ("gaussian", True), ("winckelmans", False)])
def test_weak_cluster_keeps_its_digits(kernel, transposed, fmm, strong_first):
    X, G, s = clusters(7, strong_first)
    pf = make_field(X, G, s, kernel=kernel, transposed=transposed, **({"fmm": fmm} if fmm else {}))
    P = pf._uj_params(sfs=True, fmm=fmm is not None)
    ctx = vpm._context(0)
    ctx.check(N.lib().vpmx_uj(ctx.ptr, pf._ptr(), pf.np, ctypes.byref(pf.layout), ctypes.byref(P)))
    E, J = vpm.get_SFS(pf), vpm.get_J(pf).copy()
    assert np.linalg.norm(J[:M], axis=1).min() > 1e5 * np.linalg.norm(J[M:], axis=1).max()
    ref = O.estr_direct(kernel, transposed, X, J, X, G, s, J)
    r = np.linalg.norm(X[:, None] - X[None], axis=2)
    w = zeta(kernel, r / s[None]) / s[None] ** 3 * np.linalg.norm(G, axis=1)[None]
    nJ = np.linalg.norm(J, axis=1)
    bound = 4 * (2 * M + 32) * 2.0 ** -53 * (w * (nJ[:, None] + nJ[None])).sum(1)
    err = np.linalg.norm(E - ref, axis=1)
    print(kernel, transposed, fmm is not None, strong_first, (err / bound).max())
    assert (err <= bound).all(), (err / bound).max()


@pytest.mark.parametrize("fmm", [False, True])
@pytest.mark.parametrize("kernel", ["gaussianerf", "winckelmans"])
def test_dynamic_averages_of_the_weak_cluster(kernel, fmm):
    X, G, s = clusters(11, True)
    pf = make_field(X, G, s, kernel=kernel, SFS=vpm.DynamicSFS(), relaxation=vpm.norelaxation,
                    fmm=LEAF, UJ=vpm.UJ_fmm_gpu if fmm else vpm.UJ_gpu)
    vpm.euler_gpu(pf, 1e-12)
    P = O.make_params(kernel, True, "rVPM", sfs="dynamic")
    F = O.Field(X, G, s)
    O.euler_step(P, F, 1e-12, False)
    C = pf.particles[vpm.C_INDEX, M:2 * M].T
    for k in (1, 2):
        ref = F.C[M:, k]
        err = np.abs(C[:, k] - ref).max() / np.abs(ref).max()
        print(kernel, fmm, k, err)
        assert err <= 1e-10, (k, err)
