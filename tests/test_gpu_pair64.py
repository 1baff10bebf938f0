"""FP64 pair kernels at the edges of their tiles, runs and branches.

  One pair at separations around every branch of the radial functions (series
  below rho = 1.5, erfcx form above, singular form from rho = 9.5) against
  50-digit closed forms.  A and B carry a few roundings each (the polynomials'
  own errors are below 1e-17): U = A c is asked to 16 units of 2^-53, J (two
  terms of opposite sign) to 64.
  Single-leaf FMM fields of every kind of lane packing (1 to 65 targets in a
  leaf) against the all-pairs oracle, U, J <= 1e-12; a dynamic-SFS step, whose
  near-field pass also sums D[J], with the numerator's average <= 1e-12 of its
  largest value.
  Fields whose sizes straddle the 64-target workgroups, the 64- and 256-source
  runs and the segment splits against the oracle, <= 1e-12 as everywhere.
"""
import numpy as np
import pytest

from flowunsteady_amd import vpm
from helpers import make_field, normwise
from oracle import oracle as O

mp = pytest.importorskip("mpmath")
pytestmark = pytest.mark.gpu

EPS = 2.0 ** -53
RHOS = [1e-6, 1e-3, 0.05, 0.3, 0.8, 1.0, 1.4999, 1.5, 1.5001, 2.0, 3.3, 5.0, 7.0, 9.4999, 9.5001,
        12.0, 40.0]


def closed(kernel, r, s):
    """A = g/r^3 and B = g'/(s r^4) - 3 g/r^5 to 50 digits."""
    with mp.workdps(60):
        r, s = mp.mpf(r), mp.mpf(s)
        q = r / s
        if kernel == "gaussianerf":
            c = mp.sqrt(2 / mp.pi)
            g = mp.erf(q / mp.sqrt(2)) - c * q * mp.exp(-q * q / 2)
            dg = c * q * q * mp.exp(-q * q / 2)
        else:
            g = q ** 3 * (q * q + mp.mpf(5) / 2) / (q * q + 1) ** mp.mpf(2.5)
            dg = mp.mpf(15) / 2 * q * q / (q * q + 1) ** mp.mpf(3.5)
        return g / r ** 3, dg / (s * r ** 4) - 3 * g / r ** 5


@pytest.mark.parametrize("kernel", ["gaussianerf", "winckelmans"])
def test_one_pair_against_closed_forms(kernel):
    s, G = 0.25, np.array([0.3, -0.7, 0.55])
    for rho in RHOS:
        dX = rho * s * np.array([0.36, -0.48, 0.8])
        X = np.stack([dX, np.zeros(3)])
        pf = make_field(X, np.stack([np.zeros(3), G]), np.array([s, s]), kernel=kernel)
        vpm.UJ_gpu(pf)
        r = mp.sqrt(sum(mp.mpf(float(v)) ** 2 for v in dX))
        A, B = closed(kernel, r, s)
        d = [mp.mpf(float(v)) for v in dX]
        g = [mp.mpf(float(v)) for v in G]
        c = [d[1] * g[2] - d[2] * g[1], d[2] * g[0] - d[0] * g[2], d[0] * g[1] - d[1] * g[0]]
        k = -1 / (4 * mp.pi)
        U = np.array([float(k * A * v) for v in c])
        eps = lambda a, b: {(0, 1): g[2], (1, 2): g[0], (2, 0): g[1], (1, 0): -g[2],
                            (2, 1): -g[0], (0, 2): -g[1]}.get((a, b), 0)
        J = np.array([float(k * (B * c[a] * d[l] + A * eps(a, l))) for l in range(3) for a in range(3)])
        eu = np.abs(vpm.get_U(pf)[0] - U).max() / np.abs(U).max()
        ej = np.abs(vpm.get_J(pf)[0] - J).max() / np.abs(J).max()
        print(kernel, rho, eu / EPS, ej / EPS)
        assert eu <= 16 * EPS and ej <= 64 * EPS, (rho, eu, ej)


@pytest.mark.parametrize("kernel", ["gaussianerf", "gaussian", "winckelmans", "singular"])
@pytest.mark.parametrize("n", [2, 63, 64, 65, 129, 255, 257, 1025, 4161])
def test_field_sizes_against_oracle(kernel, n):
    rng = np.random.default_rng(n)
    X = rng.uniform(-1, 1, (n, 3))
    X[n // 2] = X[0]                     # a coincident pair, skipped
    G = rng.normal(0, 1e-2, (n, 3))
    s = rng.uniform(0.02, 0.08, n)
    pf = make_field(X, G, s, kernel=kernel)
    vpm.UJ_gpu(pf)
    U, J = O.uj_direct(kernel, X, X, G, s)
    if n == 2:                           # only the coincident pair: nothing is induced
        assert not vpm.get_U(pf).any() and not vpm.get_J(pf).any()
        return
    assert normwise(vpm.get_U(pf), U)[0] < 1e-12 and normwise(vpm.get_J(pf), J)[0] < 1e-12


@pytest.mark.parametrize("kernel", ["gaussianerf", "gaussian", "winckelmans", "singular"])
def test_fmm_leaf_sizes_against_oracle(kernel):
    for n in (1, 2, 3, 4, 5, 7, 9, 12, 16, 17, 21, 22, 31, 32, 33, 50, 63, 64, 65, 70):
        rng = np.random.default_rng(100 + n)
        X, G = rng.uniform(-1, 1, (n, 3)), rng.normal(0, 1e-2, (n, 3))
        s = rng.uniform(0.05, 0.4, n)
        pf = make_field(X, G, s, kernel=kernel, fmm=vpm.FMM(p=2, ncrit=70, theta=0.4))
        vpm.UJ_fmm_gpu(pf)
        assert int(vpm._context(0).fmm_stats()["leaves"]) == 1
        U, J = O.uj_direct(kernel, X, X, G, s)
        if n == 1:
            assert not vpm.get_U(pf).any() and not vpm.get_J(pf).any()
            continue
        eu, ej = normwise(vpm.get_U(pf), U)[0], normwise(vpm.get_J(pf), J)[0]
        assert eu < 1e-12 and ej < 1e-12, (n, eu, ej)


@pytest.mark.parametrize("kernel", ["gaussianerf", "gaussian", "winckelmans"])
@pytest.mark.parametrize("n", [3, 20, 32, 33, 65])
def test_fmm_dynamic_leaf_sizes_against_oracle(kernel, n):
    rng = np.random.default_rng(200 + n)
    X, G = rng.uniform(-1, 1, (n, 3)), rng.normal(0, 1e-2, (n, 3))
    s = rng.uniform(0.2, 0.6, n)
    pf = make_field(X, G, s, kernel=kernel, SFS=vpm.DynamicSFS(), relaxation=vpm.norelaxation,
                    fmm=vpm.FMM(p=2, ncrit=70, theta=0.4))
    pf.UJ = vpm.UJ_fmm_gpu
    vpm.euler_gpu(pf, 1e-3)
    P = O.make_params(kernel, True, "rVPM", sfs="dynamic")
    F = O.Field(X, G, s)
    O.euler_step(P, F, 1e-3, False)
    C = pf.particles[vpm.C_INDEX, :n].T
    for k in (1, 2):
        assert np.abs(C[:, k] - F.C[:, k]).max() <= 1e-12 * np.abs(F.C[:, k]).max(), k
    assert normwise(vpm.get_J(pf), F.J.reshape(n, 9))[0] < 1e-12
