"""Close pairs of the gaussian kernel, g = 1 - e^{-rho^3}, against 50-digit closed
forms: separations from 1e-6 cores on, around the end of the series at rho = 0.9
and beyond, on the all-pairs kernel, the near field of one FMM leaf, and that
near field with the dynamic model's core-size derivatives.  A and B carry a few
roundings each: U = A c is asked to 16 units of 2^-53, J (two terms of opposite
sign) to 64, as for the other kernels.  (1 - e^{-y} formed as a difference is 0
below y = 1e-16 and off by 1e-16 / y above.)"""
import numpy as np
import pytest

from flowunsteady_amd import vpm
from helpers import make_field

mp = pytest.importorskip("mpmath")
pytestmark = pytest.mark.gpu

EPS = 2.0 ** -53
RHOS = [1e-6, 1e-4, 1e-3, 0.01, 0.05, 0.3, 0.6, 0.8, 0.8999, 0.9, 0.9001, 1.0, 1.5, 2.0, 3.0, 9.4]


def closed(r, s):
    """A = g/r^3 and B = g'/(s r^4) - 3 g/r^5 to 50 digits."""
    with mp.workdps(90):
        q = r / mp.mpf(s)
        g, dg = -mp.expm1(-q ** 3), 3 * q * q * mp.exp(-q ** 3)
        return g / r ** 3, dg / (mp.mpf(s) * r ** 4) - 3 * g / r ** 5


@pytest.mark.parametrize("rho", RHOS)
@pytest.mark.parametrize("path", ["direct", "leaf", "dynamic leaf"])
def test_one_pair(path, rho):
    s, G = 0.25, np.array([0.3, -0.7, 0.55])
    dX = rho * s * np.array([0.36, -0.48, 0.8])
    pf = make_field(np.stack([dX, np.zeros(3)]), np.stack([np.zeros(3), G]), np.array([s, s]),
                    kernel="gaussian", fmm=vpm.FMM(p=2, ncrit=50, theta=0.4),
                    SFS=vpm.DynamicSFS() if path == "dynamic leaf" else vpm.noSFS,
                    relaxation=vpm.norelaxation)
    pf.UJ = vpm.UJ_gpu if path == "direct" else vpm.UJ_fmm_gpu
    if path == "dynamic leaf":
        vpm.euler_gpu(pf, 0.0)
    else:
        pf.UJ(pf)
    d, g = [mp.mpf(float(v)) for v in dX], [mp.mpf(float(v)) for v in G]
    with mp.workdps(90):
        A, B = closed(mp.sqrt(sum(v * v for v in d)), s)
        c = [d[1] * g[2] - d[2] * g[1], d[2] * g[0] - d[0] * g[2], d[0] * g[1] - d[1] * g[0]]
        k = -1 / (4 * mp.pi)
        U = np.array([float(k * A * v) for v in c])
        eps = {(0, 1): g[2], (1, 2): g[0], (2, 0): g[1], (1, 0): -g[2], (2, 1): -g[0], (0, 2): -g[1]}
        J = np.array([float(k * (B * c[a] * d[l] + A * eps.get((a, l), 0)))
                      for l in range(3) for a in range(3)])
    eu = np.abs(vpm.get_U(pf)[0] - U).max() / np.abs(U).max()
    ej = np.abs(vpm.get_J(pf)[0] - J).max() / np.abs(J).max()
    print(path, rho, eu / EPS, ej / EPS)
    assert eu <= 16 * EPS and ej <= 64 * EPS, (eu / EPS, ej / EPS)
