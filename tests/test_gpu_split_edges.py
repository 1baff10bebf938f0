"""Direct sums at the last sizes whose source range is split and the first that
run whole: 1024 / 1025 blocks of 256 targets (mixed), 2048 / 2049 blocks of 64
(FP64).  The segments hold half the sources each and the partial sums fill their
buffer.  Against the oracle at 96 targets, the first and last slots' among them,
normwise as everywhere: <= 1e-12 (FP64), 1e-6 for U and 3e-6 for J (mixed)."""
import numpy as np
import pytest

from flowunsteady_amd import vpm
from helpers import make_field, normwise, sample_targets
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,n", [("fp64", 131072), ("fp64", 131073), ("mixed", 262143),
                                         ("mixed", 262144), ("mixed", 262145)])
@pytest.mark.parametrize("kernel", ["gaussianerf", "winckelmans"])
def test_last_split_sizes(kernel, precision, n):
    rng = np.random.default_rng(n)
    X, G = rng.uniform(-1.0, 1.0, (n, 3)), rng.standard_normal((n, 3))
    s = np.full(n, 0.5 / n ** (1.0 / 3.0))
    pf = make_field(X, G, s, kernel=kernel, precision=precision)
    vpm.UJ_gpu(pf)
    t = np.unique(np.concatenate([sample_targets(n, 90, seed=1), np.argsort(X.sum(1))[[0, 1, -2, -1]],
                                  [0, n - 1]]))
    U, J = O.uj_direct(kernel, X[t], X, G, s)
    tol = (1e-12, 1e-12) if precision == "fp64" else (1e-6, 3e-6)
    assert np.isfinite(vpm.get_U(pf)).all() and np.isfinite(vpm.get_J(pf)).all()
    assert normwise(vpm.get_U(pf)[t], U)[0] < tol[0] and normwise(vpm.get_J(pf)[t], J)[0] < tol[1]
