"""The device traversal's output slots (blocks of 1,024 frontier pairs, partial
blocks, levels of one pair and of many blocks): the counts of every list equal
the host plan's, and so do the sums, since a slot written twice or left out
loses pairs: U, J against the CPU FMM over the same lists, <= 1e-12 as
everywhere."""
import numpy as np
import pytest

from flowunsteady_amd import _native as N
from flowunsteady_amd import vpm
from helpers import make_field, normwise
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ncrit", [(1, 1), (9, 1), (40, 4), (300, 1), (1000, 1), (20011, 30)])
def test_lists_equal_the_host_plan(n, ncrit):
    rng = np.random.default_rng(n)
    X, G = rng.normal(0, 0.3, (n, 3)), rng.normal(0, 1e-2, (n, 3))
    s = np.full(n, 0.2 / n ** (1.0 / 3.0))
    pf = make_field(X, G, s, fmm=vpm.FMM(p=4, ncrit=ncrit, theta=0.4, nonzero_sigma=True))
    vpm.UJ_fmm_gpu(pf)
    st = vpm._context(0).fmm_stats()
    want = N.fmm_plan_counts(X, s, ncrit, 0.4, 7.0)
    assert int(st["m2l_pairs"]) == want["nm2l"]
    assert int(st["p2p_leaf_pairs"]) == want["np2p"]
    assert int(st["p2p_pairs"]) == want["p2p_pairs"]
    if n > 1:
        U, J, _ = O.uj_fmm("gaussianerf", X, G, s, p=4, ncrit=ncrit, theta=0.4, sigcut=7.0)
        assert normwise(vpm.get_U(pf), U)[0] < 1e-12
        assert normwise(vpm.get_J(pf), J.reshape(n, 9))[0] < 1e-12


@pytest.mark.parametrize("n,ncrit", [(2, 1), (255, 1), (257, 1), (5000, 2), (70001, 8)])
def test_tree_equals_the_host_plan(n, ncrit):
    """Cells and leaves of the device tree, with coincident particles at both
    corners of the cube and inside, which split down to the last level always
    into the first, the last or some inner octant."""
    rng = np.random.default_rng(n + 1)
    X = rng.uniform(-1.0, 1.0, (n, 3))
    k = max(1, n // 8)
    X[:k], X[k:2 * k] = -1.0, 1.0
    if n > 16:
        X[2 * k:3 * k] = (0.3, -0.2, 0.1)
    s = np.full(n, 0.2 / n ** (1.0 / 3.0))
    pf = make_field(X, rng.normal(0, 1e-2, (n, 3)), s,
                    fmm=vpm.FMM(p=1, ncrit=ncrit, theta=0.4, nonzero_sigma=True))
    vpm.UJ_fmm_gpu(pf)
    st = vpm._context(0).fmm_stats()
    want = N.fmm_plan_counts(X, s, ncrit, 0.4, 7.0)
    assert int(st["cells"]) == want["ncell"] and int(st["leaves"]) == want["nleaf"]
    assert int(st["p2p_pairs"]) == want["p2p_pairs"]
