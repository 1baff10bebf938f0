"""A core size that is not a number shows in every velocity it enters, on arrays
the library does not check (device pointers): all targets but the particle
itself, whose own pair is skipped."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

pytest.importorskip("torch")


@pytest.mark.parametrize("n", [3, 70, 1000])
@pytest.mark.parametrize("kernel", ["gaussian", "gaussianerf", "winckelmans"])
def test_nan_core_is_seen(kernel, n):
    from flowunsteady_amd import vpm
    from test_zz_no_alloc import _cloud, _noalloc
    X, G, s = _cloud(n, n)
    s[1] = np.nan
    U, J = _noalloc(vpm._context(0), X, G, s, kernel)
    others = np.arange(n) != 1
    assert np.isfinite(U[1]).all() and np.isfinite(J[1]).all()
    assert np.isnan(U[others]).all() and np.isnan(J[others]).all()
