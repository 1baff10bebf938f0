"""Mixed direct sums where the split of the source range changes: one segment,
segments of one tile, a partial last tile, a last segment of one particle, and
the sizes around the last split one.  Against the FP64 path over all targets,
normwise <= 1e-6 for U and 3e-6 for J, the bounds of the mixed path everywhere
(the split only regroups FP64 additions)."""
import numpy as np
import pytest

from flowunsteady_amd import vpm
from helpers import make_field, normwise

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 256, 257, 2049, 10007, 131073])
@pytest.mark.parametrize("kernel", ["gaussianerf", "winckelmans"])
def test_split_against_fp64(kernel, n):
    rng = np.random.default_rng(n)
    X, G = rng.uniform(-1.0, 1.0, (n, 3)), rng.standard_normal((n, 3))
    s = np.full(n, 0.5 / n ** (1.0 / 3.0))
    a, b = (make_field(X, G, s, kernel=kernel, precision=p) for p in ("fp64", "mixed"))
    vpm.UJ_gpu(a)
    vpm.UJ_gpu(b)
    if n == 1:
        assert not vpm.get_U(b).any() and not vpm.get_J(b).any()
        return
    assert normwise(vpm.get_U(b), vpm.get_U(a))[0] < 1e-6
    assert normwise(vpm.get_J(b), vpm.get_J(a))[0] < 3e-6
