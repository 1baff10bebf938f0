"""Gathering the caller's matrix and scattering the results on several host
threads: sizes around the first split of the work and with an uneven last
share, every row of the field, rows the library leaves alone, the first refused
particle of several, and batches whose fields straddle the shares.  The values
are copied, so everything is compared bitwise."""
import ctypes

import numpy as np
import pytest

from flowunsteady_amd import _native as N
from flowunsteady_amd import vpm
from helpers import make_field

pytestmark = pytest.mark.gpu


def field(n, seed):
    rng = np.random.default_rng(seed)
    return rng.uniform(-1, 1, (n, 3)), rng.normal(0, 1e-2, (n, 3)), rng.uniform(0.01, 0.02, n)


@pytest.mark.parametrize("n", [1, 32767, 32768, 49157, 270001])
def test_rows_come_back(n):
    X, G, s = field(n, n)
    pf = make_field(X, G, s, precision="mixed")
    pf.particles[vpm.STATIC_INDEX, :n] = np.arange(n) % 3 == 1
    ctx = vpm._context(0)
    ctx.check(N.lib().vpmx_upload(ctx.ptr, pf._ptr(), pf.np, ctypes.byref(pf.layout)))
    before = pf.particles.copy()
    state = (vpm.X_INDEX, vpm.GAMMA_INDEX, vpm.SIGMA_INDEX)
    for rows in state:
        pf.particles[rows, :n] = -1.0
    ctx.check(N.lib().vpmx_download(ctx.ptr, pf._ptr(), pf.np, ctypes.byref(pf.layout)))
    for rows in state + (vpm.STATIC_INDEX, vpm.VOL_INDEX, vpm.M_INDEX):
        assert np.array_equal(pf.particles[rows], before[rows])
    vpm.UJ_gpu(pf)
    U, J = vpm.get_U(pf).copy(), vpm.get_J(pf).copy()
    vpm.UJ_gpu(pf, reset=False)   # U, J go up with the field and come back doubled
    assert np.array_equal(vpm.get_U(pf), 2 * U) and np.array_equal(vpm.get_J(pf), 2 * J)


def test_first_refused_particle_is_named():
    X, G, s = field(100003, 5)
    pf = make_field(X, G, s, precision="mixed")
    for first, second in ((40000, 99000), (17, 16)):
        p = pf.particles.copy()
        pf.particles[vpm.SIGMA_INDEX, first] = 0.0
        pf.particles[vpm.X_INDEX.start, second] = np.nan
        with pytest.raises(Exception) as e:
            vpm.UJ_gpu(pf)
        want = min(first, second)
        assert f"particle {want + 1} " in str(e.value)
        assert ("sigma" if want == first else "non-finite") in str(e.value)
        pf.particles[:] = p


def test_batch_fields_straddle_the_shares():
    sizes = [20000, 0, 1, 30011, 16384, 5]
    one = [make_field(*field(n, 90 + n), precision="fp64") for n in sizes]
    many = [make_field(*field(n, 90 + n), precision="fp64") for n in sizes]
    vpm.UJ_gpu_batch(many)
    for a, b in zip(one, many):
        if a.np == 0:
            continue
        vpm.UJ_gpu(a)
        for get in (vpm.get_U, vpm.get_J):
            d = np.abs(get(a) - get(b)).max()
            assert d <= 1e-13 * max(np.abs(get(a)).max(), 1e-300)
