"""Host threads may not make a call slower: the matrix goes up and the state comes
back, again and again, right above the size from which threads help (35,500) and
right below it (32,000).  Per particle the former may not cost more (15 % allowed;
0.8 is usual).  Equal shares for two threads, of which the late one writes lines
that the caller's cache holds, cost up to 1.8 times as much, now and then: nine of
twelve medians have to pass.  And every particle is moved exactly once, whatever
the share of each thread."""
import ctypes
import time

import numpy as np
import pytest

from flowunsteady_amd import _native as N
from flowunsteady_amd import vpm
from helpers import make_field

pytestmark = pytest.mark.gpu


def field(n):
    rng = np.random.default_rng(n)
    return make_field(rng.uniform(-1, 1, (n, 3)), rng.normal(0, 1, (n, 3)),
                      rng.uniform(0.1, 0.2, n))


def there_and_back(pf):
    ctx, L = vpm._context(0), N.lib()
    ctx.check(L.vpmx_upload(ctx.ptr, pf._ptr(), pf.np, ctypes.byref(pf.layout)))
    ctx.check(L.vpmx_download(ctx.ptr, pf._ptr(), pf.np, ctypes.byref(pf.layout)))


def per_particle(pf):
    t = []
    for _ in range(30):
        a = time.perf_counter()
        there_and_back(pf)
        t.append(time.perf_counter() - a)
    return np.median(t) / pf.np


def test_threads_do_not_cost_more_than_they_save():
    below, above = field(32000), field(35500)
    ratios = sorted(per_particle(above) / per_particle(below) for _ in range(12))
    print(np.round(ratios, 2))
    assert ratios[8] < 1.15, ratios


@pytest.mark.parametrize("n", [32767, 32768, 34816, 34817, 49151, 65536, 99999, 300001])
def test_every_particle_is_moved(n):
    pf = field(n)
    before = pf.particles.copy()
    state = np.r_[vpm.X_INDEX, vpm.GAMMA_INDEX, vpm.SIGMA_INDEX]
    ctx, L = vpm._context(0), N.lib()
    for _ in range(4):
        ctx.check(L.vpmx_upload(ctx.ptr, pf._ptr(), n, ctypes.byref(pf.layout)))
        pf.particles[state] = np.nan
        ctx.check(L.vpmx_download(ctx.ptr, pf._ptr(), n, ctypes.byref(pf.layout)))
        assert np.array_equal(pf.particles[state], before[state])
