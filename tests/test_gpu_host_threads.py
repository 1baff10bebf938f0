"""When host threads gather and scatter the caller's matrix: none below 49,152
particles, where starting them costs more than they save, some from there on.
Thread ids are handed out in sequence, so the ids of two threads started right
before and after a call tell how many it started; another process can only add
to that, hence the least of several tries."""
import ctypes
import threading

import numpy as np
import pytest

from flowunsteady_amd import _native as N
from flowunsteady_amd import vpm
from helpers import make_field

pytestmark = pytest.mark.gpu


def thread_id():
    t = threading.Thread(target=lambda: None)
    t.start()
    t.join()
    return t.native_id


@pytest.mark.parametrize("n,threaded", [(1000, False), (33000, False), (49151, False),
                                        (49152, True), (65536, True), (200003, True)])
def test_threads_of_a_call(n, threaded):
    rng = np.random.default_rng(n)
    pf = make_field(rng.uniform(-1, 1, (n, 3)), rng.normal(0, 1, (n, 3)), np.full(n, 0.1))
    ctx, L = vpm._context(0), N.lib()
    before = pf.particles.copy()

    def there_and_back():
        ctx.check(L.vpmx_upload(ctx.ptr, pf._ptr(), n, ctypes.byref(pf.layout)))
        ctx.check(L.vpmx_download(ctx.ptr, pf._ptr(), n, ctypes.byref(pf.layout)))

    there_and_back()
    started = []
    for _ in range(8):
        a = thread_id()
        there_and_back()
        started.append(thread_id() - a - 1)
    state = np.r_[vpm.X_INDEX, vpm.GAMMA_INDEX, vpm.SIGMA_INDEX]
    assert np.array_equal(pf.particles[state], before[state])
    if threaded:
        assert max(started) > 0, started
    else:
        assert min(started) <= 0, started
