"""The host-pointer force calls through their thread's staging memory (up to
4096 beads) and through device buffers (above): either side of the limit, every
surface, and several threads calling at once, each with its own beads.  The
same kernel runs either way, so the results of a call equal those of the
allocation-free entry point bit for bit."""
import ctypes
import threading

import numpy as np
import pytest

import caracal_amd as cam
from caracal_amd._abi import lib

pytestmark = pytest.mark.gpu

SURFACES = {"h3": (cam.CAM_SURFACE_H3, 3), "ch4h": (cam.CAM_SURFACE_CH4H, 6), "oh3": (cam.CAM_SURFACE_OH3, 4),
            "brh2": (cam.CAM_SURFACE_BRH2, 3), "o3": (cam.CAM_SURFACE_O3, 3)}


def _beads(na, nb, seed):
    rng = np.random.default_rng(seed)
    return np.arange(na)[None, :, None] * np.array([1.6, 0.3, 0.2]) + rng.normal(0.0, 0.1, (nb, na, 3))


def _noalloc(surface, q):
    dp = ctypes.POINTER(ctypes.c_double)
    v, g = np.empty(len(q)), np.empty_like(q)
    rc = lib().cam_egrad_noalloc(surface, q.ctypes.data_as(dp), q.shape[1], len(q), v.ctypes.data_as(dp),
                                 g.ctypes.data_as(dp))
    assert rc == 0
    return v, g


@pytest.mark.parametrize("nb", [1, 65, 4096, 4097])
@pytest.mark.parametrize("name", sorted(SURFACES))
def test_staged_calls_equal_the_allocation_free_ones(name, nb):
    surface, na = SURFACES[name]
    q = _beads(na, nb, nb)
    v, g = getattr(cam, f"egrad_{name}")(q)
    vr, gr = _noalloc(surface, q)
    assert np.array_equal(v, vr) and np.array_equal(g, gr)


def test_threads_stage_apart():
    jobs = [(name, 17 + 40 * k, 100 + k) for k, name in enumerate(sorted(SURFACES) * 2)]
    bad = []

    def work(name, nb, seed):
        surface, na = SURFACES[name]
        for rep in range(20):
            q = _beads(na, nb, seed + 1000 * rep)
            v, g = getattr(cam, f"egrad_{name}")(q)
            vr, gr = _noalloc(surface, q)
            if not (np.array_equal(v, vr) and np.array_equal(g, gr)):
                bad.append((name, rep))

    threads = [threading.Thread(target=work, args=j) for j in jobs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
