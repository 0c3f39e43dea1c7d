"""Recrossing parents stepped inside the step kernel: launches that end inside
a run, bead counts without a normal-mode transform, with lane slots left over
and with the matrix-core transform, and a batch that does not fill its last
block; against the oracle."""
import time

import numpy as np
import pytest

import caracal_amd as cam
import oracle_lib as ol
from caracal_amd import workloads
from test_gpu_parent import _parents

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("surface,nb,nmk", [
    (cam.CAM_SURFACE_H3, 1, cam.CAM_NMK_AUTO), (cam.CAM_SURFACE_H3, 2, cam.CAM_NMK_AUTO),
    (cam.CAM_SURFACE_H3, 6, cam.CAM_NMK_AUTO), (cam.CAM_SURFACE_H3, 64, cam.CAM_NMK_MFMA),
    (cam.CAM_SURFACE_CH4H, 1, cam.CAM_NMK_AUTO), (cam.CAM_SURFACE_CH4H, 12, cam.CAM_NMK_AUTO),
    (cam.CAM_SURFACE_CH4H, 64, cam.CAM_NMK_AUTO)])
def test_parent_steps_match_oracle_across_launches(surface, nb, nmk):
    """Ten steps as launches of four, four and two, run as 7 + 3.  Tolerances
    as the parent's other parity test: 1e-10 relative in the positions, where
    the constraint's stopping rule (|xi| < 1e-10) is the largest term."""
    ntraj = 64 // nb + 1                             # four lanes per bead; the last block holds one trajectory
    w, q, p, beta, rx = _parents(surface, nb, ntraj, seed=nb + 5)
    kw = dict(andersen_step=4, seed=3)
    with cam.RPMDEngine(surface, nb, ntraj, w["dt"], w["masses"], ensemble=cam.CAM_ENS_PARENT, reaction=rx,
                        nm_kernel=nmk, steps_per_launch=4, **kw) as e:
        e.set_state(q, p, beta)
        e.begin_parent(0.2)
        e.run(7)
        e.run(3)
        qe, pe = e.get_state()
        flags = e.observables()["flags"]
    assert not flags.any()
    s, orx = ol.make_sys(surface, nb, w["dt"], w["masses"]), ol.make_rx(rx)
    for t in (0, ntraj - 1):
        o = ol.OracleTraj(s, q[t], p[t], float(beta[t]), rx=orx, ensemble=3, traj=t, **kw)
        o.parent_begin(0.2)
        for _ in range(10):
            o.step()
        assert np.abs(qe[t] - o.q).max() <= 1e-10 * np.abs(o.q).max(), np.abs(qe[t] - o.q).max()
        assert np.abs(pe[t] - o.p).max() <= 1e-9 * np.abs(o.p).max(), np.abs(pe[t] - o.p).max()


def test_a_partly_filled_block_costs_no_more_than_a_full_one():
    """The slots past the last trajectory hold a copy of it: nine BrH2 parents
    of eight beads (eight to a block) take the time of sixteen.  Run on what
    their LDS happened to hold, those slots went NaN, and a NaN matrix keeps
    the eigenvalue iteration busy to its limit, for the whole wave: seven
    times the step."""
    best = {}
    for ntraj in (16, 9):
        w = workloads.brh2_nve(nbeads=8)
        rng = np.random.default_rng(3)
        q = w["q"][None] + rng.normal(0.0, 0.01, (ntraj,) + w["q"].shape)
        p = rng.normal(size=q.shape) * np.sqrt(w["masses"][:, None] * 8 / w["beta"])
        with cam.RPMDEngine(cam.CAM_SURFACE_BRH2, 8, ntraj, w["dt"], w["masses"], ensemble=cam.CAM_ENS_PARENT,
                            reaction=workloads.brh2_reaction(), seed=3) as e:
            e.set_state(q, p, w["beta"])
            e.begin_parent(0.2)
            times = []
            for _ in range(6):
                t = time.perf_counter()
                e.run(300)
                e.sync()
                times.append(time.perf_counter() - t)
        best[ntraj] = min(times)
    print({n: f"{t * 1e6 / 300:.1f} us a step" for n, t in best.items()}, flush=True)
    assert best[9] < 3.0 * best[16]
