"""Recrossing parents stepped inside the step kernel: launches that end inside
a run, bead counts without a normal-mode transform, with lane slots left over
and with the matrix-core transform, and a batch that does not fill its last
block; against the oracle."""
import numpy as np
import pytest

import caracal_amd as cam
import oracle_lib as ol
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
    per_block = 256 // ((4 if surface == cam.CAM_SURFACE_CH4H else 1) * nb)
    ntraj = per_block + 1
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
