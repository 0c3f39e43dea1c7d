"""Removal of translation and rotation inside the fused step kernel: several
steps per launch, a batch that does not fill its last block, bead counts on
both sides of the wave size and of the four lanes that add a sum."""
import numpy as np
import pytest

import caracal_amd as cam
import oracle_lib as ol
from caracal_amd import workloads

pytestmark = pytest.mark.gpu

SURF = {"h3": (cam.CAM_SURFACE_H3, 1, [1.008] * 3, workloads.H3_TS),
        "ch4h": (cam.CAM_SURFACE_CH4H, 2, [1.008, 12.011] + [1.008] * 4, workloads.CH4H_TS),
        "oh3": (cam.CAM_SURFACE_OH3, 3, workloads.MASSES_OH3_AMU, workloads.OH3_TS)}


@pytest.mark.parametrize("name,nb,nmk,ens", [
    ("h3", 1, cam.CAM_NMK_VALU, cam.CAM_ENS_NVE), ("h3", 2, cam.CAM_NMK_VALU, cam.CAM_ENS_ANDERSEN),
    ("h3", 6, cam.CAM_NMK_VALU, cam.CAM_ENS_NVE), ("h3", 64, cam.CAM_NMK_MFMA, cam.CAM_ENS_ANDERSEN),
    ("oh3", 24, cam.CAM_NMK_VALU, cam.CAM_ENS_ANDERSEN), ("ch4h", 1, cam.CAM_NMK_VALU, cam.CAM_ENS_NVE),
    ("ch4h", 12, cam.CAM_NMK_VALU, cam.CAM_ENS_ANDERSEN), ("ch4h", 64, cam.CAM_NMK_VALU, cam.CAM_ENS_NVE)])
def test_transrot_in_the_step_loop_matches_oracle(name, nb, nmk, ens):
    """Seven steps as launches of three, three and one.  Tolerance: seven
    steps of about 200 dependent roundings are 2e-13 of the largest momentum;
    a nearly linear molecule's tensor amplifies its angular velocity's
    rounding by the ratio of its length to its width, here up to 50, in a
    part of the momentum that is smaller by the same ratio."""
    surface, osurf, amu, ts = SURF[name]
    masses = cam.mass_au(amu)
    ntraj = 64 // nb + 1                             # four lanes per bead; the last block holds one trajectory
    rng = np.random.default_rng(nb)
    beta = float(cam.beta_of(300.0))
    q = ts + rng.normal(0.0, 0.02, (ntraj, nb) + ts.shape) + rng.normal(0.0, 2.0, (ntraj, 1, 1, 3))
    p = workloads.mb_momenta(rng, masses, nb, beta, q.shape)
    kw = dict(ensemble=ens, remove_com=True, steps_per_launch=3, nm_kernel=nmk, seed=9)
    if ens == cam.CAM_ENS_ANDERSEN:
        kw["andersen_step"] = 4
    dt = 0.1 * cam.FS_TO_AU
    with cam.RPMDEngine(surface, nb, ntraj, dt, masses, **kw) as e:
        e.set_state(q, p, beta)
        e.run(7)
        qe, pe = e.get_state()
    s = ol.make_sys(osurf, nb, dt, masses)
    for t in (0, 1, ntraj - 1):
        o = ol.OracleTraj(s, q[t], p[t], beta, ensemble=1 if ens == cam.CAM_ENS_ANDERSEN else 0, remove_com=True,
                          andersen_step=4, seed=9, traj=t)
        for _ in range(7):
            o.step()
        assert np.abs(qe[t] - o.q).max() <= 1e-12 * np.abs(o.q).max(), (t, np.abs(qe[t] - o.q).max())
        assert np.abs(pe[t] - o.p).max() <= 1e-12 * np.abs(o.p).max(), (t, np.abs(pe[t] - o.p).max())
