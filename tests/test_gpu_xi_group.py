"""The window bias inside the fused step (a group of lanes per trajectory)
against the split schedule's kernel (one wave per trajectory, another
formulation of the same derivatives): reactions of several bonds and three
reactants, bead counts with one and with many trajectories per block."""
import numpy as np
import pytest

import caracal_amd as cam
from caracal_amd import workloads
from caracal_amd.engine import Reaction

pytestmark = pytest.mark.gpu


def _reaction(name):
    if name == "h3":
        return workloads.h3_reaction()
    ts = workloads.CH4H_TS
    d = lambda a, b: float(np.linalg.norm(ts[a - 1] - ts[b - 1]))
    form, brk = [(3, 6), (1, 6)], [(2, 3), (2, 4), (2, 5)]
    return Reaction(bond_form=form, bond_break=brk, form_ref=[d(*b) for b in form], break_ref=[d(*b) for b in brk],
                    reactants=[[1, 2, 4], [3, 5], [6]], r_inf=14.0, xi_ideal=0.8)


@pytest.mark.parametrize("name,nb,ntraj", [("h3", 2, 1), ("h3", 4, 65), ("h3", 64, 5), ("ch4h", 1, 9), ("ch4h", 2, 33),
                                           ("ch4h", 16, 6)])
def test_fused_window_steps_equal_split_steps(name, nb, ntraj):
    """Eight steps, two of them with a momentum draw.  Tolerance: the two
    evaluations differ by some hundred roundings per step, 1e-13 of the bias
    gradient, which at the force constant used is at most ten times the
    surface's; eight steps of it stay below 1e-11 of the momenta."""
    surface, amu, ts = ((cam.CAM_SURFACE_H3, [1.008] * 3, workloads.H3_TS) if name == "h3" else
                        (cam.CAM_SURFACE_CH4H, [1.008, 12.011] + [1.008] * 4, workloads.CH4H_TS))
    masses, beta = cam.mass_au(amu), float(cam.beta_of(300.0))
    rng = np.random.default_rng(nb)
    q = ts + rng.normal(0.0, 0.02, (ntraj, nb) + ts.shape)
    p = workloads.mb_momenta(rng, masses, nb, beta, q.shape)
    xi, kf = rng.uniform(0.95, 1.0, ntraj), np.full(ntraj, 1.5)
    res = {}
    for sched in (cam.CAM_SCHED_FUSED, cam.CAM_SCHED_SPLIT):
        with cam.RPMDEngine(surface, nb, ntraj, 0.1 * cam.FS_TO_AU, masses, ensemble=cam.CAM_ENS_UMBRELLA,
                            reaction=_reaction(name), andersen_step=3, remove_com=True, schedule=sched,
                            nm_kernel=cam.CAM_NMK_VALU, steps_per_launch=0 if sched == cam.CAM_SCHED_SPLIT else 5) as e:
            e.set_windows(xi, kf)
            e.set_state(q, p, beta)
            e.begin_umbrella(bias=True)
            e.run(8)
            res[sched] = e.get_state() + e.umbrella_stats()
    (qf, pf, af, vf), (qs, ps, as_, vs) = res[cam.CAM_SCHED_FUSED], res[cam.CAM_SCHED_SPLIT]
    for a, b, tol in ((qf, qs, 1e-12), (pf, ps, 1e-11), (af, as_, 1e-12)):
        assert np.abs(a - b).max() <= tol * np.abs(b).max(), (np.abs(a - b).max(), np.abs(b).max())
    # the variance is mean(xi^2) - mean(xi)^2 with xi near 1: its rounding is
    # some epsilon of those squares (2.2e-16 each), not of the difference
    assert np.abs(vf - vs).max() <= 1e-14
