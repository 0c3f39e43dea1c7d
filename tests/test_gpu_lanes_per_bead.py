"""The H3, OH3, BrH2 and O3 step kernels take four lanes per bead in small
batches and one in large ones: the same trajectories on both sides of the line
(the largest batch of the one, the smallest of the other), and the four-lane
surfaces against the oracle where their lanes branch differently."""
import numpy as np
import pytest

import caracal_amd as cam
import oracle_lib as ol
from caracal_amd import workloads

pytestmark = pytest.mark.gpu

SURF = {"h3": (cam.CAM_SURFACE_H3, [1.008] * 3, workloads.H3_TS),
        "oh3": (cam.CAM_SURFACE_OH3, workloads.MASSES_OH3_AMU, workloads.OH3_TS),
        "brh2": (cam.CAM_SURFACE_BRH2, workloads.MASSES_BRH2_AMU, workloads.BRH2_TS),
        "o3": (cam.CAM_SURFACE_O3, workloads.MASSES_O3_AMU, workloads.O3_TS)}


@pytest.mark.parametrize("name,ens,prec", [
    (n, e, cam.CAM_PREC_FP64) for n in SURF for e in (cam.CAM_ENS_NVE, cam.CAM_ENS_ANDERSEN)]
    + [("h3", cam.CAM_ENS_NVE, cam.CAM_PREC_MIXED), ("h3", cam.CAM_ENS_NHC, cam.CAM_PREC_MIXED)])
def test_both_sides_of_the_line_give_the_same_trajectories(name, ens, prec):
    """64 beads (one trajectory per block on four lanes): the line is a number
    of trajectories.  Forces of both forms are within 1e-13 hartree/bohr of
    each other in FP64 (O3, whose polynomial terms cancel from 1e5 kcal/mol;
    1e-15 the others) and 2e-8 with H3's binary32 corrections, and five steps
    move a momentum by 5 dt |dF| at most."""
    surface, amu, ts = SURF[name]
    limit = 256 if name == "brh2" else 1536 if ens == cam.CAM_ENS_NVE else 512
    masses, beta, dt = cam.mass_au(amu), float(cam.beta_of(300.0)), 0.1 * cam.FS_TO_AU
    rng = np.random.default_rng(1)
    q = ts + rng.normal(0.0, 0.05, (limit + 1, 64) + ts.shape)
    p = workloads.mb_momenta(rng, masses, 64, beta, q.shape)
    kw = dict(ensemble=ens, precision=prec, seed=4)
    if ens == cam.CAM_ENS_ANDERSEN:
        kw["andersen_step"] = 3
    if ens == cam.CAM_ENS_NHC:
        kw["nose_q"] = 20 * dt
    out = []
    for n in (limit, limit + 1):
        with cam.RPMDEngine(surface, 64, n, dt, masses, **kw) as e:
            e.set_state(q[:n], p[:n], beta)
            v, g = e.get_forces()
            e.run(5)
            out.append((v[:limit], g[:limit]) + tuple(x[:limit] for x in e.get_state()))
    df = 2e-8 if prec == cam.CAM_PREC_MIXED else 1e-12 if name == "o3" else 1e-14
    (v4, g4, q4, p4), (v1, g1, q1, p1) = out
    assert np.abs(v4 - v1).max() <= df and np.abs(g4 - g1).max() <= df
    assert np.abs(p4 - p1).max() <= 5 * dt * df + 1e-13 * np.abs(p1).max()
    assert np.abs(q4 - q1).max() <= 25 * dt * dt * df / masses.min() + 1e-13 * np.abs(q1).max()
    assert not np.array_equal(g4, g1) or name != "h3"       # two forms ran: their roundings differ


REACTION = {"h3": workloads.h3_reaction, "oh3": workloads.oh3_reaction, "brh2": workloads.brh2_reaction,
            "o3": workloads.o3_reaction}


@pytest.mark.parametrize("kind,nb,nmk", [
    (kind, nb, nmk) for nb, nmk in ((64, cam.CAM_NMK_VALU), (24, cam.CAM_NMK_VALU), (64, cam.CAM_NMK_MFMA))
    for kind in ("nve transrot", "andersen transrot", "parent", "nhc", "window", "window transrot")
    if nmk == cam.CAM_NMK_VALU or kind in ("nve transrot", "andersen transrot", "parent")])
@pytest.mark.parametrize("name", list(SURF))
def test_both_sides_of_the_line_with_what_a_step_adds(name, kind, nb, nmk):
    """transrot, the chain, the window's bias and the parent's constraints in the
    kernels of one and of four lanes per bead, five steps as launches of three
    and two; the larger batch does not fill its last one-lane block at 24 beads.
    Tolerances as where these are compared to the oracle: 1e-12 of the largest
    position and momentum for transrot and the chain, 1e-11 of the momenta for
    the bias, 1e-10 and 1e-9 under the constraint, whose iteration stops at
    |xi| < 1e-10; O3's forces add 1e-12 hartree/bohr."""
    surface, amu, ts = SURF[name]
    limit = (256 if name == "brh2" else 512) * (64 // nb)
    masses, beta, dt = cam.mass_au(amu), float(cam.beta_of(300.0)), 0.1 * cam.FS_TO_AU
    rng = np.random.default_rng(2)
    q = ts + rng.normal(0.0, 0.02, (limit + 1, nb) + ts.shape)
    p = workloads.mb_momenta(rng, masses, nb, beta, q.shape)
    kw = dict(seed=4, steps_per_launch=3, nm_kernel=nmk, remove_com="transrot" in kind)
    kw["ensemble"] = {"nve": cam.CAM_ENS_NVE, "andersen": cam.CAM_ENS_ANDERSEN, "window": cam.CAM_ENS_UMBRELLA,
                      "parent": cam.CAM_ENS_PARENT, "nhc": cam.CAM_ENS_NHC}[kind.split()[0]]
    if kind == "nhc":
        kw["nose_q"] = 20 * dt
    elif not kind.startswith("nve"):
        kw["andersen_step"] = 4
    steered = kind.startswith(("window", "parent"))
    if steered:
        kw["reaction"] = REACTION[name]()
    out = []
    for n in (limit, limit + 1):
        with cam.RPMDEngine(surface, nb, n, dt, masses, **kw) as e:
            if kind.startswith("window"):
                e.set_windows(np.linspace(0.9, 1.05, limit + 1)[:n], np.full(n, 1.5))
            e.set_state(q[:n], p[:n], beta)
            if kind.startswith("window"):
                e.begin_umbrella(bias=True)
            if kind == "parent":
                assert not e.constrain(project_p=True).any()
                e.begin_parent(0.2)
            e.run(5)
            out.append([x[:limit] for x in e.get_state()])
            if kind.startswith("window"):
                out[-1] += [x[:limit] for x in e.umbrella_stats()]
            if kind == "parent":
                assert not e.observables()["flags"].any()
    (q4, p4), (q1, p1) = out[0][:2], out[1][:2]
    tq, tp = (1e-10, 1e-9) if kind == "parent" else (1e-12, 1e-11 if kind.startswith("window") else 1e-12)
    df = 1e-12 if name == "o3" else 1e-14
    assert np.isfinite(q4).all() and np.isfinite(p4).all()
    assert np.abs(p4 - p1).max() <= 5 * dt * df + tp * np.abs(p1).max()
    assert np.abs(q4 - q1).max() <= 25 * dt * dt * df / masses.min() + tq * np.abs(q1).max()
    for a, b in zip(out[0][2:], out[1][2:]):                # mean and variance of xi, itself about 1
        assert np.abs(a - b).max() <= 1e-12
    assert not np.array_equal(p4, p1)                       # two forms ran: their roundings differ


@pytest.mark.parametrize("name", list(SURF))
def test_four_lane_forces_match_oracle_in_every_branch(name):
    """Compressed and stretched geometries, every atom in turn moved away (H3's
    compact terms on one, two and three distances, OH3's switching factors
    past 37.6 bohr, where the reference's shared derivative stands in)."""
    surface, amu, ts = SURF[name]
    rng = np.random.default_rng(2)
    x = np.concatenate([ts * s + rng.normal(0.0, w, (24,) + ts.shape)
                        for s, w in ((1.0, 0.01), (1.0, 0.3), (0.5, 0.1), (0.35, 0.02), (2.5, 0.3))])
    for a in range(len(ts)):
        for d in (6.0, 30.0, 45.0):
            y = ts + rng.normal(0.0, 0.05, (4,) + ts.shape)
            y[:, a, 0] += d
            x = np.concatenate([x, y])
    n = len(x) // 4 * 4
    with cam.RPMDEngine(surface, 4, n // 4, 1.0, cam.mass_au(amu)) as e:
        e.set_state(x[:n].reshape(-1, 4, len(ts), 3), np.zeros((n // 4, 4, len(ts), 3)))
        v, g = (t.reshape((n,) + t.shape[2:]) for t in e.get_forces())
    vr, gr = getattr(ol, "egrad_" + name)(x[:n])
    # O3: at half the bond lengths its polynomial terms, tenth powers of
    # variables up to 3 with coefficients up to 1e5 kcal/mol, reach 1e9
    # kcal/mol: an epsilon of that is 3e-10 hartree
    tol = 3e-9 if name == "o3" else 1e-12
    np.testing.assert_allclose(v, vr, rtol=tol, atol=tol)
    assert np.all(np.abs(g - gr).reshape(n, -1).max(1) <= tol * np.maximum(1.0, np.abs(gr).reshape(n, -1).max(1)))
