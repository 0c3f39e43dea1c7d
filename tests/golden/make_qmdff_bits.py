"""Writes qmdff_bits.npz: QMDFF gradients and trajectories of the loaded
library, bit for bit.

    python make_qmdff_bits.py [output.npz]

The committed file was written on an MI355X by the kernels that walk the atoms
one after the other (commit 4a86d16); tests/test_gpu_qmdff_bits.py compares
every later arrangement of the same sums with it."""
import os
import sys

HERE = os.path.dirname(os.path.abspath(__file__))

import numpy as np
import torch

import caracal_amd as cam
from caracal_amd import ff as cff
from caracal_amd.units import mass_au

sys.path.append(os.path.dirname(HERE))
import qmdff_fixtures as qf
from test_gpu_qmdff_terms import _subset

# name: molecules, periodic, Zahn electrostatics, whole molecules some boxes away, beads
FORCES = {
    "liquid": (29, 1, 0, False, 2),
    "zahn_away": (29, 1, 1, True, 1),
    "cluster": (9, 0, 0, False, 2),
}
MASS = {1: 1.008, 6: 12.011, 8: 15.999}
NMOL, NBEADS, STEPS = 16, 4, 20


def force_inputs(name):
    nmol, periodic, zahn, away, nb = FORCES[name]
    p, x = _subset(nmol)
    p["periodic"], p["zahn"] = periodic, zahn
    rng = np.random.default_rng(11)
    xs = x[None] + rng.normal(0.0, 0.03, (nb,) + x.shape)
    if away:
        mol = np.asarray(p["molnum"]).astype(int) - 1
        xs = xs + (rng.integers(-2, 3, (nmol, 3)) * np.asarray(p["box"]))[mol][None]
    return p, np.ascontiguousarray(xs)


def forces(p, xs, precision):
    """Gradient of every bead."""
    ff = cff.ForceField.qmdff(p)
    g = ff.forces(None, torch.tensor(xs, device="cuda"), precision=precision)[1].cpu().numpy()
    ff.close()
    return g


def trajectory(nose, transrot, cuts, precision=cam.CAM_PREC_FP64, nmol=NMOL, nbeads=NBEADS, nose_steps=20):
    """q and p after runs of the given lengths of a box."""
    p, x = _subset(nmol)
    rng = np.random.default_rng(5)
    xs = x[None] + rng.normal(0.0, 0.02, (nbeads,) + x.shape)
    m = mass_au([MASS[int(z)] for z in p["at"]])
    beta, dt = float(cam.beta_of(200.0)), 0.5 * cam.FS_TO_AU
    ff = cff.ForceField.qmdff(p)
    eng = cff.BoxEngine(ff, nbeads, dt, m, beta, None, precision=precision)
    if nose:
        eng.set_nhc(nose_steps * dt)
    if transrot:
        eng.set_transrot(True)
    eng.set_state(xs, rng.normal(size=xs.shape) * np.sqrt(m[None, :, None] * nbeads / beta))
    for n in cuts:
        eng.run(n)
    q, pm = eng.get_state()
    eng.close()
    ff.close()
    return q, pm


if __name__ == "__main__":
    out = {}
    for name in FORCES:
        p, xs = force_inputs(name)
        for tag, prec in (("fp64", cam.CAM_PREC_FP64), ("mixed", cam.CAM_PREC_MIXED)):
            out[f"g_{name}_{tag}"] = forces(p, xs, prec)
    out["q"], out["p"] = trajectory(True, True, (STEPS,))
    np.savez_compressed(sys.argv[1] if len(sys.argv) > 1 else os.path.join(HERE, "qmdff_bits.npz"), **out)
