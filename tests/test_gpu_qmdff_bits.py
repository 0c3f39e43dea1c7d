"""QMDFF gradients and box trajectories against recorded ones, bit for bit.

The kernels may be arranged in any way, but an atom's terms are added in the
order, and with the operations, of lanes that walk the atoms one after the
other.  The reference's torsion divides by sin(phi): next to planar it makes
one rounding of a position 1e-9 of the momenta within 50 steps, so a
trajectory repeats only if every force, and every sum of the box step, does.
The record is of such kernels (golden/make_qmdff_bits.py)."""
import os
import sys

import numpy as np
import pytest

import caracal_amd as cam

sys.path.append(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden"))
import make_qmdff_bits as mk

pytestmark = pytest.mark.gpu
RECORD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "qmdff_bits.npz")


@pytest.mark.parametrize("name", sorted(mk.FORCES))
@pytest.mark.parametrize("tag,precision", [("fp64", cam.CAM_PREC_FP64), ("mixed", cam.CAM_PREC_MIXED)])
def test_gradients_are_the_recorded_ones(name, tag, precision):
    p, xs = mk.force_inputs(name)
    g = mk.forces(p, xs, precision)
    r = np.load(RECORD)[f"g_{name}_{tag}"]
    print(f"{name} {tag}: {(g != r).sum()} of {g.size} differ, by at most {np.abs(g - r).max():.1e}", flush=True)
    assert np.array_equal(g, r)


def test_trajectory_is_the_recorded_one():
    """Nose-Hoover chain, wrap and transrot; and the same cut into runs."""
    r = np.load(RECORD)
    for cuts in ((mk.STEPS,), (7, mk.STEPS - 7)):
        q, p = mk.trajectory(True, True, cuts)
        print(f"runs of {cuts}: {(q != r['q']).sum()} positions, {(p != r['p']).sum()} momenta differ", flush=True)
        assert np.array_equal(q, r["q"]) and np.array_equal(p, r["p"])


@pytest.mark.parametrize("transrot", [False, True])
def test_a_run_may_be_cut_anywhere(transrot):
    """The kinetic energy of the chain is the same sum whichever kernel left
    it: at the start of a run, after the kick, after transrot or the scaling.
    A stiff chain (one step's time) shows a last bit of it within 40 steps."""
    whole = mk.trajectory(True, transrot, (40,), nose_steps=1)
    cut = mk.trajectory(True, transrot, (1,) * 40, nose_steps=1)
    assert np.array_equal(whole[0], cut[0]) and np.array_equal(whole[1], cut[1])
