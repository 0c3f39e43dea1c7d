"""The QMDFF terms kernel at the edges of its split: one wave per atom, four
atoms to a block, 64 candidate atoms at a time (eight of each eighth of the
atoms) from tiles of 256, accepted ones queued and evaluated 64 at a time.

Subsets of the ethanol box (9 atoms a molecule) around those sizes, with no,
some and every pair inside the cutoff, molecules displaced by whole boxes, both
electrostatics, one and several beads, FP64 and mixed, against the oracle.

Tolerances: an energy or gradient component is a sum of at most n terms whose
own relative error is below 1e-13 in FP64 (2 ulp exp and erfc) and 1e-6 in
binary32 (1 ulp quotient and root of a squared distance, times the exponent
8); terms of opposite sign cancel to no less than a hundredth of their size in
these liquids, so 1e-11 and 1e-4 of the largest component."""
import numpy as np
import pytest
import torch

import caracal_amd as cam
import oracle_lib as ol
import qmdff_fixtures as qf
from caracal_amd import ff as cff

pytestmark = pytest.mark.gpu


def _subset(nmol):
    """The first nmol molecules of the ethanol box, with its cell."""
    p, x = qf.ethanol_box()
    k = nmol / p["nmols"]
    n = int(round(p["natoms"] * k))
    p = dict(p)
    for name in ("bond", "vbond", "angl", "vangl", "tors", "vtors", "nci"):
        p[name] = p[name][:int(round(len(p[name]) * k))]
    for name in ("at", "q", "molnum"):
        p[name] = p[name][:n]
    p["c6xy"] = np.ascontiguousarray(p["c6xy"][:n, :n])
    p["natoms"], p["nmols"] = n, nmol
    return p, np.ascontiguousarray(x[:n])


@pytest.mark.parametrize("nmol,periodic,zahn,cut,nb", [
    (1, 1, 0, 1.0, 1),        # no other molecule: no intermolecular block
    (2, 1, 0, 1.0, 1),        # 18 atoms: one partly filled group of 64
    (2, 0, 0, 1.0, 3),
    (7, 1, 0, 1.0, 2),        # 63 and 72 atoms: either side of a group
    (8, 0, 1, 1.0, 2),
    (28, 1, 1, 1.0, 1),       # 252 and 261: either side of a tile
    (29, 1, 0, 1.0, 5),
    (29, 0, 0, 1.0, 1),       # every pair inside
    (57, 1, 0, 0.02, 2),      # 513 atoms; no pair inside
    (57, 1, 0, 1.3, 2),       # about half of them
])
def test_terms_at_the_edges_match_the_oracle(nmol, periodic, zahn, cut, nb):
    p, x = _subset(nmol)
    p["periodic"], p["zahn"] = periodic, zahn
    for k in ("vdw_cut", "coul_cut", "cut_low"):
        p[k] = float(p[k]) * cut
    rng = np.random.default_rng(nmol)
    xs = x[None] + rng.normal(0.0, 0.02, (nb,) + x.shape)
    if periodic:                                    # whole molecules, some boxes away
        mol = np.asarray(p["molnum"]).astype(int) - 1
        xs = xs + (rng.integers(-2, 3, (nmol, 3)) * np.asarray(p["box"]))[mol][None]
    ff = cff.ForceField.qmdff(p)
    res = {}
    for prec in (cam.CAM_PREC_FP64, cam.CAM_PREC_MIXED):
        e, g, _, _ = ff.forces(None, torch.tensor(np.ascontiguousarray(xs), device="cuda"), precision=prec)
        res[prec] = (e.cpu().numpy(), g.cpu().numpy())
    ff.close()
    o = ol.QmdffOracle(p)
    for b in range(nb):
        er, gr, _ = o.eval(xs[b])
        for prec, tol in ((cam.CAM_PREC_FP64, 1e-11), (cam.CAM_PREC_MIXED, 1e-4)):
            de = abs(res[prec][0][b] - er) / abs(er)
            dg = np.abs(res[prec][1][b] - gr).max() / np.abs(gr).max()
            print(f"{len(x)} atoms, bead {b}, precision {prec}: rel dE {de:.1e}, dg {dg:.1e}", flush=True)
            assert de <= tol and dg <= tol
