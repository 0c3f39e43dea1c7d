"""The box engine's step kernels with the work of their neighbours in them --
the periodic wrap and the Nose-Hoover factor in the normal-mode step, the
kinetic energy in the kick, transrot and the scaling -- at the edges: one bead,
beads of one column over several waves, a last block with idle columns, atoms
whose beads straddle a face (several shifts of one atom in one step) and atoms
that start boxes away, each thermostat and transrot switch, against the oracle.

The steps are sums of at most a few hundred terms and the wrap is exact but for
one rounding of a position per shift; 1e-11 of the largest position and 1e-9 of
the largest momentum are the bounds of the engine's other oracle tests."""
import numpy as np
import pytest

import caracal_amd as cam
import oracle_lib as ol
from box_oracle import BoxRPMD, QmdffFF
from caracal_amd import ff as cff
from caracal_amd.units import mass_au
from test_gpu_qmdff import AMU
from test_gpu_qmdff_terms import _subset

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nmol,nb,nose,transrot", [
    (2, 1, True, True),
    (3, 4, False, True),
    (3, 16, True, False),
    (2, 64, True, True),
    (2, 128, False, False),
    (2, 256, True, True),
    (30, 4, True, True),       # 1080 (bead, atom) pairs: several blocks of every sum
])
def test_box_steps_match_the_oracle(nmol, nb, nose, transrot):
    p, x = _subset(nmol)
    box = np.asarray(p["box"])
    rng = np.random.default_rng(nb)
    x = x - x[0]                                    # an atom on the corner: its beads straddle three faces
    x = x + (rng.integers(-2, 3, (nmol, 3)) * box)[np.asarray(p["molnum"]).astype(int) - 1]
    xs = x[None] + rng.normal(0.0, 0.02, (nb,) + x.shape)
    m = mass_au([AMU[int(z)] for z in p["at"]])
    beta = float(cam.beta_of(200.0))
    dt = 0.5 * cam.FS_TO_AU
    pm = rng.normal(size=xs.shape) * np.sqrt(m[None, :, None] * nb / beta)
    nose_q = 20 * dt if nose else 0.0
    steps = 3
    ff = cff.ForceField.qmdff(p)
    eng = cff.BoxEngine(ff, nb, dt, m, beta, None, precision=cam.CAM_PREC_FP64, nm_mode=cam.CAM_NM_REFERENCE)
    if nose:
        eng.set_nhc(nose_q)
    if transrot:
        eng.set_transrot(True)
    eng.set_state(xs, pm)
    eng.run(1)
    eng.run(steps - 1)
    q, pq = eng.get_state()
    eng.close()
    ff.close()
    ref = BoxRPMD(QmdffFF(ol.QmdffOracle(p)), np.zeros(10), xs, pm, dt, m, beta, nose_q=nose_q, wrap_box=p["box"],
                  remove_com=transrot)
    moved = 0
    for _ in range(steps):
        before = ref.q.copy()
        ref.step()
        moved += int((np.abs(ref.q - before).max(axis=0) > 0.5 * box).sum())
    err = np.abs(q - ref.q).max() / np.abs(ref.q).max()
    perr = np.abs(pq - ref.p).max() / np.abs(ref.p).max()
    print(f"{len(x)} atoms, {nb} beads: {moved} coordinates moved, rel dq {err:.1e}, dp {perr:.1e}", flush=True)
    assert moved > 0
    assert err <= 1e-11 and perr <= 1e-9
