"""MIXED energies and virials at every number of lanes a particle, one and two
types, in thin replicas too, against the oracle on the same positions.  Pair
energies are FP32: with A and B the sums of 4 eps (s/r)^12 and 4 eps (s/r)^6, both
known from the oracle's energy A - B and virial 6 (2A - B) (no shift), a pair's
relative errors (1/r^2 within 2 units of 2^-24, cubed, a few products: 10 units)
and a lane's running sum of at most 80 terms give 90 2^-24 (2A + B) for the energy
and 6 times 90 2^-24 (4A + B) for the virial.  Kinetic energy: velocities half a
step on, forces to 1e-5 of 1e2 rms, dt/2 = 5e-4, speeds of 1: 1e-6 relative."""
import numpy as np
import pytest

import particlebase_amd as pb
from particlebase_amd import workloads

pytestmark = pytest.mark.gpu
RC2 = 6.25
SE = {1: [1.0, 1.0], 2: [1.0, 1.0, 0.9, 0.7, 0.9, 0.7, 0.8, 0.5]}


# 8, 4, 2 lanes and one lane a particle; replicas thinner than three cells
@pytest.mark.parametrize("sizes", [(700,), (6145,), (32769,), (98305,), (300, 900, 2000)])
@pytest.mark.parametrize("nt", [1, 2])
def test_first_record(ctx, orc, sizes, nt):
    print(f"\n[case] mixed energies, sizes={sizes}, types={nt}", flush=True)
    ws = []
    for n in sizes:
        w = workloads.lj_fcc(int(np.ceil((n / 4) ** (1 / 3) - 1e-12)), 0.8, 0.72, seed=n % 83, natoms=n)
        w.r = w.r + 0.03 * workloads.normals(n % 79, 3 * n).reshape(n, 3)
        w.type = (np.arange(n) % 5 == 0).astype(np.uint32) * (nt - 1)
        ws.append(w)
    s = pb.System(ctx, list(sizes))
    s.set_cell(np.concatenate([w.cell for w in ws]))
    s.import_particles(np.concatenate([w.r for w in ws]), np.concatenate([w.m for w in ws]),
                       v=np.concatenate([w.v for w in ws]), type=np.concatenate([w.type for w in ws]))
    s.lj_set_params(np.asarray(SE[nt]), nt)
    s.lj_set_cutoff(RC2, shifted=False)
    s.clear_force(True)
    e, _ = s.lj_run(0.001, 2, precision=pb.PB_MIXED, skin=0.3, rebuild_every=5, energy_every=1)
    s.close()
    p = orc.lj_params(np.asarray(SE[nt]), nt, RC2, False)
    u = 90 * 2.0 ** -24
    for q, w in enumerate(ws):
        r = orc.wrap(w.r, w.cell).reshape(-1, 3)
        force = orc.lj_forces_brute if w.L < 7.6 else orc.lj_forces_cells
        F, pe, vir = force(r, w.type, w.cell, RC2, p)
        A, B = vir / 6 - pe, vir / 6 - 2 * pe
        assert A > 0 and B > 0
        v = w.v + F * (0.5 * 0.001 / w.m)[:, None]
        ke, pg, vg = np.asarray(e)[0, q]
        assert ke == pytest.approx(0.5 * (w.m[:, None] * v * v).sum(), rel=1e-6)
        assert abs(pg - pe) < u * (2 * A + B), (q, pg, pe)
        assert abs(vg - vir) < 6 * u * (4 * A + B), (q, vg, vir)
