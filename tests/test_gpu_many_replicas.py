"""More replicas than the pinned results hold (2046 in a force evaluation, 2048 in a
reduction): forces, energies, virials and kinetic energies of 2046, 2047, 2048 and
2049 replicas of 20 to 43 particles.  FP64: 1e-12 of the sums' terms, bounded here
by 1e-11 of the largest value over the replicas."""
import numpy as np
import pytest

import particlebase_amd as pb
from particlebase_amd import workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nrep", [2046, 2047, 2048, 2049])
def test_force_and_sums(ctx, orc, nrep):
    print(f"\n[case] {nrep} replicas", flush=True)
    kinds = []
    for k in range(24):                      # every replica is one of 24 kinds
        w = workloads.lj_fcc(3, 0.5, 0.9, seed=k, natoms=20 + k)
        w.r = w.r + 0.03 * workloads.normals(k + 50, 3 * w.n).reshape(w.n, 3)
        kinds.append(w)
    ws = [kinds[q * 7 % 24] for q in range(nrep)]
    s = pb.System(ctx, [w.n for w in ws])
    s.set_cell(np.concatenate([w.cell for w in ws]))
    s.import_particles(np.concatenate([w.r for w in ws]), np.concatenate([w.m for w in ws]),
                       v=np.concatenate([w.v for w in ws]))
    rc2 = min(w.L for w in kinds) ** 2 / 4.01
    s.lj_set_params([1.0, 1.0], 1)
    s.lj_set_cutoff(rc2, shifted=True)
    pe, vir = s.lj_force(pb.PB_FP64)
    F, mv2 = s.get("F"), np.asarray(s.mv2())
    s.close()
    p = orc.lj_params([1.0, 1.0], 1, rc2, True)
    want = {}
    for w in kinds:
        Fo, peo, wo = orc.lj_forces_brute(orc.wrap(w.r, w.cell).reshape(-1, 3), w.type, w.cell, rc2, p)
        want[id(w)] = Fo, peo, wo, (w.m[:, None] * w.v * w.v).sum()
    top = [max(np.abs(x[c]).max() for x in want.values()) for c in range(4)]
    at = 0
    for q, w in enumerate(ws):
        got = F[at:at + w.n], pe[q], vir[q], mv2[q]
        for c in range(4):
            assert np.abs(got[c] - want[id(w)][c]).max() <= 1e-11 * top[c], (q, c)
        at += w.n
