"""Fused runs whose windows exceed the LDS stage (16-bit rows, candidates and pairs
read from memory) at every number of lanes a particle, with the short and the long
pair bodies, against the oracle's loop.  A cube of spacing 0.4 in a larger box,
cutoff 1.5 + skin 0.3: 91 particles a list cell, 4000 and more in the smallest
window (the stage holds 2816).  FP64: sums of about 220 terms of order 1 over six
steps of 0.0005 with dF/dr up to 1e2: 1e-11 on r and v, energies to 1e-11 of the
largest.  MIXED: pair forces to 1e-6 of about 1, 220 of them, 0.003 of time: 1e-6
on v, 1e-8 on r."""
import numpy as np
import pytest

import particlebase_amd as pb
from particlebase_amd import workloads

pytestmark = pytest.mark.gpu
RC2, DT, STEPS = 2.25, 0.0005, 6
ONE = ([0.33, 0.05], 1)
TWO = ([0.33, 0.05, 0.31, 0.04, 0.31, 0.04, 0.30, 0.03], 2)


# 8, 4, 2 lanes and one lane a particle
@pytest.mark.parametrize("n", [3000, 20000, 40000, 99000])
@pytest.mark.parametrize("se,prec,every", [(ONE, pb.PB_FP64, 0), (TWO, pb.PB_FP64, 1),
                                           (ONE, pb.PB_MIXED, 0), (TWO, pb.PB_MIXED, 0)])
def test_dense_cluster(ctx, orc, n, se, prec, every):
    print(f"\n[case] unstaged windows n={n} types={se[1]} prec={prec} energies={every}", flush=True)
    k = int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(k)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    r = 0.4 * g + 3.0 + 1e-3 * workloads.normals(8, 3 * n).reshape(n, 3)
    v = 0.1 * workloads.normals(9, 3 * n).reshape(n, 3)
    ty = (np.arange(n) % se[1]).astype(np.uint32)
    cell = np.array([0, 0.4 * k + 30.0] * 3)
    s = pb.System(ctx, [n])
    s.set_cell(cell)
    s.import_particles(r, np.ones(n), v=v, type=ty)
    s.lj_set_params(np.asarray(se[0]), se[1])
    s.lj_set_cutoff(RC2, shifted=True)
    s.clear_force(True)
    e, _ = s.lj_run(DT, STEPS, precision=prec, skin=0.3, rebuild_every=3, energy_every=every)
    rg, vg = s.get("r"), s.get("v")
    s.close()
    p = orc.lj_params(np.asarray(se[0]), se[1], RC2, True)
    f, eo = np.zeros_like(r), []
    for _ in range(STEPS):
        F, pe, vir = orc.lj_forces_cells(r, ty, cell, RC2, p)
        v = v + (F + f) * (0.5 * DT)
        eo.append([0.5 * (v * v).sum(), pe, vir])
        r, f = r + v * DT + F * (0.5 * DT ** 2), F
    rtol, vtol = (1e-11, 1e-11) if prec == pb.PB_FP64 else (1e-8, 1e-6)
    assert np.abs(rg - r).max() < rtol and np.abs(vg - v).max() < vtol
    if every:
        assert np.abs(np.asarray(e)[:, 0] - eo).max() < 1e-11 * np.abs(eo).max()
