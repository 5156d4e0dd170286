"""The step variants with long pair bodies (FP64 energies, several types), whose
pairs interleave two by two within the register cap, at every number of lanes a
particle, and their uncapped form where one replica is thinner than three cells:
trajectories and, in FP64, per-step energies of two-type fluids against the oracle's
loop.  FP64: 1e-11 as for the other runs.  MIXED: 1e-4 on positions after five steps
of 0.005 (pair forces to 1e-6 of about 1e2), ten times that on velocities."""
import numpy as np
import pytest

import particlebase_amd as pb
from test_gpu_lj_lanes import fluid, oracle_run, same, system

pytestmark = pytest.mark.gpu
SE = (1.0, 1.0, 0.9, 0.7, 0.9, 0.7, 0.8, 0.5)     # sigma, eps of (0,0) (0,1) (1,0) (1,1)


@pytest.mark.parametrize("prec", [pb.PB_FP64, pb.PB_MIXED])
@pytest.mark.parametrize("sizes", [(700,), (6145,), (32769,), (98305,), (300, 900)])
def test_two_types_energies(ctx, orc, sizes, prec):
    print(f"\n[case] two types, energies every step, sizes={sizes}, prec={prec}", flush=True)
    ws = [fluid(n, 0.8, n % 83) for n in sizes]
    for w in ws:
        w.type = (np.arange(w.n) % 5 == 0).astype(np.uint32)
    s = system(ctx, ws, SE, 2)
    e, _ = s.lj_run(0.005, 5, precision=prec, skin=0.3, rebuild_every=3, energy_every=1)
    r, v = s.get("r"), s.get("v")
    at = 0
    for q, w in enumerate(ws):
        ro, vo, eo = oracle_run(orc, w, 5, SE, 2)
        tol = 1e-11 if prec == pb.PB_FP64 else 1e-4
        assert same(r[at:at + w.n], ro, w.L) < tol
        assert np.abs(v[at:at + w.n] - vo).max() < 10 * tol
        if prec == pb.PB_FP64:
            assert np.abs(np.asarray(e)[:, q] - eo).max() < 1e-11 * np.abs(eo).max()
        at += w.n
    s.close()
