"""The Gaussian step where its solves move into the kernels that need them (512
wavefronts of the largest replica) and back into kernels of their own, one and
several replicas, both exits of the loop's test: against the oracle's Newton loop.  Tolerances of the other tests of this step:
1e-13 of max|v| for one-pass exits, ten times the loop's tolerance for converged
ones."""
import numpy as np
import pytest

import particlebase_amd as pb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(1,), (64,), (65,), (32768,), (32769,), (40, 900, 200),
                                   (40, 32769, 200)])
@pytest.mark.parametrize("xi0,tol", [(0.07, 1e-10), (0.0, 1e-8)])
def test_solve_forms(ctx, orc, sizes, xi0, tol):
    print(f"\n[case] Gaussian step, replicas {sizes}, xi0={xi0}", flush=True)
    rng = np.random.default_rng(sum(sizes))
    n = sum(sizes)
    r, v, F = rng.uniform(0, 10, (n, 3)), rng.normal(size=(n, 3)), rng.normal(scale=3.0, size=(n, 3))
    Fold, m, dt = F + rng.normal(scale=0.3, size=(n, 3)), rng.uniform(0.5, 2.0, n), 0.01
    s = pb.System(ctx, list(sizes))
    s.set_cell(np.tile([0.0, 10.0] * 3, len(sizes)))
    s.import_particles(r, m, v=v, a=Fold)
    s.set("F", F)
    s.gt_xi(set_xi=[xi0] * len(sizes))
    s.gt_step(dt, tol)
    vg, rg, (xi, bad) = s.get("v"), s.get("r"), s.gt_xi()
    assert bad == 0
    at = 0
    for q, k in enumerate(sizes):
        c = slice(at, at + k)
        ro, vo, _, xio, it = orc.gt_step(r[c], v[c], F[c], Fold[c], 1 / m[c], dt, xi0, tol)
        assert it > 0
        vtol = 1e-13 if it == 1 else 10 * tol
        assert np.abs(vg[c] - vo).max() < vtol * np.abs(vo).max(), (q, it)
        assert xi[q] == pytest.approx(xio, rel=max(1e-12, 100 * tol), abs=1e-16)
        assert np.abs(rg[c] - ro).max() < max(1e-12, dt * vtol) * 10.0
        at += k
    s.close()
