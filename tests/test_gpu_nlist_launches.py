"""Neighbour list and list forces of more rows than one launch takes (2^20): a
simple cubic lattice of 102^3 particles, 6 neighbours a row at distance 1.  Forces
vanish by symmetry (each pair's is 24 in size: 1e-12 allows for rounding of the
coordinates up to 102), the energy is 3 phi(1) a particle (1e6 terms: 1e-11)."""
import numpy as np
import pytest

import particlebase_amd as pb

pytestmark = pytest.mark.gpu


def test_lattice_of_two_launches(ctx):
    print("\n[case] neighbour list, lattice of 102^3", flush=True)
    k = 102
    g = np.stack(np.meshgrid(*[np.arange(k)] * 3, indexing="ij"), -1).reshape(-1, 3)
    n = len(g)
    s = pb.System(ctx, [n])
    s.set_cell([0, k] * 3)
    s.import_particles(g.astype(float), np.ones(n))
    s.setup_cells(1.2)
    s.bin()
    rc2 = np.float32(1.44)
    assert np.array_equal(s.coord_counts(rc2), np.full(n, 6))
    assert s.nlist_build(rc2) == 6 * n
    row, col = s.nlist_get()
    assert np.array_equal(row, 6 * np.arange(n + 1))
    want = np.sort(np.concatenate([(((g + d) % k) @ np.array([k * k, k, 1]))[:, None]
                                   for a in range(3) for d in (np.eye(3, dtype=int)[a],
                                                               -np.eye(3, dtype=int)[a])], 1), 1)
    assert np.array_equal(col.reshape(n, 6), want)
    s.lj_set_params([0.95, 1.0], 1)
    s.lj_set_cutoff(1.44, shifted=False)
    pe, vir = s.lj_force_nlist()
    s6 = 0.95 ** 6
    assert np.abs(s.get("F")).max() < 1e-12
    assert pe == pytest.approx(3 * n * 4 * s6 * (s6 - 1), rel=1e-11)
    assert vir == pytest.approx(3 * n * 24 * s6 * (2 * s6 - 1), rel=1e-11)
    s.close()
