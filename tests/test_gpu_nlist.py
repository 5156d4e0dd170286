"""The neighbour list's wavefront rows where their forms change: rows longer
than the LDS row (512), pairs exactly at the list radius (a lattice), particles
up to a quarter box outside (beyond the range of the folded distance's bound),
grids of three cells along an axis (the wrap visits every cell once),
non-periodic grids, a list that outgrows the arrays of the one before, and list
forces of rows of 0, 1, 7, 8, 9 and hundreds of columns.  The CSR and the
counts equal the oracle's; forces to 1e-12 of the largest (sums of the same
terms in another order: a few hundred roundings of 1.1e-16)."""
import numpy as np
import pytest

import particlebase_amd as pb

pytestmark = pytest.mark.gpu


def build(ctx, r, cell, rmax, periodic=True):
    s = pb.System(ctx, [len(r)])
    s.set_cell(cell)
    s.import_particles(r, np.ones(len(r)))
    s.setup_cells(rmax, periodic=periodic)
    s.bin()
    return s


def box(L):
    return np.array([0, L[0], 0, L[1], 0, L[2]], dtype=float)


def cases():
    g = np.random.default_rng(17)
    k = np.stack(np.meshgrid(*[np.arange(12.0)] * 3, indexing="ij"), -1).reshape(-1, 3)
    spill = (g.random((2000, 3)) * 1.5 - 0.25) * 13.0
    return {"rows_over_512": (g.random((3900, 3)) * 9.0, box([9, 9, 9]), 3.0),
            "lattice_at_the_radius": (k, box([12, 12, 12]), 2.0),
            "outside_the_box": (spill, box([13, 13, 13]), 2.5),
            "three_cells": (g.random((700, 3)) * [7.6, 20, 7.7], box([7.6, 20, 7.7]), 2.5),
            "sparse": (g.random((300, 3)) * 30.0, box([30, 30, 30]), 2.0),
            "one_particle": (np.array([[1.0, 2.0, 3.0]]), box([9, 9, 9]), 3.0)}


@pytest.mark.parametrize("name", cases())
def test_rows_against_oracle(ctx, orc, name):
    print(f"\n[case] nlist {name}", flush=True)
    r, cell, rmax = cases()[name]
    rt2 = np.float32(rmax * rmax)
    s = build(ctx, r, cell, rmax)
    nnz = s.nlist_build(rt2)
    row, col = s.nlist_get()
    orow, ocol = orc.nlist_f32(r, cell, rmax, rt2)
    assert nnz == len(ocol)
    assert np.array_equal(row, orow) and np.array_equal(col, ocol)
    assert np.array_equal(s.coord_counts(rt2), np.diff(orow))
    s.close()


def test_outgrown_list(ctx, orc):
    print("\n[case] nlist rebuilt with a larger radius, then a smaller one", flush=True)
    r, cell, _ = cases()["sparse"]
    s = build(ctx, r, cell, 6.0)
    for rt in (2.0, 6.0, 3.0):
        s.nlist_build(np.float32(rt * rt))
        row, col = s.nlist_get()
        orow, ocol = orc.nlist_f32(r, cell, 6.0, np.float32(rt * rt))
        assert np.array_equal(row, orow) and np.array_equal(col, ocol)
    s.close()


def test_non_periodic_counts(ctx):
    print("\n[case] counts on a non-periodic grid against every pair", flush=True)
    g = np.random.default_rng(5)
    r = (g.random((900, 3)) * 4.0 + 3.0).astype(np.float32)     # far from the faces: no fold
    s = build(ctx, r.astype(float), box([10, 10, 10]), 1.5, periodic=False)
    d = r[:, None, :] - r[None, :, :]
    r2 = (d * d)[..., 0] + (d * d)[..., 1] + (d * d)[..., 2]    # FP32, the reference's order
    want = (r2 < np.float32(2.25)).sum(1) - 1
    assert np.array_equal(s.coord_counts(np.float32(2.25)), want)
    s.close()


@pytest.mark.parametrize("n", [1, 2, 65, 900])
def test_list_forces_row_lengths(ctx, orc, n):
    print(f"\n[case] list forces, {n} particles in one cluster of growing density", flush=True)
    g = np.random.default_rng(n)
    # spacing grows away from the origin, so row lengths run from 0 upwards
    k = np.stack(np.meshgrid(*[np.arange(10.0)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    r = 20.0 * (k / 10.0) ** 1.6 + 0.05 * g.random((n, 3)) + 1.0
    cell = box([30, 30, 30])
    s = build(ctx, r, cell, 3.0)
    s.lj_set_params([0.3, 1.0], 1)
    s.lj_set_cutoff(6.25, shifted=True)
    s.nlist_build(np.float32(9.0))
    row, col = s.nlist_get()
    pe, w = s.lj_force_nlist()
    F = s.get("F")
    p = orc.lj_params([0.3, 1.0], 1, 6.25, True)
    Fo, peo, wo = orc.lj_forces_list(r, np.zeros(n, np.uint32), cell, 6.25, p, row, col)
    assert np.abs(F - Fo.reshape(-1, 3)).max() <= 1e-12 * max(np.abs(Fo).max(), 1.0)
    assert abs(pe - peo) <= 1e-12 * max(abs(peo), 1.0) and abs(w - wo) <= 1e-12 * max(abs(wo), 1.0)
    s.close()
