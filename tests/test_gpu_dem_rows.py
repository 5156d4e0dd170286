"""Rows of the contact matrix at the lengths where their treatment changes (0, 1,
8, 9, 16 contacts in registers, 17 and 40 in memory), against the oracle: CSR bit
for bit, forces, torques and history of both laws, over calls in which contacts
stay, go and come, and the matrix outgrows its arrays.  FP64 on both sides, sums
of at most 40 terms: 1e-11 of the largest, as for the other contact tests."""
import numpy as np
import pytest

import particlebase_amd as pb

pytestmark = pytest.mark.gpu
E, MU, SIG, MU_R = 2.0e5, 0.4, 0.29, 0.1
S2 = (2 - SIG) / 2 / (1 - SIG)
G2 = -np.log(0.8) / np.sqrt(np.pi ** 2 + np.log(0.8) ** 2) * 2
LENGTHS = (0, 1, 8, 9, 16, 17, 40)
BIG, SMALL, PITCH = 2.0, 0.2, 6.0


def flowers(seed, touching):
    """A large sphere of each length with small ones around it; `touching` of them
    touch, the others stand off by one small diameter.  Shuffled order."""
    rng = np.random.default_rng(seed)
    r, rad = [], []
    for c, m in enumerate(LENGTHS):
        o = np.array([3.0 + PITCH * c, 3.0, 3.0])
        r.append(o)
        rad.append(BIG)
        k = np.arange(m) + 0.5
        th, z = np.pi * (1 + 5 ** 0.5) * k, 1 - 2 * k / max(m, 1)
        rho = np.sqrt(1 - z * z)
        d = np.where(np.arange(m) < touching * m, 0.99, 1.2)[:, None] * (BIG + SMALL)
        r.extend(o + d * np.stack([rho * np.cos(th), rho * np.sin(th), z], 1))
        rad.extend([SMALL] * m)
    order = np.random.default_rng(77).permutation(len(r))
    r, rad = np.array(r)[order], np.array(rad)[order]
    return r + rng.uniform(-1e-3, 1e-3, r.shape), rad


@pytest.mark.parametrize("law", [0, 1])
def test_row_lengths(ctx, orc, law):
    print(f"\n[case] contact rows of {LENGTHS}, law {law}", flush=True)
    rng = np.random.default_rng(3)
    x, rad = flowers(0, 0.5)
    n = len(rad)
    m, move = rng.uniform(0.5, 2.0, n), np.ones(n, np.uint8)
    v, w = rng.normal(scale=0.2, size=(n, 3)), rng.normal(scale=0.5, size=(n, 3))
    s = pb.System(ctx, [n])
    s.set_cell(np.array([0.0, PITCH * len(LENGTHS), 0.0, 13.0, 0.0, 13.0]))
    s.import_particles(x, m, v=v)
    kn, kt = 1e4, 2e4 / 7
    if law:
        s.dem_set_linear(kn, 0.8, kt, MU, rad)
    else:
        s.dem_set_properties(E, MU, SIG, G2, MU_R, rad)
    s.rot_set_inertia(rad)
    s.setup_cells(2 * rad.max(), periodic=False)
    s.set("w", w)
    width, dt = (3, 1e-4) if law else (1, 1e-4)
    prow = pcol = pval = None
    for call, touching in enumerate((0.5, 1.0, 1.0, 0.0, 1.0)):
        x, _ = flowers(call, touching)
        s.set("r", x)
        s.bin()
        nnz = s.dem_calc_force(dt, autotune=True)
        row, col, val = s.dem_contacts()
        orow, ocol = orc.dem_contacts(x, rad, move)
        assert nnz == len(ocol) and np.array_equal(row, orow) and np.array_equal(col, ocol), call
        if touching == 1.0:
            assert set(LENGTHS) <= set(np.diff(orow))
        h = np.zeros((nnz, width))
        if prow is not None:
            h = orc.dem_carry_w(prow, pcol, pval, orow, ocol, width).reshape(-1, width)
        if law:
            F, T, h, _ = orc.dem_force_lsd(x, v, w, rad, 1 / m, move, orow, ocol, h, kn,
                                           orc.lsd_zeta(0.8), kt, MU, dt)
        else:
            F, T, h, _ = orc.dem_force(x, v, w, rad, 1 / m, move, orow, ocol, h[:, 0],
                                       E * (1 - SIG ** 2), MU, S2, G2, MU_R, dt)
        for got, want in ((s.get("F"), F), (s.get("T"), T), (val.ravel(), np.ravel(h))):
            if want.size:
                assert np.abs(got - want).max() <= 1e-11 * np.abs(want).max(), call
        prow, pcol, pval = orow, ocol, h


@pytest.mark.parametrize("scale", [1e-20, 1.0, 1e19])
@pytest.mark.parametrize("single", [False, True])
def test_contacts_beyond_fp32(ctx, orc, scale, single):
    """Contacts of particles outside the grid (binned into its edge cells), and at
    scales whose squares leave FP32: the CSR bit for bit."""
    print(f"\n[case] contacts outside the grid, scale {scale}, 125 cells {single}", flush=True)
    rng = np.random.default_rng(6)
    if single:                                # at most one particle a cell of the grid
        g = (np.arange(8) + 0.5) * 0.98
        x = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
        x += rng.uniform(-5e-3, 5e-3, x.shape)
        rad, box = np.full(len(x), 0.5), 8 * 0.98
    else:
        x, box = rng.uniform(0.0, 8.0, (800, 3)), 8.0
        rad = rng.uniform(0.4, 0.6, len(x))
    far = [(1e3, 4.0, 4.0), (1e3, 4.3, 4.0), (-40.0, -40.0, -40.0), (4.0, 4.0, 1e9), (4.0, 4.4, 1e9)]
    x = np.concatenate([x, far]) * scale
    rad = np.concatenate([rad, np.full(len(far), 0.5)]) * scale
    n = len(x)
    s = pb.System(ctx, [n])
    s.set_cell(np.array([0.0, box, 0.0, box, 0.0, box]) * scale)
    s.import_particles(x, np.ones(n))
    s.dem_set_properties(E, MU, SIG, G2, MU_R, rad)
    s.rot_set_inertia(rad)
    s.setup_cells(scale * (2 * 0.5 / np.sqrt(3.0) if single else 1.2), periodic=False,
                  single_particle=single)
    s.bin()
    nnz = s.dem_calc_force(1e-9, autotune=True)
    row, col, _ = s.dem_contacts()
    orow, ocol = orc.dem_contacts(x, rad, np.ones(n, np.uint8))
    assert nnz == len(ocol) and np.array_equal(row, orow) and np.array_equal(col, ocol)
    assert np.diff(orow)[-2:].tolist() == [1, 1]        # a pair outside touches
