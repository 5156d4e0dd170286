"""SPH passes where the number of lanes a particle changes (8, 4, 2, 1 by the
particles and the physics): copies of one block, moved by exact distances, with
thin and dense parts (windows of one to several hundred candidates, hit lists
worked off several times), against the oracle for one copy.  The sums are of at
most 512 terms in FP64: the tolerances of the other tests of this path (1e-11
relative on densities, 1e-9 B on pressures, 1e-9 of max|a|) leave them five digits."""
import numpy as np
import pytest

import particlebase_amd as pb

pytestmark = pytest.mark.gpu
H, N0, PITCH = 0.25, 512, 2.0
TAIT_B = 1.0 * 10.0 ** 2 / 7


def block():
    """512 particles of the unit cube: a third in a clump, a sheet, the rest loose."""
    rng = np.random.default_rng(12)
    r = rng.uniform(0.0, 1.0, (N0, 3))
    r[:170] = 0.45 + 0.1 * r[:170]
    r[170:250, 2] = 0.02
    return np.round(r * 2 ** 20) / 2 ** 20, rng


@pytest.mark.parametrize("physics", ["lucy", "config"])
@pytest.mark.parametrize("n", [1, 512, 24576, 24577, 49152, 49153, 98304, 98305, 131072, 131073])
def test_lane_counts(ctx, orc, physics, n):
    print(f"\n[case] SPH {physics} n={n}", flush=True)
    r0, rng = block()
    v0, m0 = rng.normal(scale=0.1, size=(N0, 3)), rng.uniform(0.5, 1.5, N0) * 1e-2
    mu0, c0 = rng.uniform(0.01, 0.1, N0), rng.uniform(1.0, 2.0, N0)
    copies, single = n // N0, n % N0                       # single: one particle by itself
    g = int(np.ceil((copies + 1) ** (1 / 3)))
    at = PITCH * np.stack(np.unravel_index(np.arange(copies + single), (g, g, g)), 1)
    x = np.concatenate([(r0[None] + at[:copies, None]).reshape(-1, 3), 0.5 + at[copies:]])
    tile = lambda f: np.concatenate([np.tile(f, (copies,) + (1,) * (f.ndim - 1)), f[:single]])
    s = pb.System(ctx, [n])
    s.set_cell(np.array([-0.5, PITCH * g] * 3))
    s.import_particles(x, tile(m0), v=tile(v0))
    if physics == "lucy":
        s.sph_set_properties(tile(mu0), tile(c0), H)
        s.setup_cells(H, periodic=False)
    else:
        s.sph_set_wcsph(H, 1.0, 10.0, 7.0, 0.1, 0.0)
        s.setup_cells(2 * H, periodic=False)
    s.bin()
    s.sph_density()
    s.sph_acceleration()
    num, rhoinv, a = s.get("sph_num"), s.get("sph_rhoinv"), s.get("a")

    def oracle(r, v, m, mu, c):
        if physics == "lucy":
            no, ro = orc.sph_density(r, m, mu, H)
            return no, ro, orc.sph_accel(r, v, m, c ** 2, ro, no[:, 2], H)
        no, ro = orc.wc_density(r, m, H, 1.0, 10.0, 7.0, 0.0)
        return no, ro, orc.wc_accel(r, v, m, no[:, 1], no[:, 2], H, 10.0, 0.1)

    parts = []
    if copies:
        parts.append((slice(0, copies * N0), oracle(r0, v0, m0, mu0, c0)))
    if single:
        parts.append((slice(copies * N0, n), oracle(x[-1:], v0[:1], m0[:1], mu0[:1], c0[:1])))
    for where, (no, ro, ao) in parts:
        for got, want, atol in ((num[where, 0], no[:, 0], 0), (num[where, 1], no[:, 1], 0),
                                (num[where, 2], no[:, 2], TAIT_B * 1e-9), (rhoinv[where], ro, 0)):
            assert np.allclose(got.reshape(-1, len(r0) if len(want) > 1 else 1), want, rtol=1e-11,
                               atol=atol if physics == "config" else 0)
        assert np.abs(a[where].reshape((-1,) + ao.shape) - ao).max() <= 1e-9 * np.abs(ao).max()
