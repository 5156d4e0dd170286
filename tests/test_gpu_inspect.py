"""inspect_velocity over one and many workgroups, with ties (lowest index) and sizes
at the edges of waves, blocks and the grid's limit; and the passes that store only
what changed.  The maximum is one division of one root: equal to numpy's
to the bit; the boundary passes copy or clip, exact."""
import numpy as np
import pytest

import particlebase_amd as pb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 257, 131071, 131073, 700001])
def test_inspect_sizes(ctx, n):
    print(f"\n[case] inspect_velocity n={n}", flush=True)
    rng = np.random.default_rng(n)
    v = rng.normal(size=(n, 3))
    s = pb.System(ctx, [n])
    s.set_cell(np.array([0.0, 1.0] * 3))
    s.import_particles(rng.uniform(size=(n, 3)), np.ones(n), v=v)
    for fast in ({n - 1}, {0, n // 2, n - 1}, {n // 3}):
        w = v.copy()
        w[list(fast)] = (60.0, 0.0, 0.0)
        s.set("v", w)
        for _ in range(2):
            res, ratio, imax = s.inspect_velocity(100.0, 0.7, 0.2)
            assert (res, ratio, imax) == (0, 0.6, min(fast))


@pytest.mark.parametrize("n", [1, 65, 40000])
def test_boundaries_store_changes(ctx, n):
    print(f"\n[case] absolute / reflecting boundary, leap-frog with fixed particles n={n}", flush=True)
    rng = np.random.default_rng(n)
    r = rng.uniform(-0.02, 1.02, (n, 3))
    r[n // 2:] = np.clip(r[n // 2:], 0.1, 0.9)          # whole wavefronts inside
    v = rng.normal(size=(n, 3))
    fixed = (np.arange(n) % 200 < 90).astype(np.uint8)
    s = pb.System(ctx, [n])
    s.set_cell(np.array([0.0, 1.0] * 3))
    s.import_particles(r, np.ones(n), v=v, is_fixed=fixed)
    s.treat_reflect()
    want = np.where(r < 0, np.abs(v), np.where(r > 1, -np.abs(v), v))
    assert np.array_equal(s.get("v"), want)
    s.set("v", v)
    s.treat_absolute()
    assert np.array_equal(s.get("r"), np.clip(r, 0.0, 1.0))
    s.set("r", r)
    s.clear_force(True)
    s.add_force(2, 3.0)
    s.calc_acceleration()
    s.lf_step(0.25)
    move = (1.0 - fixed)[:, None]
    vn = v + 0.25 * np.array([0.0, 0.0, 3.0]) * move
    assert np.array_equal(s.get("v"), vn)
    assert np.abs(s.get("r") - (r + 0.25 * vn * move)).max() <= 4e-16 * (1 + np.abs(vn).max())
