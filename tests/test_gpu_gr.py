"""g(r) histograms against the oracle, bin by bin, where the kernel's shortcut
and its work split can go wrong: distances exactly on bin boundaries (lattice),
edges of the 256-particle tiles and of the slices they are cut into, boxes with
unequal edges, particles outside the box (which void the shortcut's bound), a
single bin, the largest histogram, coarse and very fine bins, several replicas,
a particle that is not finite, and bins so fine that the bound covers several
of them.  Whole numbers: equality."""
import numpy as np
import pytest

import particlebase_amd as pb
from particlebase_amd import workloads

pytestmark = pytest.mark.gpu


def boxed(rng, n, L, lo=(0.0, 0.0, 0.0), spill=0.0):
    L, lo = np.asarray(L, float), np.asarray(lo, float)
    r = lo + (rng.random((n, 3)) * (1 + 2 * spill) - spill) * L
    return r.astype(np.float32), np.stack([lo, lo + L], 1).reshape(-1).astype(np.float32)


def lattice(n, a):
    k = int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(k)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n] * a
    return g.astype(np.float32), np.array([0, k * a] * 3, dtype=np.float32)


CASES = {
    # name: (systems, rstep or steps per half edge, bins)
    "lattice_on_boundaries": (lambda g: [lattice(1331, 1.0)], 0.25, 40),
    "lattice_half_steps": (lambda g: [lattice(1000, 2.0)], 4.0 / 3.0, 30),
    "tile_edges": (lambda g: [boxed(g, n, [12, 12, 12]) for n in (1, 2, 255, 256, 257, 512, 513)],
                   None, 200),
    "slices": (lambda g: [boxed(g, 3000, [30, 30, 30])], None, 127),
    "unequal_edges_shifted": (lambda g: [boxed(g, 1500, [9, 31, 74], (-40, 3, 500))], None, 333),
    "outside_the_box": (lambda g: [boxed(g, 1200, [20, 25, 20], spill=0.4),
                                   boxed(g, 700, [20, 25, 20])], None, 100),
    "one_bin": (lambda g: [boxed(g, 600, [15, 15, 15])], 3.0, 1),
    "largest_histogram": (lambda g: [boxed(g, 1100, [40, 40, 40])], None, 16384),
    "fine_beyond_the_bound": (lambda g: [boxed(g, 900, [50, 50, 50])], 1e-6, 4000),
    "coarse": (lambda g: [boxed(g, 900, [50, 50, 50])], 40.0, 5),
}


@pytest.mark.parametrize("name", CASES)
def test_gr_against_oracle(ctx, orc, name):
    print(f"\n[case] g(r) {name}", flush=True)
    make, rstep, rnum = CASES[name]
    systems = make(np.random.default_rng(sum(map(ord, name))))
    rsteps = np.array([np.float32(rstep if rstep else (c[1::2] - c[0::2]).max() / 2 / rnum)
                       for _, c in systems], dtype=np.float32)
    s = pb.System(ctx, [r.shape[0] for r, _ in systems])
    s.set_cell(np.concatenate([c for _, c in systems]).astype(np.float64))
    r = np.concatenate([r for r, _ in systems]).astype(np.float64)
    s.import_particles(r, np.ones(len(r)))
    h = s.gr_hist(rsteps, rnum)
    for k, (rk, c) in enumerate(systems):
        ri = np.float32(1.0 / np.float64(rsteps[k]))
        assert np.array_equal(h[k], orc.gr_hist_f32(rk, c, ri, rnum)), (name, k)
    s.close()


def test_gr_particle_not_finite(ctx):
    """Pairs with a particle that is not finite land in bin 0, as dropped pairs;
    the others are counted as without it."""
    print("\n[case] g(r) with a NaN and an infinite coordinate", flush=True)
    rng = np.random.default_rng(3)
    r, c = boxed(rng, 700, [20, 20, 20])
    hist = []
    for bad in (False, True):
        x = r.astype(np.float64)
        keep = np.ones(700, bool)
        keep[[10, 600]] = False
        if bad:
            x[10, 1], x[600, 2] = np.nan, np.inf
        else:
            x = x[keep]
        s = pb.System(ctx, [len(x)])
        s.set_cell(c.astype(np.float64))
        s.import_particles(x, np.ones(len(x)))
        hist.append(s.gr_hist(np.float32(0.05), 200)[0].astype(np.int64))
        s.close()
    assert np.array_equal(hist[0][1:], hist[1][1:])
    assert hist[1].sum() == 700 * 699 // 2
