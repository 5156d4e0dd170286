"""The fused run where the number of lanes a particle changes (8, 4, 2, 1 by the
particles of the system; one with the persistent option), where rows are shared
by the lanes: thin replicas with the minimum image, dense windows beyond the LDS
stage, several types, several replicas, graph replay, a continued list, and the
same list length reported by every form.  FP64 positions against the oracle's
loop over 10 steps to 1e-11 (each step rounds sums of about 60 terms to 1e-16
relative, amplified by less than e), energies to 1e-11."""
import numpy as np
import pytest

import particlebase_amd as pb
from particlebase_amd import workloads

pytestmark = pytest.mark.gpu
RC2 = 6.25


def fluid(n, rho, seed, jit=0.03):
    w = workloads.lj_fcc(int(np.ceil((n / 4) ** (1 / 3) - 1e-12)), rho, 0.72, seed=seed, natoms=n)
    w.r = w.r + jit * workloads.normals(seed + 9, 3 * n).reshape(n, 3)
    return w


def system(ctx, ws, se=(1.0, 1.0), nt=1):
    s = pb.System(ctx, [w.n for w in ws])
    s.set_cell(np.concatenate([w.cell for w in ws]))
    s.import_particles(np.concatenate([w.r for w in ws]), np.concatenate([w.m for w in ws]),
                       v=np.concatenate([w.v for w in ws]),
                       type=np.concatenate([w.type for w in ws]))
    s.lj_set_params(np.asarray(se, float), nt)
    s.lj_set_cutoff(RC2, shifted=True)
    s.clear_force(True)
    return s


def oracle_run(orc, w, steps, se=(1.0, 1.0), nt=1):
    p = orc.lj_params(np.asarray(se, float), nt, RC2, True)
    r, v, f = orc.wrap(w.r, w.cell).reshape(-1, 3), w.v.copy(), np.zeros_like(w.r)
    e = []
    minv = 1.0 / w.m
    force = orc.lj_forces_brute if min(w.cell[1::2]) < 7.6 else orc.lj_forces_cells
    for _ in range(steps):
        F, pe, vir = force(r, w.type, w.cell, RC2, p)
        v = v + (F + f) * (0.5 * 0.005 * minv)[:, None]
        e.append([0.5 * (w.m[:, None] * v * v).sum(), pe, vir])
        r = r + v * 0.005 + F * (0.5 * 0.005 ** 2 * minv)[:, None]
        f = F
        r = orc.wrap(r, w.cell).reshape(-1, 3)
    return r, v, np.array(e)


def same(a, b, L):
    d = a - b
    return np.abs(d - L * np.rint(d / L)).max()


# slots are whole wavefronts: 6144, 32768 and 98304 are the last of 8, 4, 2 lanes
@pytest.mark.parametrize("n", [700, 6144, 6145, 32768, 32769, 98304, 98305])
def test_run_lane_counts(ctx, orc, n):
    print(f"\n[case] run lanes n={n}", flush=True)
    w = fluid(n, 0.8442, n % 89)
    s = system(ctx, [w])
    e, _ = s.lj_run(0.005, 10, precision=pb.PB_FP64, skin=0.3, rebuild_every=4, energy_every=1)
    r, v, eo = oracle_run(orc, w, 10)
    assert same(s.get("r"), r, w.L) < 1e-11 and np.abs(s.get("v") - v).max() < 1e-11
    assert np.allclose(e[:, 0], eo, rtol=1e-11, atol=1e-7)
    nn = s.lj_run_stats()["max_nn"]
    # one lane (the persistent form) builds a list of the same pairs
    t = system(ctx, [w])
    t.lj_run(0.005, 10, precision=pb.PB_FP64, skin=0.3, rebuild_every=4, energy_every=0,
             persistent=True)
    assert t.lj_run_stats()["max_nn"] == nn
    assert same(t.get("r"), r, w.L) < 1e-11
    s.close()
    t.close()


@pytest.mark.parametrize("prec", [pb.PB_FP64, pb.PB_MIXED])
def test_thin_replicas_types_and_continued_list(ctx, orc, prec):
    print(f"\n[case] run lanes, thin replicas and three types, prec={prec}", flush=True)
    se = [1.0, 1.0, 1.02, 0.9, 0.97, 1.1, 1.02, 0.9, 1.04, 0.8, 0.99, 1.0, 0.97, 1.1, 0.99, 1.0,
          0.94, 1.2]
    ws = []
    for k, (n, rho) in enumerate([(260, 0.8), (500, 0.85), (1500, 0.7), (3000, 0.75)]):
        w = fluid(n, rho, 60 + k, 0.02)
        w.type = (np.arange(n) * 5 % 3).astype(np.uint32)
        ws.append(w)
    s = system(ctx, ws, se, 3)
    for steps in (3, 5):
        s.lj_run(0.005, steps, precision=prec, skin=0.3, rebuild_every=20, energy_every=0)
    r, v, at = s.get("r"), s.get("v"), 0
    # mixed: pair forces to 1e-6 of about 1e2, over 8 steps of 0.005
    tol = 1e-11 if prec == pb.PB_FP64 else 1e-4
    for w in ws:
        ro, vo, _ = oracle_run(orc, w, 8, se, 3)
        assert same(r[at:at + w.n], ro, w.L) < tol and np.abs(v[at:at + w.n] - vo).max() < tol
        at += w.n
    s.close()


@pytest.mark.parametrize("n", [3000, 20000])
def test_dense_cluster_and_graph(ctx, n):
    """Windows beyond the LDS stage (16-bit rows of global reads), run eagerly
    and as a replayed graph of the same schedule: the same bits."""
    print(f"\n[case] run lanes, dense cluster n={n}, eager and graph", flush=True)
    k = int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(k)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    w = fluid(n, 0.02, 3)
    w.r = 0.4 * g + 3.0 + 1e-3 * workloads.normals(8, 3 * n).reshape(n, 3)
    w.v = 0.1 * w.v
    out = []
    for graph in (False, True):
        s = system(ctx, [w], (0.33, 0.05), 1)
        s.lj_run(0.0005, 25, precision=pb.PB_FP64, skin=0.3, rebuild_every=8, energy_every=0,
                 use_graph=graph)
        out.append((s.get("r"), s.get("v")))
        s.close()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    assert np.isfinite(out[0][0]).all()
