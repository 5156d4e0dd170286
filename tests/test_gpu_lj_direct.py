"""pb_lj_force's list-free kernel at the particle counts where the number of
lanes a particle changes, in replicas thinner than three cells (minimum image,
one window), in windows larger than the LDS stage (dense), with several types,
mixed precision, several replicas at once, with and without energies, and twice
in a row on a moved system (the kept layout of cells and segments).  FP64
against the oracle to 1e-12 F_rms (sums of up to 4e2 terms of FP64 rounding),
1e-11 where the summed terms exceed the result (dense); mixed to 1e-5 F_rms."""
import numpy as np
import pytest

import particlebase_amd as pb
from particlebase_amd import workloads

pytestmark = pytest.mark.gpu
RC2 = 6.25


def fluid(n, rho, seed):
    w = workloads.lj_fcc(int(np.ceil((n / 4) ** (1 / 3) - 1e-12)), rho, 0.72, seed=seed, natoms=n)
    w.r = w.r + 0.04 * workloads.normals(seed + 9, 3 * n).reshape(n, 3)
    return w


def system(ctx, ws, se, nt, rc2=RC2):
    s = pb.System(ctx, [w.n for w in ws])
    s.set_cell(np.concatenate([w.cell for w in ws]))
    s.import_particles(np.concatenate([w.r for w in ws]), np.concatenate([w.m for w in ws]),
                       type=np.concatenate([w.type for w in ws]))
    s.lj_set_params(se, nt)
    s.lj_set_cutoff(rc2, shifted=True)
    return s


def check(s, orc, ws, se, nt, prec, tol, rc2=RC2, cells=True):
    p = orc.lj_params(se, nt, rc2, True)
    pe, vir = s.lj_force(prec)
    F, at = s.get("F"), 0
    for k, w in enumerate(ws):
        r = orc.wrap(w.r, w.cell).reshape(-1, 3)
        f = orc.lj_forces_cells if cells else orc.lj_forces_brute
        Fo, peo, wo = f(r, w.type, w.cell, rc2, p)
        frms = np.sqrt((Fo ** 2).sum(1).mean())
        assert np.abs(F[at:at + w.n] - Fo).max() <= tol * frms, (k, w.n)
        rel = 1e-12 if prec == pb.PB_FP64 else 1e-5
        assert pe[k] == pytest.approx(peo, rel=rel, abs=1e-9) and vir[k] == pytest.approx(wo, rel=rel, abs=1e-9)
        at += w.n
    F1 = F.copy()
    s.lj_force(prec, energies=False)
    assert np.array_equal(s.get("F"), F1)


# slots are whole wavefronts: 12288 and 65536 are the last of 16 and 8 lanes
@pytest.mark.parametrize("n", [865, 12288, 12289, 65536, 65537])
@pytest.mark.parametrize("prec", [pb.PB_FP64, pb.PB_MIXED])
def test_lane_counts(ctx, orc, n, prec):
    print(f"\n[case] direct force n={n} prec={prec}", flush=True)
    w = fluid(n, 0.8, n % 97)
    s = system(ctx, [w], [1.0, 1.0], 1)
    check(s, orc, [w], [1.0, 1.0], 1, prec, 1e-12 if prec == pb.PB_FP64 else 1e-5)
    w.r = w.r + 0.01 * workloads.normals(5, 3 * n).reshape(n, 3)
    s.set("r", w.r)
    check(s, orc, [w], [1.0, 1.0], 1, prec, 1e-12 if prec == pb.PB_FP64 else 1e-5)
    s.close()


@pytest.mark.parametrize("prec", [pb.PB_FP64, pb.PB_MIXED])
def test_thin_replicas_and_types(ctx, orc, prec):
    print(f"\n[case] direct force, replicas of 100 to 5000, three types, prec={prec}", flush=True)
    se = np.array([[1.0, 1.0], [1.05, 0.8], [0.9, 1.2], [1.05, 0.8], [1.1, 0.6], [0.95, 1.0],
                   [0.9, 1.2], [0.95, 1.0], [0.8, 1.5]])
    ws = []
    for k, (n, rho) in enumerate([(150, 0.9), (257, 0.9), (500, 0.85), (64, 0.3), (5000, 0.7)]):
        w = fluid(n, rho, 40 + k)
        w.type = (np.arange(n) * 7 % 3).astype(np.uint32)
        ws.append(w)
    s = system(ctx, ws, se, 3)
    check(s, orc, ws, se, 3, prec, 1e-12 if prec == pb.PB_FP64 else 1e-5, cells=False)
    s.close()


@pytest.mark.parametrize("n", [4000, 80000])
def test_windows_larger_than_the_stage(ctx, orc, n):
    """A cluster far denser than the box: windows of more than 2816 particles."""
    print(f"\n[case] direct force, dense cluster n={n}", flush=True)
    w = fluid(n, 0.02, 3)
    k = int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(k)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    w.r = 0.35 * g + 0.01 * workloads.normals(8, 3 * n).reshape(n, 3) + 3.0
    s = system(ctx, [w], [0.3, 1.0], 1)
    check(s, orc, [w], [0.3, 1.0], 1, pb.PB_FP64, 1e-11)
    s.close()
