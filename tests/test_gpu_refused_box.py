"""A box that pb_sys_set_cell refuses leaves the system as it was: an LJ run after
it equals the run of a system that never saw it, bit for bit."""
import numpy as np
import pytest

import particlebase_amd as pb
from particlebase_amd import workloads

pytestmark = pytest.mark.gpu


def test_run_after_a_refused_box(ctx):
    print("\n[case] LJ run after a refused box", flush=True)
    ws = [workloads.lj_fcc(5, 0.8, 0.72, seed=k) for k in (3, 4)]
    out = []
    for refused in (False, True):
        s = pb.System(ctx, [w.n for w in ws])
        s.set_cell(np.concatenate([w.cell for w in ws]))
        s.import_particles(np.concatenate([w.r for w in ws]), np.concatenate([w.m for w in ws]),
                           v=np.concatenate([w.v for w in ws]))
        s.lj_set_params([1.0, 1.0], 1)
        s.lj_set_cutoff(6.25, shifted=True)
        s.clear_force(True)
        if refused:
            bad = np.concatenate([2.0 * ws[0].cell, ws[1].cell])
            bad[7] = bad[6]                       # the second replica's box is empty
            with pytest.raises(pb.PBError):
                s.set_cell(bad)
        e, _ = s.lj_run(0.004, 12, precision=pb.PB_FP64, skin=0.3, rebuild_every=5, energy_every=3)
        pe, _ = s.lj_force(pb.PB_FP64)
        out.append((np.asarray(e), np.asarray(pe), s.get("r"), s.get("v"), s.get("F")))
        s.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
