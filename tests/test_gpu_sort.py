"""The cell sort where its forms change: cell counts on both sides of one scan
block (4096) and of the one-launch scan (16384), cells of 0, 1, 7, 8, 9 and
hundreds of particles (the ordering reads eight keys at a time), particle
counts on both sides of a wavefront, and a second sort on the same counters.
Equality with the oracle's stable sort."""
import numpy as np
import pytest

import particlebase_amd as pb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb", [(3, 3, 3), (15, 13, 21), (16, 16, 16), (25, 25, 26), (29, 5, 113),
                                (16, 16, 64), (40, 41, 42)])
@pytest.mark.parametrize("n", [1, 64, 65, 6001])
def test_bins_against_oracle(ctx, orc, nb, n):
    print(f"\n[case] sort {nb} cells, {n} particles", flush=True)
    rng = np.random.default_rng(n + nb[2])
    cell = np.array([0, nb[0], 0, nb[1], 0, nb[2]], dtype=np.float32)
    s = pb.System(ctx, [n])
    s.set_cell(cell.astype(np.float64))
    s.setup_cells(1.0, periodic=True)
    bn, bl = s.cell_info()
    assert tuple(bn) == nb
    for again in range(2):
        r = (rng.random((n, 3)) * np.array(nb)).astype(np.float32)
        if n > 2000:                       # crowded cells: 300, 9, 8, 7
            at = 0
            for k, m in enumerate((300, 9, 8, 7)):
                r[at:at + m] = rng.random((m, 3)).astype(np.float32) * 0.9 + [1, k % 3, 1]
                at += m
            r = rng.permutation(r)
        s.import_particles(r.astype(np.float64), np.ones(n))
        s.bin()
        pid, bid, bindex = s.get_bins()
        opid, obid, obindex = orc.sort_bins(orc.calc_bid(r, bl, bn), int(np.prod(nb)))
        assert np.array_equal(pid, opid)
        assert np.array_equal(bid, obid)
        assert np.array_equal(bindex, obindex)
    s.close()
