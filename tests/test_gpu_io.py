"""The host boundary (import / get / set) at the sizes where its transfer form
changes: directly written pinned memory up to 256 KiB a field, one 1 MiB
chunk, two ring slots, and several rounds of the ring with a short last
chunk.  Values are copied, so every comparison is exact; the storage order is
permuted (an LJ force sorts it) between the import and the reads."""
import numpy as np
import pytest

import particlebase_amd as pb

pytestmark = pytest.mark.gpu


def fields(rng, n):
    return {"r": rng.uniform(0.0, 40.0, (n, 3)), "v": rng.normal(size=(n, 3)),
            "a": rng.normal(size=(n, 3)), "m": rng.uniform(0.5, 2.0, n),
            "type": rng.integers(0, 5, n).astype(np.uint32),
            "fixed": (rng.random(n) < 0.3).astype(np.uint8)}


# 24 n bytes a vector field: 10922 is the last direct one, 43690 the last of
# one chunk, 87381 the last of two
@pytest.mark.parametrize("counts", [[1], [63, 1, 64], [10922], [10923], [43690], [43691], [87381],
                                    [100000, 77, 31000]])
def test_import_get_set_roundtrip(ctx, rng, counts):
    n = int(sum(counts))
    print(f"\n[case] io {counts}", flush=True)
    f = fields(rng, n)
    s = pb.System(ctx, counts)
    s.set_cell(np.tile([0.0, 40.0] * 3, len(counts)))
    s.import_particles(f["r"], f["m"], v=f["v"], a=f["a"], type=f["type"], is_fixed=f["fixed"])

    def check(exp):
        for k in ("r", "v", "a", "F"):
            assert np.array_equal(s.get(k), exp[k]), k
        assert np.array_equal(s.get("minv"), exp["minv"])
        assert np.array_equal(s.get("type"), exp["type"])
        assert np.array_equal(s.get("move"), exp["move"])

    exp = {"r": f["r"], "v": f["v"], "a": f["a"], "F": np.zeros((n, 3)), "minv": 1.0 / f["m"],
           "type": f["type"].astype(np.uint16), "move": 1 - f["fixed"]}
    check(exp)
    # a sort permutes the storage (r inside the box stays as it is); F is
    # replaced through set below
    s.lj_set_params(np.ones(50), 5)
    s.lj_set_cutoff(4.0, shifted=True)
    s.lj_force(pb.PB_FP64, energies=False)
    new = fields(rng, n)
    check({**exp, "F": s.get("F")})
    for k in ("r", "v", "a"):
        s.set(k, new[k])
    s.set("F", new["v"] + 1.0)
    s.set("minv", new["m"])
    s.set("type", new["type"])
    s.set("move", new["fixed"])
    check({"r": new["r"], "v": new["v"], "a": new["a"], "F": new["v"] + 1.0, "minv": new["m"],
           "type": new["type"].astype(np.uint16), "move": new["fixed"]})
    # a refused import changes nothing
    bad = new["m"].copy()
    bad[-1] = 0.0
    with pytest.raises(pb.PBError):
        s.import_particles(f["r"], bad)
    assert np.array_equal(s.get("r"), new["r"])
    s.import_particles(f["r"], f["m"])
    check({"r": f["r"], "v": np.zeros((n, 3)), "a": np.zeros((n, 3)), "F": np.zeros((n, 3)),
           "minv": 1.0 / f["m"], "type": np.zeros(n, np.uint16), "move": np.ones(n, np.uint8)})
    s.close()
