"""A replica's sums have the same bits alone and in any company: kinetic energies
and Gaussian steps of replicas by themselves and together, where the forms of the
reduction change (a workgroup for all, a wavefront each from 4 replicas, the
workgroup again beyond 2048 wavefronts a replica on average; the Gaussian solves
in kernels of their own beyond 512 wavefronts of the largest replica)."""
import numpy as np
import pytest

import particlebase_amd as pb

pytestmark = pytest.mark.gpu
SIZES = [(5000, 33000), (5000, 64, 9000, 1), (5000, 33000, 1, 64, 12345),
         tuple(range(4000, 4320, 20)), (180000, 3, 180000, 180001)]


def state(n):
    g = np.random.default_rng(n)
    return (g.uniform(0, 10, (n, 3)), g.normal(size=(n, 3)), g.normal(scale=3.0, size=(n, 3)),
            g.uniform(0.5, 2.0, n))


def loaded(ctx, sizes):
    r, v, F, m = (np.concatenate(x) for x in zip(*[state(n) for n in sizes]))
    s = pb.System(ctx, list(sizes))
    s.set_cell(np.tile([0.0, 10.0] * 3, len(sizes)))
    s.import_particles(r, m, v=v, a=0.9 * F)
    s.set("F", F)
    return s


@pytest.mark.parametrize("sizes", SIZES)
def test_alone_and_together(ctx, sizes):
    print(f"\n[case] sums of {len(sizes)} replicas, alone and together", flush=True)

    def run(part, first):
        s = loaded(ctx, part)
        e0 = np.array(s.mv2())
        s.gt_xi(set_xi=[0.05 - 0.02 * (first + k) for k in range(len(part))])
        for _ in range(2):
            s.gt_step(0.002, 1e-9)
        out = e0, np.array(s.mv2()), s.gt_xi()[0], s.get("v"), s.get("r")
        s.close()
        return out
    both = run(sizes, 0)
    at = 0
    for q, n in enumerate(sizes):
        alone = run((n,), q)
        for a, b in zip(alone[:3], both[:3]):
            assert a[0] == b[q], (q, n)
        for a, b in zip(alone[3:], both[3:]):
            assert np.array_equal(a, b[at:at + n]), (q, n)
        at += n
