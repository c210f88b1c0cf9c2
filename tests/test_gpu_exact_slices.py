"""All-pairs repulsion at the edges of its split (16 runs of a graph's nodes, blocks of 64 bodies
that may hold the end of one graph and the start of the next) against float64."""
import numpy as np
import pytest

from gpugraphlayout_amd import GFA2_FORCE_REPULSION, BatchEngine, graphs

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 15, 16, 17, 31, 32, 33, 63, 64, 65, 130, 1000, 4]


@pytest.mark.parametrize("group", [32, 64])
def test_repulsion_of_many_sizes(group):
    print(f"case exact slices group {group}", flush=True)
    empty = np.zeros(0, np.int32)
    mass = [np.random.default_rng(n).integers(1, 9, n).astype(np.float32) for n in SIZES]
    pos = [graphs.uniform_positions(n, 2 * np.sqrt(n), n) for n in SIZES]
    eng = BatchEngine([(n, empty, empty) for n in SIZES], masses=mass, scale=3.0, group_size=group, use_barneshut=0)
    eng.set_capture(True)
    eng.set_positions(np.concatenate(pos))
    eng.step(1)
    eng.sync()
    eps = float(np.float32(0.05 * 0.05))
    for p, m, got in zip(pos, mass, eng.split(eng.forces(GFA2_FORCE_REPULSION))):
        d = p[:, None].astype(np.float64) - p[None]
        term = d * (3.0 * m[:, None] * m[None] / ((d * d).sum(2) + eps))[..., None]
        # per term: two roundings of d, three of d^2 + eps, the reciprocal (1 ulp), two products,
        # then at most len + 16 additions of partial sums
        bound = (16 + len(p) + 16) * 2.0 ** -24 * np.abs(term).sum(1)
        assert np.all(np.abs(got - term.sum(1)) <= bound)
    assert np.array_equal(eng.batch_stats()["interactions"], np.array(SIZES) ** 2)
    eng.close()
