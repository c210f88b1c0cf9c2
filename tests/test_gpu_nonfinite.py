"""Positions that are not finite, or so far apart that the root's radius is not: no kernel is led out
of its arrays by them (places come from the keys' bits, never from a coordinate), and a graph alone
(the one-block tree or the tiled one, speed and displacement in one launch) moves as it does in a
batch (the tiled tree, a block per graph; from 32,769 nodes on the launches of large graphs)."""
import numpy as np
import pytest

from gpugraphlayout_amd import BatchEngine, Engine, graphs

pytestmark = pytest.mark.gpu


def spoiled(pos, kind):
    pos = pos.copy()
    if kind == "nan":
        pos[7, 0] = np.nan
    elif kind == "inf":
        pos[7] = np.inf
    elif kind == "mixed":
        pos[3], pos[9], pos[11] = [np.nan, 1], [-np.inf, 2], [np.inf, np.nan]
    elif kind == "far":
        pos[5], pos[6] = [3e38, -3e38], [-3e38, 3e38]
    elif kind == "all":
        pos[:] = np.nan
    return pos


@pytest.mark.parametrize("kind", ["nan", "inf", "mixed", "far", "all"])
@pytest.mark.parametrize("n", [40, 300, 3000, 6000, 40_000])
def test_alone_as_in_a_batch(n, kind):
    print(f"case not finite n={n} {kind}", flush=True)
    s, t = graphs.barabasi_albert(n, 3, n)
    good = graphs.uniform_positions(n, 2 * np.sqrt(n), 1)
    moved = []
    for pos in (spoiled(good, kind), good):
        eng = Engine(n, s, t, scale=2.0)
        eng.set_positions(pos)
        eng.step(3)
        eng.sync()
        tree = eng.tree()
        assert tree["count"][0] == n and sorted(tree["perm"].tolist()) == list(range(n))
        moved.append(eng.positions())
        eng.close()
    eng = BatchEngine([(n, s, t)] * 2, scale=2.0)
    eng.set_positions(np.concatenate([spoiled(good, kind), good]))
    eng.step(3)
    eng.sync()
    np.testing.assert_array_equal(eng.positions(), np.concatenate(moved))     # (NaN where NaN is)
    eng.close()
    assert np.isfinite(moved[1]).all() and not np.isfinite(moved[0]).all()
