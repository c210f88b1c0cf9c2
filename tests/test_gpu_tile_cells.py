"""Cells that reach past their tile of 512 sorted positions: graphs that end at, before and past a
tile's end, cells over two to all tiles, more than 1,024 tiles (a second look at the tiles' least
lcps) and more than 2,048 (the tiles' sums scanned), cells from the root down to level 32 over one
border, bodies at one point over several tiles, cells too heavy for a sum and tiles whose sums
wrap; in a batch, graphs of one body between them: the whole tree equal to the oracle's and repulsion
(by the child lists) within the usual bar."""
import numpy as np
import pytest

from gpugraphlayout_amd import GFA2_FORCE_REPULSION, BatchEngine, Engine, graphs

pytestmark = pytest.mark.gpu


def chain(n):
    a = np.arange(n - 1, dtype=np.int32)
    return a, a + 1


def masses(n, kind):
    rng = np.random.default_rng(n + 7)
    if kind == "heavy":          # cells over 2^24 a few levels up, some of them inside a tile
        return np.floor(rng.uniform(2e4, 6e4, n)).astype(np.float32)
    if kind == "wrap":           # sums over a tile near the largest that whole masses reach
        m = np.ones(n, np.float32)
        m[rng.integers(0, n, 50)] = 2.0 ** 24 - 1
        return m
    return rng.integers(1, 9, n).astype(np.float32)


def check(oracle, n, pos, m):
    eng = Engine(n, *chain(n), mass=m, scale=2.0)
    eng.set_capture(True)
    eng.set_positions(pos)
    eng.step(1)
    eng.sync()
    tree, ref = eng.tree(), oracle.tree(pos, m)
    for key in ("level", "count", "mass", "perm"):
        np.testing.assert_array_equal(tree[key], ref[key], err_msg=key)
    np.testing.assert_allclose(tree["xy"], ref["xy"], rtol=1e-5, atol=1e-5 * np.abs(pos).max())
    if n <= 20_000:
        rep, _ = oracle.bh_repulsion(pos, m, 2.0, group=32)
        assert np.linalg.norm(eng.forces(GFA2_FORCE_REPULSION) - rep) <= 1e-4 * np.linalg.norm(rep)
    eng.close()


@pytest.mark.parametrize("n,kind", [(4607, "plain"), (4608, "plain"), (4609, "plain"), (5120, "heavy"), (20_000, "heavy"),
                                    (20_000, "wrap"), (131_073, "plain"), (524_800, "plain"), (1_048_576, "plain"),
                                    (1_049_100, "plain"), (1_200_000, "wrap")])
def test_tree(oracle, n, kind):
    print(f"case tile cells n={n} {kind}", flush=True)
    check(oracle, n, graphs.uniform_positions(n, 2 * np.sqrt(n), n), masses(n, kind))


@pytest.mark.parametrize("n", [5000, 6144])
def test_deep_cells(oracle, n):
    """Half of the bodies within 2^-20 of the box, on a lattice: cells of all levels down to there
    over the same borders."""
    print(f"case tile cells deep n={n}", flush=True)
    pos = graphs.uniform_positions(n, 1.0, n).astype(np.float64)
    k = np.arange(n // 2)
    pos[: n // 2] = 0.3125 + np.stack([k % 64, k // 64], 1) * 2.0 ** -22
    check(oracle, n, pos.astype(np.float32), masses(n, "plain"))


def test_bodies_at_one_point():
    """3,000 bodies at one point: a level-32 cell over several tiles, its children its bodies."""
    print("case tile cells point", flush=True)
    n = 9000
    pos = graphs.uniform_positions(n, 2 * np.sqrt(n), 3)
    pos[1000:4000] = pos[1000]
    eng = Engine(n, *chain(n), scale=2.0)
    eng.set_positions(pos)
    eng.step(1)
    eng.sync()
    tree = eng.tree()
    assert sorted(tree["count"][tree["level"] == 32])[-1] == 3000
    assert tree["count"][0] == n and tree["level"].max() == 32
    # every cell's bodies are its children's, which follow it: counts fall along each run of deeper cells
    inside = np.flatnonzero(tree["level"][1:] > tree["level"][:-1])
    assert (tree["count"][inside + 1] <= tree["count"][inside]).all()
    eng.close()


def test_batch(oracle):
    print("case tile cells batch", flush=True)
    sizes = [1, 511, 1, 2, 512, 513, 1, 1, 3000, 1535, 1, 700]
    pos = [graphs.uniform_positions(n, 2 * np.sqrt(n) + 1, k) for k, n in enumerate(sizes)]
    m = [masses(n, "plain") for n in sizes]
    eng = BatchEngine([(n, *chain(n)) for n in sizes], masses=m, scale=2.0)
    eng.set_capture(True)
    eng.set_positions(np.concatenate(pos))
    eng.step(1)
    eng.sync()
    tree, rep = eng.tree(), eng.split(eng.forces(GFA2_FORCE_REPULSION))
    eng.close()
    roots = np.append(np.flatnonzero(tree["level"] == 0), len(tree["level"]))
    off = np.concatenate([[0], np.cumsum(sizes)])
    for k, n in enumerate(sizes):
        ref = oracle.tree(pos[k], m[k])
        for key in ("level", "count", "mass"):
            np.testing.assert_array_equal(tree[key][roots[k]:roots[k + 1]], ref[key], err_msg=f"graph {k} {key}")
        np.testing.assert_array_equal(tree["perm"][off[k]:off[k + 1]] - off[k], ref["perm"])
        want, _ = oracle.bh_repulsion(pos[k], m[k], 2.0, group=32)
        assert np.linalg.norm(rep[k] - want) <= 1e-4 * np.linalg.norm(want)
