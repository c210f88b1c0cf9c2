"""The summaries of trees with fractional masses in blocks of 4,096 records: less than one block,
cells across one border and across all of them, trees of the largest size whose blocks are one group
and past it, many bodies at one point over a border, two far clumps (cells from the root down to the
deepest levels across one border): every cell's bits equal to those with a launch more, which room
for more cells selects, and the oracle's tree where no two bodies coincide."""
import numpy as np
import pytest

from gpugraphlayout_amd import BatchEngine, Engine, graphs

pytestmark = pytest.mark.gpu


def positions(n, kind):
    rng = np.random.default_rng(n)
    if kind == "uniform":
        return graphs.uniform_positions(n, 2 * np.sqrt(n), n)
    p = rng.normal(size=(n, 2))
    if kind == "far":            # two clumps, each within 2^-14 of the box
        p = np.where(np.arange(n)[:, None] < n // 2, -1.0, 1.0) + p * 1e-5
    if kind == "point":          # a third of the bodies at one point
        p[n // 3:2 * n // 3] = p[0]
    return p.astype(np.float32)


@pytest.mark.parametrize("n,kind", [(4097, "uniform"), (5500, "far"), (8193, "point"), (20_000, "uniform"),
                                    (20_000, "far"), (41_000, "point"), (63_000, "uniform"), (63_300, "uniform")])
def test_fractional_tree(oracle, n, kind):
    print(f"case fractional tree n={n} {kind}", flush=True)
    pos = positions(n, kind)
    m = np.random.default_rng(n + 1).uniform(0.5, 9.0, n).astype(np.float32)
    i = np.arange(n, dtype=np.int32)
    trees = []
    for room in (3, 254_000 // n + 1):           # cells per body; from 253,952 records on two levels of groups
        eng = Engine(n, i, (i + 1) % n, mass=m, scale=2.0, strong_gravity=1, cell_factor=room)
        eng.set_positions(pos)
        eng.step(1)
        eng.sync()
        trees.append(eng.tree())
        eng.close()
    for key in ("level", "count", "mass", "xy", "perm"):
        np.testing.assert_array_equal(trees[0][key], trees[1][key], err_msg=key)
    if kind == "uniform":
        ref = oracle.tree(pos, m)
        for key in ("level", "count", "mass", "perm"):
            np.testing.assert_array_equal(trees[0][key], ref[key], err_msg=key)
        np.testing.assert_allclose(trees[0]["xy"], ref["xy"], rtol=1e-5, atol=1e-5 * np.abs(pos).max())


def test_fractional_batch():
    """Graphs of 1 to 5,000 bodies one after another: their cells share blocks and cross borders."""
    print("case fractional batch", flush=True)
    sizes = [1, 2, 3000, 4095, 1, 5000, 700, 33]
    rng = np.random.default_rng(8)
    ring = [(n, np.arange(n - 1, dtype=np.int32), np.arange(1, n, dtype=np.int32)) for n in sizes]
    masses = [rng.uniform(0.5, 9.0, n).astype(np.float32) for n in sizes]
    pos = np.concatenate([positions(n, "uniform" if n != 4095 else "far") for n in sizes])
    trees = []
    for room in (3, 254_000 // sum(sizes) + 1):
        eng = BatchEngine(ring, masses=masses, scale=2.0, cell_factor=room)
        eng.set_positions(pos)
        eng.step(1)
        eng.sync()
        trees.append(eng.tree())
        eng.close()
    for key in ("level", "count", "mass", "xy", "perm"):
        np.testing.assert_array_equal(trees[0][key], trees[1][key], err_msg=key)


@pytest.mark.parametrize("n,kind", [(63_500, "uniform"), (180_000, "uniform"), (240_000, "clumps"),
                                    (1_000_000, "uniform"), (4_000_000, "uniform")])
def test_fractional_groups(oracle, n, kind):
    """Trees of more blocks than one group holds (253,952 records): cells across the groups' borders,
    room for more than 62 groups (from 3.9M bodies on)."""
    print(f"case fractional groups n={n} {kind}", flush=True)
    pos = positions(n, "uniform")
    if kind == "clumps":
        rng = np.random.default_rng(n)
        pos = np.where(np.arange(n)[:, None] < n // 3, -1.0, 1.0) + rng.normal(size=(n, 2)) * 0.03
        pos = pos.astype(np.float32)
        assert len(np.unique(pos, axis=0)) == n
    m = np.random.default_rng(n + 1).uniform(0.5, 9.0, n).astype(np.float32)
    i = np.arange(n, dtype=np.int32)
    eng = Engine(n, i, (i + 1) % n, mass=m, scale=2.0, strong_gravity=1)
    eng.set_positions(pos)
    eng.step(1)
    eng.sync()
    tree = eng.tree()
    eng.close()
    ref = oracle.tree(pos, m)
    for key in ("level", "count", "mass", "perm"):
        np.testing.assert_array_equal(tree[key], ref[key], err_msg=key)
    np.testing.assert_allclose(tree["xy"], ref["xy"], rtol=1e-5, atol=1e-5 * np.abs(pos).max())
