"""Cells and child lists of graphs past the one-block tree: clumps of just under, at and over 16 and
272 bodies, 20,000 to 32,769 bodies, fractional masses and a batch: the whole tree equal to the
oracle's."""
import numpy as np
import pytest

from gpugraphlayout_amd import GFA2_FORCE_REPULSION, BatchEngine, Engine, graphs

pytestmark = pytest.mark.gpu


def ring(n):
    a = np.arange(n, dtype=np.int32)
    return a, ((a + 1) % n).astype(np.int32)


def clumps(n, size):
    """Clumps of `size` bodies, each a lattice far smaller than the distance to the next."""
    rng = np.random.default_rng(n + size)
    k = np.arange(n) % size
    centre = np.repeat(rng.uniform(-1, 1, (n // size + 1, 2)), size, 0)[:n]
    return (centre + np.stack([k % 17, k // 17], 1) * 2e-6).astype(np.float32)


def compare(oracle, tree, pos, m):
    ref = oracle.tree(pos, m)
    for key in ("level", "count", "mass", "perm"):
        np.testing.assert_array_equal(tree[key], ref[key], err_msg=key)


@pytest.mark.parametrize("n,size", [(5000, 15), (5000, 16), (5000, 17), (9000, 18), (9000, 271), (9000, 272),
                                    (9000, 290), (32_768, 0), (32_769, 0), (20_000, 0)])
def test_tree(oracle, n, size):
    print(f"case cells n={n} clumps of {size}", flush=True)
    pos = clumps(n, size) if size else graphs.uniform_positions(n, 2 * np.sqrt(n), n)
    m = np.full(n, 3, np.float32)
    eng = Engine(n, *ring(n), scale=2.0)
    eng.set_capture(True)
    eng.set_positions(pos)
    eng.step(1)
    eng.sync()
    compare(oracle, eng.tree(), pos, m)
    rep, _ = oracle.bh_repulsion(pos, m, 2.0, group=32)
    assert np.linalg.norm(eng.forces(GFA2_FORCE_REPULSION) - rep) <= 1e-4 * np.linalg.norm(rep)
    eng.close()


def test_fractional_masses(oracle):
    print("case cells masses", flush=True)
    n = 7000
    pos = graphs.uniform_positions(n, 2 * np.sqrt(n), 1)
    m = np.random.default_rng(2).uniform(0.5, 9.0, n).astype(np.float32)
    eng = Engine(n, *ring(n), mass=m)
    eng.set_positions(pos)
    eng.step(1)
    eng.sync()
    compare(oracle, eng.tree(), pos, m)
    eng.close()


def test_batch(oracle):
    print("case cells batch", flush=True)
    sizes = [3, 700, 1, 4999, 2, 260]
    pos = [graphs.uniform_positions(n, 2 * np.sqrt(n), n) for n in sizes]
    none = np.zeros(0, np.int32)
    eng = BatchEngine([(n, none, none) for n in sizes], scale=2.0)
    eng.set_capture(True)
    eng.set_positions(np.concatenate(pos))
    eng.step(1)
    eng.sync()
    rep = eng.split(eng.forces(GFA2_FORCE_REPULSION))
    for n, p, r in zip(sizes, pos, rep):
        want, _ = oracle.bh_repulsion(p, np.ones(n, np.float32), 2.0, group=32)
        assert np.linalg.norm(r - want) <= 1e-4 * np.linalg.norm(want)
    eng.close()
