"""The one-block tree of small graphs at its edges: one body, wave and row borders (64, 1,024), the
sizes where its form changes (2,048 and 4,096 bodies, and just past them), tied runs that the
sort's top digits leave (ordered by counting up to 64 bodies, by a second, full sort beyond),
coincident bodies, fractional masses and too few cells: the whole tree equal to the oracle's, and
repulsion, attraction and order as the other tests hold them."""
import numpy as np
import pytest

from gpugraphlayout_amd import GFA2_FORCE_REPULSION, Engine, GFA2Error, graphs

pytestmark = pytest.mark.gpu


def ring(n):
    a = np.arange(n if n > 2 else n - 1, dtype=np.int32)
    return a, ((a + 1) % n).astype(np.int32)


def positions(n, kind):
    rng = np.random.default_rng(n)
    if kind == "uniform":
        return graphs.uniform_positions(n, 2 * np.sqrt(n), n)
    p = rng.normal(size=(n, 2)).astype(np.float32)
    if kind == "far":            # two bodies far away: nearly all others share the top levels
        p *= 0.5                 # (the tree's depth stays under the 32 levels of a key)
        p[0], p[-1] = (-5e5, -4e5), (6e5, 5e5)
    if kind == "clump":          # clumps of 40 bodies, a lattice within 2^-16 of the box each
        k = np.arange(n) % 40
        p = np.repeat(rng.normal(size=(n // 40 + 1, 2)), 40, 0)[:n] + np.stack([k % 7, k // 7], 1) * 1e-5
    return p.astype(np.float32)


def check(oracle, n, pos, mass=None):
    s, t = ring(n) if n > 1 else (np.zeros(0, np.int32),) * 2
    eng = Engine(n, s, t, mass=mass, scale=2.0, strong_gravity=1)
    eng.set_capture(True)
    eng.set_positions(pos)
    m = (np.bincount(s, minlength=n) + np.bincount(t, minlength=n) + 1).astype(np.float32) if mass is None else mass
    for it in range(3):          # full sorts first, then by the previous tree's cells
        pos = eng.positions()
        eng.step(1)
        eng.sync()
        tree, ref = eng.tree(), oracle.tree(pos, m)
        for key in ("level", "count", "mass", "perm"):
            np.testing.assert_array_equal(tree[key], ref[key], err_msg=f"{key} at iteration {it}")
        # centroids: exact integer moments rounded once (whole masses) or the oracle's own order
        np.testing.assert_allclose(tree["xy"], ref["xy"], rtol=1e-5, atol=1e-5 * np.abs(pos).max())
        rep, _ = oracle.bh_repulsion(pos, m, 2.0, group=32)
        got = eng.forces(GFA2_FORCE_REPULSION)
        assert np.linalg.norm(got - rep) <= 1e-4 * np.linalg.norm(rep)
    eng.close()


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1023, 1024, 1025, 2047, 2048, 2049, 3000, 4095, 4096, 4097])
def test_tree_sizes(oracle, n):
    print(f"case small tree n={n}", flush=True)
    check(oracle, n, positions(n, "uniform"))


@pytest.mark.parametrize("n", [700, 2048, 3000, 4096])
@pytest.mark.parametrize("kind", ["far", "clump"])
def test_tied_runs(oracle, kind, n):
    print(f"case small tree {kind} n={n}", flush=True)
    check(oracle, n, positions(n, kind))


@pytest.mark.parametrize("n", [33, 1500, 4000])
def test_fractional_masses(oracle, n):
    print(f"case small tree masses n={n}", flush=True)
    check(oracle, n, positions(n, "uniform"), np.random.default_rng(n).uniform(0.5, 9.0, n).astype(np.float32))


def test_coincident_bodies_and_cell_capacity():
    """Bodies at one place share the level-32 cell in id order; too many cells are reported and
    leave the positions alone."""
    print("case small tree coincident", flush=True)
    n = 1200
    pos = positions(n, "uniform")
    pos[100:190] = pos[100]
    s, t = ring(n)
    eng = Engine(n, s, t)
    eng.set_positions(pos)
    eng.step(1)
    eng.sync()
    tree = eng.tree()
    deepest = tree["level"] == 32
    assert deepest.sum() == 1 and tree["count"][deepest][0] == 90
    at = np.flatnonzero(tree["perm"] == 100)[0]
    np.testing.assert_array_equal(tree["perm"][at:at + 90], np.arange(100, 190))
    eng.close()
    pairs = np.repeat(positions(n // 2, "uniform"), 2, 0)
    eng = Engine(n, s, t, cell_factor=1)
    eng.set_positions(pairs)
    eng.step(1)
    with pytest.raises(GFA2Error):
        eng.sync()
    np.testing.assert_array_equal(eng.positions(), pairs)
    eng.close()
