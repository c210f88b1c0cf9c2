"""Repulsion of bodies at one point where the walk opens their level-32 cell (a root radius of 1e5,
so that the deepest opening distance does not round away beside the softening): each of them is met
directly, however many they are."""
import numpy as np
import pytest

from gpugraphlayout_amd import GFA2_FORCE_REPULSION, BatchEngine, Engine

pytestmark = pytest.mark.gpu

EMPTY = np.zeros(0, np.int32)


def lattice(side, sets, seed):
    """side x side bodies over a square of 2e5, jittered; each set's bodies at its first one's place."""
    rng = np.random.default_rng(seed)
    i = np.arange(side * side)
    step = 2e5 / (side - 1)
    pos = np.stack([i % side, i // side], 1) * step - 1e5 + rng.uniform(-0.2, 0.2, (side * side, 2)) * step
    pos = pos.astype(np.float32)
    ids = rng.permutation(side * side)
    for k in sets:
        pos[ids[:k]] = pos[ids[0]]
        ids = ids[k:]
    return pos


def direct(pos, mass, k_r, eps2):
    """(sums, sums of the terms' sizes) in 64 bits."""
    p, m = pos.astype(np.float64), mass.astype(np.float64)
    out, size = np.empty_like(p), np.empty_like(p)
    for a in range(0, len(p), 500):
        d = p[a:a + 500, None] - p[None]
        w = k_r * m[a:a + 500, None] * m / ((d * d).sum(2) + eps2)
        out[a:a + 500] = (d * w[..., None]).sum(1)
        size[a:a + 500] = (np.abs(d) * w[..., None]).sum(1)
    return out, size


def repulsion(eng, pos):
    eng.set_capture(True)
    eng.set_positions(pos)
    eng.step(1)
    eng.sync()
    return eng.forces(GFA2_FORCE_REPULSION)


@pytest.mark.parametrize("group", [32, 64])
@pytest.mark.parametrize("count", [5, 6, 17, 30])
def test_one_group_meets_every_body(count, group):
    """Bodies of one vote group: every one meets every body record, itself included."""
    side = 5 if group == 32 else 7
    print(f"case coincident bodies={count} group={group}", flush=True)
    n = side * side
    pos = lattice(side, [min(count, n - 4)], 1)
    eng = Engine(n, EMPTY, EMPTY, scale=2.0, group_size=group)
    got = repulsion(eng, pos)
    assert eng.stats()["interactions"] == n * n
    eng.close()
    want, size = direct(pos, np.ones(n), 2.0, 0.0025)
    # at most 5 roundings and a reciprocal of one unit per term, n additions in a row
    assert (np.abs(got - want) <= (n + 16) * 2.0 ** -24 * size).all()


@pytest.mark.parametrize("side", [50, 71])
@pytest.mark.parametrize("group,mode", [(32, 0), (64, 0), (32, 1)])
def test_larger_sets(side, group, mode):
    """Sets up to more than the walk's list holds, by the one-block tree and the tiled one; at this
    opening angle nothing but the level-32 cells is ever accepted whole."""
    print(f"case coincident sets n={side * side} group={group} mode={mode}", flush=True)
    n = side * side
    pos = lattice(side, [5, 6, 9, 20, 33, 70, 130, 300], 2)
    params = dict(scale=2.0, theta=1e-3, group_size=group)
    eng = Engine(n, EMPTY, EMPTY, **params)
    eng.set_launch_config(256, 8, mode, 0)
    got = repulsion(eng, pos)
    eng.close()
    want, size = direct(pos, np.ones(n), 2.0, 0.0025)
    assert (np.abs(got - want) <= (n + 16) * 2.0 ** -24 * size).all()
    eng = BatchEngine([(n, EMPTY, EMPTY)] * 2, **params)
    np.testing.assert_array_equal(repulsion(eng, np.concatenate([pos, pos])), np.concatenate([got, got]))
    eng.close()
