"""Speed and displacement at the sizes where their launch form changes (one graph of 2,048 walk
groups of 32, a batch of graphs of 32,768 nodes): every iteration's sums, speed, positions and the
next attraction (which gathers from the displacement's ranked copy) against the oracle."""
import numpy as np
import pytest

from gpugraphlayout_amd import GFA2_FORCE_ATTRACTION_GRAVITY, BatchEngine, Engine, graphs

pytestmark = pytest.mark.gpu


def ring(n, seed):
    """A cycle with chords (no edge for one node)."""
    if n < 2:
        return np.zeros(0, np.int32), np.zeros(0, np.int32)
    rng = np.random.default_rng(seed)
    a = np.concatenate([np.arange(n), rng.integers(0, n, n // 3)])
    b = np.concatenate([(np.arange(n) + 1) % n, rng.integers(0, n, n // 3)])
    key = np.unique(np.minimum(a, b)[a != b] * n + np.maximum(a, b)[a != b])
    return (key // n).astype(np.int32), (key % n).astype(np.int32)


def check(oracle, eng, sizes, edges, stats_of):
    off = np.concatenate([[0], np.cumsum(sizes)])
    src = np.concatenate([s + o for (s, _), o in zip(edges, off)])
    dst = np.concatenate([t + o for (_, t), o in zip(edges, off)])
    mass = (np.bincount(src, minlength=off[-1]) + np.bincount(dst, minlength=off[-1]) + 1).astype(np.float64)
    speed = np.ones(len(sizes), np.float32)
    fprev = np.zeros((off[-1], 2), np.float32)
    for it in range(3):
        before = eng.positions()
        eng.step(1)
        eng.sync()
        after, f = eng.positions(), eng.forces()
        fga = eng.forces(GFA2_FORCE_ATTRACTION_GRAVITY).astype(np.float64)
        p = before.astype(np.float64)
        want = -p * mass[:, None]                         # strong gravity, k_g = 1
        np.add.at(want, src, p[dst] - p[src])
        np.add.at(want, dst, p[src] - p[dst])
        # at most a few hundred float32 additions per node, each half an ulp of the terms' size
        size = np.abs(p).max() * mass
        assert np.all(np.abs(fga - want) <= (256 * 2.0 ** -24) * size[:, None])
        stats = stats_of()
        d, s = f.astype(np.float64) - fprev, f.astype(np.float64) + fprev
        for g in range(len(sizes)):
            r = slice(off[g], off[g + 1])
            swing = (mass[r] * np.linalg.norm(d[r], axis=1)).sum()
            traction = (mass[r] * np.linalg.norm(s[r], axis=1)).sum() / 2
            # float32 terms and sums of 32 of them, then double: under 40 half-ulps
            assert stats["swing"][g] == pytest.approx(swing, rel=40 * 2.0 ** -24)
            assert stats["traction"][g] == pytest.approx(traction, rel=40 * 2.0 ** -24)
            gs = float(stats["speed"][g])
            assert gs <= speed[g] * 1.5 * (1 + 2.0 ** -22)      # the rise is capped
            speed[g] = gs
            factor = gs / (1.0 + np.sqrt(gs * np.linalg.norm(d[r], axis=1)))
            new = p[r] + f[r].astype(np.float64) * factor[:, None]
            scale = np.abs(p[r]) + np.abs(f[r] * factor[:, None])
            assert np.all(np.abs(after[r] - new) <= 4 * 2.0 ** -23 * scale)
        fprev = f


@pytest.mark.parametrize("n", [1, 33, 65_536, 65_537])
def test_one_graph(oracle, n):
    print(f"case advance n={n}", flush=True)
    e = ring(n, n)
    eng = Engine(n, *e, strong_gravity=1, scale=2.0)
    eng.set_positions(graphs.uniform_positions(n, 2 * np.sqrt(n), 3))

    def stats():
        s = eng.stats()
        return {"swing": [s["swing"]], "traction": [s["traction"]], "speed": [s["global_speed"]]}

    check(oracle, eng, [n], [e], stats)
    eng.close()


@pytest.mark.parametrize("sizes", [[5, 32_768, 1, 700], [40, 32_769]])
def test_batch(oracle, sizes):
    print(f"case advance batch {sizes}", flush=True)
    edges = [ring(n, n) for n in sizes]
    eng = BatchEngine([(n, s, t) for n, (s, t) in zip(sizes, edges)], strong_gravity=1, scale=2.0)
    eng.set_positions(np.concatenate([graphs.uniform_positions(n, 2 * np.sqrt(n), n) for n in sizes]))
    check(oracle, eng, sizes, edges, eng.batch_stats)
    eng.close()
