"""Setting positions and resetting in one launch each: an engine that has run, was given other
positions and was reset gives the bits of a fresh one, from one body to past one round of the
grid, in either order of the two calls, and for a batch of more graphs than a block has threads."""
import numpy as np
import pytest

from gpugraphlayout_amd import BatchEngine, Engine, graphs

pytestmark = pytest.mark.gpu


def run(eng, order, pos, steps):
    for call in order:
        eng.reset() if call == "reset" else eng.set_positions(pos)
    eng.step(steps)
    eng.sync()
    s = eng.stats()
    return eng.positions(), eng.forces(), [s[k] for k in sorted(s) if k != "allocated_bytes"]


def check(make, n):
    first, second = (graphs.uniform_positions(n, side * np.sqrt(n), seed) for side, seed in ((3.0, 1), (2.0, 2)))
    used = make()
    run(used, ["positions"], first, 3)
    for order in (["positions", "reset"], ["reset", "positions"]):
        fresh = make()
        got, want = run(used, order, second, 3), run(fresh, order, second, 3)
        fresh.close()
        np.testing.assert_array_equal(got[0], want[0])
        np.testing.assert_array_equal(got[1], want[1])
        assert got[2] == want[2]
    used.close()


@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 5000, 300_000])
def test_reset_is_a_fresh_engine(n):
    print(f"case reset n={n}", flush=True)
    i = np.arange(n - 1, dtype=np.int32)
    check(lambda: Engine(n, i, i + 1, scale=2.0, strong_gravity=1), n)


def test_reset_of_a_batch():
    print("case reset batch", flush=True)
    sizes = [3 + k % 5 for k in range(700)]
    ring = [(n, np.arange(n - 1, dtype=np.int32), np.arange(1, n, dtype=np.int32)) for n in sizes]
    check(lambda: BatchEngine(ring, scale=2.0), sum(sizes))
