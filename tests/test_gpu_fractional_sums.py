"""Trees with fractional masses against a serial summary in numpy: path keys restated, cells from
the keys, children added in order with one rounding each (mass from 0, centroid (sum m p) * (1 / m)),
bit for bit. Two far clumps, many bodies at one point, cells over one block border and over all of
them, graphs one after another; the one-block tree too."""
import numpy as np
import pytest

from gpugraphlayout_amd import BatchEngine, Engine, graphs

pytestmark = pytest.mark.gpu

F, WIDE = np.float32, np.longdouble


def fma(a, b, c):
    """Rounded once (a product of floats takes 48 of the 64 bits)."""
    return F(WIDE(a) * WIDE(b) + WIDE(c))


def path_keys(pos):
    lo, hi = pos.min(0), pos.max(0)
    r = F(np.max(hi - lo)) * F(0.5)
    c = np.tile((lo + hi) * F(0.5), (len(pos), 1)).astype(F)
    key = np.zeros(len(pos), np.uint64)
    for _ in range(32):
        r = r * F(0.5)
        above = c < pos
        key = key * np.uint64(4) + above[:, 0].astype(np.uint64) + above[:, 1].astype(np.uint64) * np.uint64(2)
        c = (c + np.where(above, r, -r)).astype(F)
    return key


def serial_tree(pos, mass):
    """level, count, mass and x, y of every cell in preorder, and the bodies' order."""
    n = len(pos)
    key = path_keys(pos)
    perm = np.argsort(key, kind="stable")
    k = key[perm]
    lcp = np.full(n + 1, -1)
    for i in range(n - 1):
        x = int(k[i] ^ k[i + 1])
        lcp[i] = 32 if x == 0 else (64 - x.bit_length()) // 2
    if n == 1:
        lcp[0] = 0
    level, count, out, stack = [], [], [], []

    def add(c, m, x, y):
        c[1], c[2], c[3] = fma(x, m, c[1]), fma(y, m, c[2]), F(c[3] + m)

    for i in range(n):
        for L in range((lcp[i - 1] if i > 0 else -1) + 1, lcp[i] + 1):
            stack.append([len(level), F(0), F(0), F(0), L, i])
            level.append(L)
            count.append(0)
            out.append(None)
        add(stack[-1], mass[perm[i]], pos[perm[i], 0], pos[perm[i], 1])
        while stack and (stack[-1][4] > lcp[i] or i == n - 1):
            at, x, y, m, _, first = stack.pop()
            inv = F(F(1) / m)
            out[at], count[at] = (m, F(x * inv), F(y * inv)), i + 1 - first
            if stack:
                add(stack[-1], *out[at])
    out = np.array(out, F)
    return dict(level=np.array(level), count=np.array(count), mass=out[:, 0], xy=out[:, 1:], perm=perm)


def positions(n, kind):
    rng = np.random.default_rng(n)
    p = rng.normal(size=(n, 2))
    if kind == "far":            # two clumps, each within 2^-14 of the box
        p = np.where(np.arange(n)[:, None] < n // 2, -1.0, 1.0) + p * 1e-5
    if kind == "point":          # a third of the bodies at one point
        p[n // 3:2 * n // 3] = p[0]
    return p.astype(F)


def check(eng, pos, sizes, masses):
    eng.set_positions(pos)
    eng.step(1)
    eng.sync()
    got = eng.tree()
    eng.close()
    off = np.concatenate([[0], np.cumsum(sizes)])
    want = [serial_tree(pos[a:b], m) for a, b, m in zip(off, off[1:], masses)]
    for key in ("level", "count"):
        np.testing.assert_array_equal(got[key], np.concatenate([w[key] for w in want]), err_msg=key)
    np.testing.assert_array_equal(got["perm"], np.concatenate([w["perm"] + a for w, a in zip(want, off)]))
    for key in ("mass", "xy"):
        np.testing.assert_array_equal(got[key].view(np.uint32),
                                      np.concatenate([w[key] for w in want]).view(np.uint32), err_msg=key)


@pytest.mark.parametrize("n,kind", [(900, "far"), (3000, "point"), (4097, "uniform"), (5500, "far"), (8193, "point"),
                                    (20_000, "far"), (41_000, "point"), (70_000, "uniform")])
def test_one_graph(n, kind):
    print(f"case fractional sums n={n} {kind}", flush=True)
    m = np.random.default_rng(n + 1).uniform(0.5, 9.0, n).astype(F)
    i = np.arange(n, dtype=np.int32)
    check(Engine(n, i, (i + 1) % n, mass=m, scale=2.0), positions(n, kind), [n], [m])


def test_batch():
    print("case fractional sums batch", flush=True)
    sizes = [1, 2, 3000, 4095, 1, 5000, 700, 33]
    rng = np.random.default_rng(8)
    ring = [(n, np.arange(n - 1, dtype=np.int32), np.arange(1, n, dtype=np.int32)) for n in sizes]
    masses = [rng.uniform(0.5, 9.0, n).astype(F) for n in sizes]
    pos = np.concatenate([positions(n, "far" if n == 4095 else "point" if n == 700 else "uniform") for n in sizes])
    check(BatchEngine(ring, masses=masses, scale=2.0), pos, sizes, masses)
