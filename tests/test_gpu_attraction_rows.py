"""The attraction with one to four medium rows to a wave (the count steps at 16,384, 24,576 and
32,768 such rows, the last wave's rows are fewer), rows of 33 to 2,048 entries, light rows and a
heavy one beside them: every row against 64-bit sums, and the same bits from the smaller grid of a
second stream, whose blocks read the hubs' positions from their own copy. The same of the wide
blocks of graphs with many entries of hubs."""
import numpy as np
import pytest

from gpugraphlayout_amd import GFA2_FORCE_ATTRACTION_GRAVITY, Engine, graphs

pytestmark = pytest.mark.gpu


def graph(nm):
    """nm medium rows, 6,000 light ones and one of 5,000 entries, numbered in random order."""
    rng = np.random.default_rng(nm)
    light, n = 6000, nm + 6001
    i = np.repeat(np.arange(nm), 17)                            # a ring of degree 34 ...
    s, t = [i], [(i + np.tile(np.arange(1, 18), nm)) % nm]
    for k, v in enumerate(range(0, nm, 997)):                   # ... with some longer rows
        count = (2048 - 34, 222, 223, 29, 1000)[k % 5]          # 2,048, 256, 257, 63 and 1,034 entries
        s.append(np.full(count, v))
        t.append(nm + (np.arange(count) + 1009 * k) % light)
    s.append(np.full(5000, n - 1))
    t.append(nm + np.arange(5000))
    new = rng.permutation(n)
    return n, new[np.concatenate(s)].astype(np.int32), new[np.concatenate(t)].astype(np.int32)


def check(n, s, t, linlog, weighted):
    degree = np.bincount(s, minlength=n) + np.bincount(t, minlength=n)
    pos = graphs.uniform_positions(n, 2 * np.sqrt(n), 5)
    w = np.random.default_rng(6).uniform(0.25, 4.0, len(s)).astype(np.float32) if weighted else None
    eng = Engine(n, s, t, weights=w, scale=2.0, linlog=linlog, edge_weight_influence=1.0, strong_gravity=1)
    got = []
    for config in ((256, 4, 0, 0), (256, 4, 2, 1)):
        eng.set_launch_config(*config)
        eng.reset()
        eng.set_positions(pos)
        eng.step(1)
        eng.sync()
        got.append(eng.forces(GFA2_FORCE_ATTRACTION_GRAVITY))
    eng.close()
    np.testing.assert_array_equal(got[0], got[1])
    p = pos.astype(np.float64)
    d = p[t] - p[s]
    if linlog:
        r = np.hypot(d[:, 0], d[:, 1])
        d *= (np.log1p(r) / np.where(r > 0, r, 1.0))[:, None]
    if weighted:
        d *= w.astype(np.float64)[:, None]
    gravity = -p * (degree + 1)[:, None]
    want, size = gravity.copy(), np.abs(gravity)
    for c in range(2):
        want[:, c] += np.bincount(s, d[:, c], n) - np.bincount(t, d[:, c], n)
        size[:, c] += np.bincount(s, np.abs(d[:, c]), n) + np.bincount(t, np.abs(d[:, c]), n)
    # a term rounds at most 8 times, and at most 48 additions follow one another: 32 in a light
    # row, 2048 / 64 + 6 + 1 in a medium one, 4096 / 256 + 8 + 2 in a heavy one; the smallest
    # differences of coordinates carry no error (the positions are exact)
    assert (np.abs(got[0] - want) <= 64 * 2.0 ** -24 * size).all()


@pytest.mark.parametrize("linlog,weighted", [(0, False), (1, True)])
@pytest.mark.parametrize("nm", [16383, 16384, 24577, 32771, 40000])
def test_rows_of_a_wave(nm, linlog, weighted):
    print(f"case attraction rows {nm} linlog={linlog} weighted={weighted}", flush=True)
    n, s, t = graph(nm)
    degree = np.bincount(s, minlength=n) + np.bincount(t, minlength=n)
    assert ((degree > 32) & (degree <= 2048)).sum() == nm
    check(n, s, t, linlog, weighted)


@pytest.mark.parametrize("linlog,weighted", [(0, False), (1, True)])
@pytest.mark.parametrize("nm,half", [(18001, 468), (9000, 940)])
def test_many_entries_of_hubs(nm, half, linlog, weighted):
    """Over 2^24 entries, of which the 8,192 longest rows hold a quarter or more: on one stream
    the wide blocks, beside other work the ordinary ones."""
    print(f"case attraction hubs {nm} linlog={linlog} weighted={weighted}", flush=True)
    rng = np.random.default_rng(nm)
    light, n = 9001, nm + 9001 + 3
    i = np.repeat(np.arange(nm), half)                          # a ring of degree 2 half
    s, t = [i], [(i + np.tile(np.arange(1, half + 1), nm)) % nm]
    for k, count in enumerate((2049, 5000, 9000)):              # rows of 1, 2 and 3 chunks
        s.append(np.full(count, n - 1 - k))
        t.append(nm + np.arange(count))
    new = rng.permutation(n)
    s, t = new[np.concatenate(s)].astype(np.int32), new[np.concatenate(t)].astype(np.int32)
    rows = np.sort(np.bincount(s, minlength=n) + np.bincount(t, minlength=n))
    assert 2 * len(s) >= 1 << 24 and rows[-8192:].sum() >= 2 * len(s) // 4
    check(n, s, t, linlog, weighted)
