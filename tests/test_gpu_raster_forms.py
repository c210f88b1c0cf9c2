"""gfa2_render's ways of counting: tiles, atomics from the list (many lines of a few pixels, also of
more than one list), atomics without a list (small pictures, pictures whose tiles' scratch would be
out of proportion or finds no memory). The picture is bytes: equal to the CPU rasteriser's."""
import ctypes

import numpy as np
import pytest

from gpugraphlayout_amd import Engine, Mpnn, Raster, graphs, lib
from gpugraphlayout_amd.host import HostGraph, png_frame, render_gray

pytestmark = pytest.mark.gpu

EMPTY = np.zeros(0, np.int32)


def free_memory():
    free, total = ctypes.c_size_t(0), ctypes.c_size_t(0)
    assert lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0     # of the runtime the library runs on
    return free.value


def mesh(side):
    """side x side nodes at about their own places: every line is short."""
    i = np.arange(side * side)
    x = i % side
    hg = HostGraph.from_edges(np.concatenate([i[x < side - 1], i[:-side]]),
                              np.concatenate([i[x < side - 1] + 1, i[side:]]))
    at = np.stack([x, i // side], 1) + np.random.default_rng(side).uniform(-0.3, 0.3, (len(i), 2))
    return hg, hg.arrays(), at.astype(np.float32)


@pytest.mark.parametrize("side,w,h", [(200, 600, 500), (300, 4000, 3900), (100, 8000, 7900), (1030, 1250, 1250),
                                      (1000, 600, 500), (100, 200, 256), (12, 256, 1)])
def test_short_lines(side, w, h):
    print(f"case raster forms mesh {side} {w}x{h}", flush=True)
    hg, g, pos = mesh(side)
    pos[g.n // 2] = pos[g.n // 2 + 1]           # a line of no length
    eng = Engine(g.n, g.src, g.dst)
    eng.set_positions(pos)
    f = png_frame(eng.bbox(), w, h, g.n, g.m)
    f.node_alpha, f.edge_alpha = 0.02, 0.1
    got = eng.render(f)
    np.testing.assert_array_equal(got, render_gray(hg, pos, f))
    assert got.min() < got.max()
    np.testing.assert_array_equal(got, eng.render(f))       # from the workspace that is kept
    eng.close()


@pytest.mark.parametrize("w,h", [(1, 1_200_000), (700_000, 2)])
def test_narrow_pictures(w, h):
    print(f"case raster forms {w}x{h}", flush=True)
    s, t = graphs.barabasi_albert(12, 2, 1)
    hg = HostGraph.from_edges(s, t)
    g = hg.arrays()
    pos = (np.random.default_rng(3).normal(size=(g.n, 2)) * 100).astype(np.float32)
    eng = Engine(g.n, g.src, g.dst)
    eng.set_positions(pos)
    f = png_frame(eng.bbox(), w, h, g.n, g.m)
    np.testing.assert_array_equal(eng.render(f), render_gray(hg, pos, f))
    eng.close()


def test_widest_picture():
    """2^31 - 1 pixels in a row, two nodes and no line."""
    print("case raster forms 2^31 - 1 pixels", flush=True)
    eng = Engine(2, EMPTY, EMPTY)
    eng.set_positions(np.array([[10, 0], [2000, 0]], np.float32))
    got = eng.render(Raster(0.0, 0.0, 1.0, 1.0, 0.5, 0.5, 2 ** 31 - 1, 1))
    hit = np.zeros(2 ** 31 - 1, bool)
    hit[7:14] = hit[1997:2004] = True
    assert (got[0][hit] == 128).all() and got[0][~hit].min() == 255
    eng.close()


def test_falls_back_without_memory():
    print("case raster forms out of memory", flush=True)
    hg, g, pos = mesh(30)
    eng = Engine(g.n, g.src, g.dst)
    eng.set_positions(pos)
    f = png_frame(eng.bbox(), 16000, 14000, g.n, g.m)       # 3.1 GB by tiles, 2.0 GB without
    want = eng.render(f)
    # all but 2.6 GB held by a network handle's scratch (1,616 bytes a node) and graph (136)
    n = int((free_memory() - 2.6e9) // 1752)
    m = Mpnn(seed=1)
    m.add_graph(n, np.zeros(n + 1, np.int64), EMPTY, feature_seed=1, steps=0)
    np.testing.assert_array_equal(eng.render(f), want)
    m.close()
    np.testing.assert_array_equal(eng.bbox(), [pos[:, 0].min(), pos[:, 0].max(), pos[:, 1].min(), pos[:, 1].max()])
    eng.close()
