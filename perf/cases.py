"""The work users have this engine do, as cases that can be timed and compared.

Every case goes through the package's public entry points (Engine, BatchEngine, Mpnn and the
host layer's png_frame), with graphs, starts and options drawn from a seed:

  layout   ForceAtlas2 iterations on one graph, positions read back (the main path)
  forces   one iteration from given positions, forces and positions read back
  batch    the same for many graphs at once
  grad     forward and backward pass of the learned initialiser on one training graph
  start    a learned start: features, inference into the engine, positions read back
  render   the picture of a layout
  stress   hop distances of sampled pairs and the normalized stress of a layout

listed() gives the fixed cases, draw() more of the same ranges, prepare() what a program holds
before the call, run() one pass, work() the bytes and operations a pass cannot do without and
exact() the outputs in 64 bits, computed here in plain torch.
"""
import math

import numpy as np
import torch

from gpugraphlayout_amd import BatchEngine, Engine, Mpnn, graphs, workloads
from gpugraphlayout_amd.host import png_frame

# ---- the cases --------------------------------------------------------------------------------


def listed():
    return [
        # an interactive viewer's frame on a small graph: one iteration, then the positions are drawn
        dict(name="view-ba500", kind="layout", family="ba", n=500, m=3, steps=1, strong=1, scale=2.0),
        # the Barabasi-Albert workload of the benchmark, positions read every 20 iterations
        dict(name="layout-ba10k", kind="layout", family="ba", n=10_000, m=5, steps=20, strong=1, scale=2.0),
        # one graph of the learned initialiser's set, iterations replayed as a captured graph
        dict(name="replay-sbm50k", kind="layout", family="sbm", n=50_000, steps=10, scale=2.0, capture=1),
        # forces of a given layout with every option at once: given (fractional) masses, edge
        # weights, linlog, 64-lane votes
        dict(name="options-ba20k", kind="forces", family="ba", n=20_011, m=4, scale=5.0, group=64, masses=1, weights=1,
             linlog=1),
        # the same with all-pairs repulsion, which checks the tree's and `graph_viewer ... exact` runs
        dict(name="exact-ba12k", kind="forces", family="ba", n=12_345, m=4, scale=2.0, allpairs=1),
        # the benchmark's headline graph, launch shape picked by the autotuner as the README shows
        dict(name="layout-rmat20", kind="layout", family="rmat", ids=20, n=579_581, edges=10_000_000, steps=8, scale=10.0, tune=1),
        # a graph several times that size with the default launch shape
        dict(name="layout-rmat22", kind="layout", family="rmat", ids=22, n=2_003_001, edges=32_000_000, steps=4, scale=10.0),
        # a slice of the batched workload: graphs of 100 to 20,000 nodes laid out together
        dict(name="batch-192", kind="batch", graphs=192, steps=4),
        # one training step's gradient on a graph of the learned initialiser's set
        dict(name="grad-sbm50k", kind="grad", n=50_000, offsets=8, smooth=2),
        # a learned start for the headline graph
        dict(name="start-rmat20", kind="start", ids=20, n=579_581, edges=10_000_000, smooth=1),
        # a snapshot in graph_viewer's default picture size
        dict(name="render-rmat17", kind="render", ids=17, n=71_000, edges=1_000_000, width=1250, height=1250),
        # layout quality on a million sampled pairs
        dict(name="stress-rmat18", kind="stress", ids=18, n=155_555, edges=2_500_000, sources=1024, targets=977),
    ]


def _log(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    def rmat(low, high, most):
        ids = rng.randint(low, high)
        edges = int((1 << ids) * rng.uniform(4.0, most))
        return dict(ids=ids, n=int((1 << ids) * rng.uniform(0.4, 0.6)), edges=edges)

    kind = rng.choice(["layout"] * 5 + ["forces", "forces", "batch", "grad", "start", "render", "stress"])
    if kind == "layout":
        what = rng.choice(["small", "small", "sbm", "rmat", "rmat"])
        if what == "small":
            return dict(kind=kind, family="ba", n=_log(rng, 100, 20_000), m=rng.randint(2, 8),
                        steps=rng.choice([1, 1, 5, 20]), strong=rng.randint(0, 1), scale=2.0,
                        capture=rng.randint(0, 1))
        if what == "sbm":
            return dict(kind=kind, family="sbm", n=_log(rng, 5_000, 200_000), steps=rng.choice([1, 10]), scale=2.0,
                        capture=rng.randint(0, 1))
        if what == "rmat":
            return dict(kind=kind, family="rmat", steps=rng.choice([1, 4]), scale=10.0,
                        group=rng.choice([32, 32, 64]), **rmat(15, 22, 7.6))
    if kind == "forces":
        if rng.randint(0, 1):
            return dict(kind=kind, family="ba", n=_log(rng, 300, 60_000), m=rng.randint(2, 6), scale=5.0,
                        group=rng.choice([32, 64]), masses=rng.randint(0, 1), weights=rng.randint(0, 1),
                        linlog=rng.randint(0, 1))
        return dict(kind=kind, family="ba", n=_log(rng, 500, 20_000), m=rng.randint(2, 8), scale=2.0, allpairs=1)
    if kind == "batch":
        return dict(kind=kind, graphs=_log(rng, 16, 192), steps=rng.choice([1, 4]))
    if kind == "grad":
        return dict(kind=kind, n=_log(rng, 5_000, 100_000), offsets=rng.choice([4, 8]), smooth=rng.randint(1, 2))
    if kind == "start":
        return dict(kind=kind, smooth=rng.randint(1, 2), **rmat(15, 20, 9.5))
    if kind == "render":
        return dict(kind=kind, width=rng.randint(500, 1250), height=rng.randint(500, 1250), **rmat(12, 17, 7.6))
    return dict(kind=kind, sources=rng.choice([200, 1024]), targets=rng.choice([100, 977]), **rmat(13, 18, 9.5))


# ---- inputs -----------------------------------------------------------------------------------


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _fitted(n, a, b, gen):
    """(n, rowptr, col) of undirected edges, as the symmetric CSR of a graph of exactly n
    nodes: node ids past n fold onto others, a node without an edge gets one.
    Rows ascend."""
    dev = a.device
    a, b = a % n, b % n
    alone = torch.ones(n, dtype=torch.bool, device=dev)
    alone[a] = False
    alone[b] = False
    alone = alone.nonzero().flatten()
    a = torch.cat([a, alone])
    b = torch.cat([b, torch.randint(n, (alone.numel(),), generator=gen, device=dev)])
    a, b = a[a != b], b[a != b]
    key = torch.unique(torch.cat([a * n + b, b * n + a]))
    rows = torch.div(key, n, rounding_mode="floor")
    rowptr = torch.zeros(n + 1, dtype=torch.int64, device=dev)
    rowptr[1:] = torch.bincount(rows, minlength=n).cumsum(0)
    return n, rowptr.cpu().numpy(), (key - rows * n).to(torch.int32).cpu().numpy()


def _rmat(n, ids, edges, seed):
    """R-MAT graph over 2^ids ids (a, b, c, d = 0.57, 0.19, 0.19, 0.05): distinct undirected
    edges, isolated ids dropped, the rest numbered in random order and fitted to n nodes."""
    dev = _device()
    gen = torch.Generator(device=dev).manual_seed(int(seed))
    have = torch.zeros(0, dtype=torch.int64, device=dev)
    while have.numel() < edges:
        count = int((edges - have.numel()) * 1.2) + 1024
        s = torch.zeros(count, dtype=torch.int64, device=dev)
        t = torch.zeros(count, dtype=torch.int64, device=dev)
        for _ in range(ids):
            r = torch.rand(count, generator=gen, device=dev)
            s = 2 * s + (r >= 0.76)
            t = 2 * t + ((r >= 0.57) & (r < 0.76) | (r >= 0.95))
        lo, hi = torch.minimum(s, t), torch.maximum(s, t)
        have = torch.unique(torch.cat([have, (lo * (1 << ids) + hi)[lo != hi]]))
    have = have[torch.randperm(have.numel(), generator=gen, device=dev)[:edges]]
    a, b = have >> ids, have & ((1 << ids) - 1)
    used = torch.zeros(1 << ids, dtype=torch.bool, device=dev)
    used[a] = True
    used[b] = True
    used = used.nonzero().flatten()
    new = torch.zeros(1 << ids, dtype=torch.int64, device=dev)
    new[used] = torch.randperm(used.numel(), generator=gen, device=dev)
    return _fitted(n, new[a], new[b], gen)


def _graph(case, seed):
    """(nodes, rowptr, col) of a case."""
    family = case.get("family", "rmat")
    if family == "rmat":
        return _rmat(case["n"], case["ids"], case["edges"], seed)
    if family == "ba":
        s, t = graphs.barabasi_albert(case["n"], case["m"], seed)
    else:
        s, t, _ = graphs.sbm(case["n"], 32, 2.0, seed)
    g = workloads.host_graph(s, t)
    dev = _device()
    gen = torch.Generator(device=dev).manual_seed(int(seed))
    return _fitted(case["n"], torch.from_numpy(g.src.astype(np.int64)).to(dev),
                   torch.from_numpy(g.dst.astype(np.int64)).to(dev), gen)


def _start(n, seed):
    return graphs.uniform_positions(n, 2.0 * math.sqrt(n), seed + 1)


def _finished(n, seed):
    """Positions like those of a finished layout: nodes around 32 centres, dense in the middle."""
    rng = np.random.default_rng(seed + 2)
    centre = rng.normal(size=(32, 2)) * 8.0 * math.sqrt(n)
    spread = math.sqrt(n) * rng.exponential(size=(n, 1))
    return (centre[rng.integers(32, size=n)] + spread * rng.normal(size=(n, 2))).astype(np.float32)


def _options(case, n, rowptr, col, seed):
    """Given masses per node and edge weights per CSR entry (the same both ways), or None."""
    rng = np.random.default_rng(seed + 3)
    mass = weight = None
    if case.get("masses"):
        mass = (1.0 + np.diff(rowptr) * rng.uniform(0.5, 1.5, n)).astype(np.float32)
    if case.get("weights"):
        node = rng.uniform(0.5, 2.0, n).astype(np.float32)
        weight = node[np.repeat(np.arange(n), np.diff(rowptr))] * node[col]
    return mass, weight


def _params(case):
    return dict(strong_gravity=case.get("strong", 0), gravity=1.0, scale=case.get("scale", 10.0),
                group_size=case.get("group", 32), linlog=case.get("linlog", 0),
                edge_weight_influence=1.0 if case.get("weights") else 0.0,
                use_barneshut=0 if case.get("allpairs") else 1)


def _batch(case, seed):
    """Barabasi-Albert graphs sized as the batched workload's are, each with its start."""
    rng = np.random.default_rng(2)
    nodes = np.rint(np.exp(rng.uniform(math.log(100.0), math.log(20000.0), case["graphs"]))).astype(int)
    links = rng.integers(2, 9, case["graphs"])
    made = []
    for k, (n, m) in enumerate(zip(nodes.tolist(), links.tolist())):
        g = workloads.host_graph(*graphs.barabasi_albert(n, m, (seed << 20) + k))
        made.append((g, _start(g.n, (seed << 20) + k)))
    return made


def _targets(n, seed):
    """A training target: 32 clusters of a layout, by node order (an SBM's blocks are runs of ids)."""
    return _finished(n, seed + 5)


_PARAMS = 10_498


def _weights(seed):
    """Network weights of the size training leaves them at."""
    rng = np.random.default_rng(seed + 6)
    return (rng.normal(size=_PARAMS) * 0.12).astype(np.float32)


def _offsets(case, seed):
    return np.random.default_rng(seed + 7).integers(1, case["n"] // 2, case["offsets"]).astype(np.int32)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        made = _batch(case, seed)
        engine = BatchEngine([(g.n, g.src, g.dst) for g, _ in made], **workloads.BATCH_PARAMS)
        engine.set_positions(np.concatenate([p for _, p in made]))
        return dict(kind=kind, case=case, engine=engine)
    if kind == "grad":
        n, rowptr, col = _graph(dict(family="sbm", n=case["n"]), seed)
        net = Mpnn(seed=0)
        net.set_params(_weights(seed))
        gid = net.add_graph(n, rowptr, col, target=_targets(n, seed), feature_seed=seed, steps=case["smooth"])
        return dict(kind=kind, case=case, net=net, gid=gid, offsets=_offsets(case, seed))
    n, rowptr, col = _graph(case, seed)
    mass, weight = _options(case, n, rowptr, col, seed)
    engine = Engine(n, rowptr=rowptr, col=col, mass=mass, **_params(case))
    state = dict(kind=kind, case=case, engine=engine, nodes=n, edges=int(rowptr[-1]) // 2, seed=seed)
    if weight is not None:
        engine.set_edge_weights(weight)
    if kind == "forces":
        state["start"] = _start(n, seed)
        return state
    if kind == "layout":
        engine.set_positions(_start(n, seed))
        if case.get("tune"):
            engine.autotune(10)
        if case.get("capture"):
            engine.set_graph_capture(True)
        return state
    if kind == "start":
        state["net"] = Mpnn(seed=0)
        state["net"].set_params(_weights(seed))
        return state
    engine.set_positions(_finished(n, seed))
    return state


# ---- one pass ---------------------------------------------------------------------------------


def run(state):
    kind, case = state["kind"], state["case"]
    if kind == "grad":
        loss, grad = state["net"].loss_grad(state["gid"], state["offsets"])
        return {"loss": loss, "grad": grad}
    engine = state["engine"]
    if kind in ("layout", "batch"):
        engine.step(case["steps"])
        engine.sync()
        return {"positions": engine.positions()}
    if kind == "forces":
        engine.set_positions(state["start"])
        engine.reset()
        engine.step(1)
        engine.sync()
        return {"forces": engine.forces(), "positions": engine.positions()}
    if kind == "start":
        net = state["net"]
        gid = net.add_engine_graph(engine, feature_seed=state["seed"], steps=case["smooth"])
        net.infer_to_engine(gid, 1000.0, engine)
        net.release_graph(gid)
        return {"positions": engine.positions()}
    if kind == "render":
        frame = png_frame(engine.bbox(), case["width"], case["height"], state["nodes"], state["edges"])
        return {"picture": engine.render(frame)}
    pairs = engine.stress_setup(case["sources"], case["targets"], seed=state["seed"])
    a, b, d = engine.stress_pairs()
    ns, alpha = engine.normalized_stress()
    return {"pairs": pairs, "a": a, "b": b, "hops": d, "stress": ns, "alpha": alpha}


# ---- what a pass cannot do without --------------------------------------------------------------


def _size(case):
    """Nodes and undirected edges, nearly (a random graph's are known once it is drawn)."""
    kind, family = case["kind"], case.get("family", "rmat")
    if kind == "batch":
        return 3_700 * case["graphs"], 18_500 * case["graphs"]
    if kind == "grad" or family == "sbm":
        return case["n"], int(4.25 * case["n"])
    return case["n"], case["m"] * case["n"] if family == "ba" else case["edges"]


def work(case):
    v, e = _size(case)
    kind = case["kind"]
    csr = 4 * (v + 1) + 8 * e
    if kind in ("layout", "batch", "forces"):
        # per iteration: positions and previous forces read and written, masses, the CSR once
        near = v if case.get("allpairs") else 35.0 * math.log2(max(4.0, v / 32))
        each = 36 * v + csr + (8 * e if case.get("weights") else 0)
        steps = case.get("steps", 1)
        return {"bytes": steps * each + 8 * v, "flops": steps * (12.0 * v * near + 8.0 * e)}
    dense = 2.0 * v * (2 * 16 * 64 + 2 * 64 * 64 + 2 * 64)
    if kind == "grad":
        return {"bytes": csr + (64 + 8) * v + 8 * _PARAMS, "flops": 3 * dense + 2 * 2 * e * (16 + 2 * 64)}
    if kind == "start":
        return {"bytes": csr + 16 * v, "flops": dense + 2 * e * (8 * case["smooth"] + 16 + 64)}
    if kind == "render":
        pixels = case["width"] * case["height"]
        return {"bytes": csr + 8 * v + pixels, "flops": e * 4.0 * 0.2 * case["width"]}
    pairs = case["sources"] * case["targets"]
    return {"bytes": csr + 8 * v + 16 * pairs, "flops": 2.0 * e * math.ceil(case["sources"] / 64) * 6}


# ---- 64-bit values ------------------------------------------------------------------------------


def _t(x, dev):
    return torch.as_tensor(np.asarray(x), device=dev)


def _tree_repulsion(pos, mass, scale, group):
    """Barnes-Hut repulsion with theta = 1: the quadtree of the float32 positions (cells of two or
    more bodies, 32 levels), walked by runs of `group` bodies in tree order, a cell opened unless
    every body of the run is far enough. Sums in 64 bits."""
    dev, n = pos.device, len(pos)
    eps = float(np.float32(0.05 * 0.05))
    p32 = pos.float()
    lo, hi = p32.min(0).values, p32.max(0).values
    radius = ((hi - lo).max() * 0.5).float()
    centre = ((lo + hi) * 0.5).expand(n, 2).clone()
    key = torch.zeros(n, dtype=torch.int64, device=dev)
    r = radius.clone()
    for _ in range(32):
        r = r * 0.5
        up = centre < p32
        key = key * 4 + up[:, 0].long() + 2 * up[:, 1].long()
        centre = centre + torch.where(up, r, -r)
    order = (key ^ (-(1 << 63))).sort(stable=True).indices
    key, p, m = key[order], pos[order], mass[order]
    pm = torch.cat([torch.zeros(1, 3, dtype=torch.float64, device=dev),
                    torch.cat([p * m[:, None], m[:, None]], 1).cumsum(0)])
    force = torch.zeros(n, 2, dtype=torch.float64, device=dev)
    runs = (n + group - 1) // group
    member = torch.arange(runs, device=dev)[:, None] * group + torch.arange(group, device=dev)
    real = member < n
    member = member.clamp(max=n - 1)
    acc = torch.zeros(runs, group, 2, dtype=torch.float64, device=dev)

    def add(which, xy, mm):
        for a in range(0, len(which), 1 << 18):
            w = which[a:a + (1 << 18)]
            d = p[member[w]] - xy[a:a + (1 << 18), None]
            f = d * (mm[a:a + (1 << 18), None] / ((d * d).sum(2) + eps))[..., None]
            acc.index_add_(0, w, f)

    # a frontier of (run, cell) pairs, level by level; a cell is a range [first, end) of bodies
    run_of = torch.arange(runs, device=dev)
    first = torch.zeros(runs, dtype=torch.int64, device=dev)
    end = torch.full((runs,), n, dtype=torch.int64, device=dev)
    far = float((2.0 * radius.double()) ** 2)
    for level in range(1, 34):
        if level <= 32:
            shift = 64 - 2 * level
            top = (key >> shift) if shift else key
            new = torch.ones(n + 1, dtype=torch.bool, device=dev)
            new[1:n] = top[1:] != top[:-1]
        else:
            new = torch.ones(n + 1, dtype=torch.bool, device=dev)
        starts = new.nonzero().flatten()
        index = new.long().cumsum(0) - 1
        k0, k1 = index[first], index[end]
        reps = k1 - k0
        run_of = run_of.repeat_interleave(reps)
        off = torch.arange(len(run_of), device=dev) - (reps.cumsum(0) - reps).repeat_interleave(reps)
        cell = k0.repeat_interleave(reps) + off
        first, end = starts[cell], starts[cell + 1]
        s = pm[end] - pm[first]
        single = end - first == 1
        xy = torch.where(single[:, None], p[first], s[:, :2] / s[:, 2:])
        mm = torch.where(single, m[first], s[:, 2])
        ok = single.clone()
        ask = (~single).nonzero().flatten()
        for a in range(0, len(ask), 1 << 18):
            q = ask[a:a + (1 << 18)]
            d = p[member[run_of[q]]] - xy[q, None]
            ok[q] = ((((d * d).sum(2) + eps) >= far * 0.25 ** (level - 1) + eps) | ~real[run_of[q]]).all(1)
        add(run_of[ok], xy[ok], mm[ok])
        run_of, first, end = run_of[~ok], first[~ok], end[~ok]
        if not len(run_of):
            break
    force[order] = scale * acc.reshape(-1, 2)[:n] * m[:, None]
    return force


def _all_repulsion(pos, mass, scale):
    eps = float(np.float32(0.05 * 0.05))
    out = torch.zeros_like(pos)
    for a in range(0, len(pos), 512):
        d = pos[a:a + 512, None] - pos[None]
        w = mass[None] / ((d * d).sum(2) + eps)
        out[a:a + 512] = (d * w[..., None]).sum(1)
    return scale * out * mass[:, None]


def _one_iteration(case, seed):
    """Forces of the start and positions after one iteration."""
    dev = _device()
    n, rowptr, col = _graph(case, seed)
    mass, weight = _options(case, n, rowptr, col, seed)
    degree = np.diff(rowptr)
    m = _t(degree + 1.0 if mass is None else mass, dev).double()
    p = _t(_start(n, seed), dev).double()
    rows, cols = _t(np.repeat(np.arange(n), degree), dev), _t(col, dev).long()
    scale = case.get("scale", 10.0)
    f = _all_repulsion(p, m, scale) if case.get("allpairs") else _tree_repulsion(p, m, scale, case.get("group", 32))
    d = p[cols] - p[rows]
    if case.get("linlog"):
        length = d.norm(dim=1)
        d = d * torch.where(length > 0, torch.log1p(length) / length, 0.0)[:, None]
    if weight is not None:
        d = d * _t(weight, dev).double()[:, None]
    f.index_add_(0, rows, d)
    pull = m if case.get("strong") else m / p.norm(dim=1)
    f -= p * pull[:, None]
    # the adaptive speed from its initial state (previous forces are zero)
    size = f.norm(dim=1)
    swing, traction = float((m * size).sum()), float((m * size).sum()) / 2
    tolerance = 0.05 * math.sqrt(n)
    jitter = max(math.sqrt(tolerance), min(10.0, tolerance * traction / n ** 2))
    efficiency = 1.0
    if swing / traction > 2.0:
        efficiency, jitter = 0.5, max(jitter, 1.0)
    target = jitter * efficiency * traction / swing
    speed = 1.0 + min(target - 1.0, 0.5)
    moved = p + f * (speed / (1.0 + (speed * size).sqrt()))[:, None]
    return {"forces": f.cpu().numpy(), "positions": moved.cpu().numpy()}


def _mean_over_neighbours(rows, cols, degree, h):
    s = torch.zeros_like(h).index_add_(0, rows, h[cols])
    return s / degree.clamp(min=1)[:, None]


def _features(n, rows, cols, degree, seed, smooth):
    """log(degree + 1) and 8 smoothed normal fields, standardised, padded to 16 columns."""
    def mix(z):
        z = z + np.uint64(0x9E3779B97F4A7C15)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        return z ^ (z >> np.uint64(31))

    r = mix(np.uint64(seed) ^ mix(np.arange(n * 8, dtype=np.uint64)))
    u1 = ((r >> np.uint64(40)).astype(np.float64) + 0.5) / 16777216.0
    u2 = ((r >> np.uint64(16)) & np.uint64(0xFFFFFF)).astype(np.float64) / 16777216.0
    z = _t((np.sqrt(-2.0 * np.log(u1)) * np.cos(2.0 * np.pi * u2)).reshape(n, 8), rows.device)
    for _ in range(smooth):
        z = 0.5 * (z + _mean_over_neighbours(rows, cols, degree, z))
    x = torch.cat([torch.log(degree + 1.0)[:, None], z], 1)
    x = (x - x.mean(0)) / ((x * x).mean(0) - x.mean(0) ** 2).sqrt()
    return torch.cat([x, torch.zeros(n, 7, dtype=torch.float64, device=x.device)], 1)


def _network(w, rows, cols, degree, x):
    cut = np.cumsum([1024, 1024, 64, 4096, 4096, 64, 128, 2])[:-1].tolist()
    w1s, w1n, b1, w2s, w2n, b2, wo, bo = torch.tensor_split(w, cut)
    h = torch.relu(x @ w1s.view(16, 64) + _mean_over_neighbours(rows, cols, degree, x) @ w1n.view(16, 64) + b1)
    h = torch.relu(h @ w2s.view(64, 64) + _mean_over_neighbours(rows, cols, degree, h) @ w2n.view(64, 64) + b2)
    return h @ wo.view(64, 2) + bo


def _learned(case, seed):
    dev = _device()
    n, rowptr, col = _graph(case if case["kind"] == "start" else dict(family="sbm", n=case["n"]), seed)
    degree = _t(np.diff(rowptr), dev).double()
    rows, cols = _t(np.repeat(np.arange(n), np.diff(rowptr)), dev), _t(col, dev).long()
    x = _features(n, rows, cols, degree, seed, case["smooth"])
    w = torch.from_numpy(_weights(seed)).bfloat16().double().to(dev)    # weights are held in bfloat16
    if case["kind"] == "start":
        y = _network(w, rows, cols, degree, x)
        y = y - y.mean(0)
        return {"positions": (y * (1000.0 / (y * y).sum(1).mean().sqrt())).cpu().numpy()}
    w.requires_grad_(True)
    y = _network(w, rows, cols, degree, x)
    t = _t(_targets(n, seed), dev).double()
    t = t - t.mean(0)
    t = (t / (t * t).sum(1).mean().sqrt()).float().double()     # the registered target is float32
    ids = torch.arange(n, device=dev)
    i, j = [rows], [cols]
    for o in _offsets(case, seed).tolist():
        i += [ids, ids]
        j += [(ids + o) % n, (ids - o) % n]
    i, j = torch.cat(i), torch.cat(j)
    loss = (((y[i] - y[j]).norm(dim=1) - (t[i] - t[j]).norm(dim=1)) ** 2).mean()
    grad, = torch.autograd.grad(loss, w)
    return {"loss": float(loss.detach()), "grad": grad.cpu().numpy()}


def _stress(case, seed):
    """Hop distances of the engine's seeded pairs by breadth-first search, and their stress."""
    dev = _device()
    n, rowptr, col = _graph(case, seed)
    rows, cols = _t(np.repeat(np.arange(n), np.diff(rowptr)), dev), _t(col, dev).long()
    k, t = min(case["sources"], n), case["targets"]
    # SplitMix64 draws: a partial shuffle for the sources, then the targets among the other nodes
    z = np.uint64(seed) + np.arange(1, k + k * t + 1, dtype=np.uint64) * np.uint64(0x9E3779B97F4A7C15)
    z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    z = z ^ (z >> np.uint64(31))
    perm = np.arange(n)
    for i in range(k):
        j = i + int(z[i]) % (n - i)
        perm[i], perm[j] = perm[j], perm[i]
    source = perm[:k]
    target = (z[k:] % np.uint64(n - 1)).astype(np.int64).reshape(k, t)
    target += target >= source[:, None]
    source, target = _t(source, dev), _t(target, dev)
    hops = torch.zeros(k, t, dtype=torch.float64, device=dev)
    for a in range(0, k, 64):
        width = min(64, k - a)
        front = torch.zeros(n, width, device=dev)
        front[source[a:a + width], torch.arange(width, device=dev)] = 1.0
        seen, level = front > 0, 0
        while front.any():
            level += 1
            near = torch.zeros(n, width, device=dev).index_add_(0, rows, front[cols])
            front = ((near > 0) & ~seen).float()
            seen |= front > 0
            hit = front.t().gather(1, target[a:a + width]) > 0
            hops[a:a + width] = torch.where(hit, float(level), hops[a:a + width])
    p = _t(_finished(n, seed), dev).double()
    r = ((p[source][:, None] - p[target]).norm(dim=2) / hops)[hops > 0]
    s1, s2 = float(r.sum()), float((r * r).sum())
    return {"pairs": None, "a": None, "b": None, "hops": None, "stress": 1.0 - s1 * s1 / (len(r) * s2),
            "alpha": s1 / s2}


def exact(case, seed):
    kind = case["kind"]
    if kind == "forces":
        return _one_iteration(case, seed)
    if kind == "layout" and case["steps"] == 1:
        return {"positions": _one_iteration(case, seed)["positions"]}
    if kind in ("grad", "start"):
        return _learned(case, seed)
    if kind == "stress":
        return _stress(case, seed)
    # several iterations follow a trajectory that any rounding turns; a picture is whole numbers
    return None
