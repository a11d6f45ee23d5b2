"""The calls that users of this framework make, at the sizes they make them.

Every case is one pass from a point cloud to its Euclidean minimum spanning
tree (or forest) through the package's public entry points: points in, the
whole edge list with its squared distances, and the weight out.  The sizes are
those of the repository's own configurations (10^4 to 10^7 points, the TSPLIB
sweep's instances, the batches of clouds), with odd ones among them.

A case is a dict of plain values:
  n, dim     points and their dimension (n is left out for a batch)
  cloud      "uniform", "gauss" (64 Gaussians and background), "power"
             (power-law centres), "gauss8" (eight Gaussians) or "cities"
             (integer coordinates, with ties and repeated places)
  search     "cone" (the default form) or "component" (a search every round)
  source     "device" (points resident on the GPU) or "host" (a numpy array)
  call       "tree"     initialize, run, getLinks, evaluate on a kept context
             "oneshot"  emst(points): a context made and given back inside
             "rounds"   activate() round by round with the forest's weight
                        after each, then the links and the labels
             "batch"    many clouds in one call, per-cloud results and links
  options    cone_dim (2.5D mode), learned (the shipped seed-radius model),
             one_launch, labels (the disjoint-set labels too)
"""
import importlib
import math
import os

import numpy as np
import torch

PACKAGE = "component-based-2d-3d-nns-to-gpu-parallel-2d-3d-emst_amd"
KINDS = {"uniform": 0, "gauss": 1, "power": 2, "gauss8": 3}


def _pkg():
    return importlib.import_module(PACKAGE)


def _case(name=None, **kw):
    c = {"cloud": "uniform", "search": "cone", "source": "device", "call": "tree", "cone_dim": 0, "learned": False,
         "one_launch": False, "labels": False}
    c.update(kw)
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # a TSPLIB instance as a tool reads it: a thousand cities in a host
        # array, integer coordinates, the default form; latency counts
        _case("cities_2d_1k", n=1379, dim=2, cloud="cities", source="host"),
        # a script's one call on 10^4 points in the plane
        _case("oneshot_2d_10k", n=10_000, dim=2, source="host", call="oneshot"),
        # one frame of a stream of 3D scans, with the labels for its clusters
        _case("scan_3d_131k", n=131_071, dim=3, cloud="gauss8", search="component", labels=True),
        # the forest after every round, as the reference's trace writes it
        _case("rounds_3d_200k", n=200_003, dim=3, cloud="uniform", call="rounds"),
        # 10^6 points in the default form, in the plane and in space
        _case("uniform_2d_1m", n=1_000_000, dim=2),
        _case("uniform_3d_1m", n=1_000_000, dim=3),
        # terrain: 3D points, cones over the xy plane
        _case("terrain_2p5d_3m", n=3_000_017, dim=3, cloud="gauss", cone_dim=2),
        # the cone form on a large clustered cloud, with the shipped seed model
        _case("learned_3d_4m", n=4_194_301, dim=3, cloud="gauss", learned=True),
        # the two headline clouds, in the form that large clouds are run in
        _case("power_2d_10m", n=10_000_000, dim=2, cloud="power", search="component"),
        _case("clustered_3d_10m", n=10_000_000, dim=3, cloud="gauss", search="component"),
        # many clouds at once: a service's batch of mixed sizes, and a replayed
        # batch of small ones as a single launch
        _case("batch_3d_512", clouds=512, lo=100, hi=100_000, layout=5, dim=3, cloud="gauss8", search="component",
              call="batch"),
        _case("replay_2d_256", clouds=256, lo=100, hi=10_000, layout=7, dim=2, cloud="uniform", search="component",
              call="batch", one_launch=True),
    ]


def _log_size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))))) | rng.randrange(2)


def draw(rng):
    form = rng.choice(["tree", "tree", "tree", "tree", "oneshot", "rounds", "terrain", "learned", "batch"])
    dim = rng.choice([2, 3])
    cloud = rng.choice(["uniform", "gauss", "power", "gauss8"])
    if form == "tree":
        search = rng.choice(["cone", "component"])
        if rng.random() < 0.25:
            return _case(n=_log_size(rng, 500, 200_000), dim=2, cloud="cities", source="host", search=search)
        return _case(n=_log_size(rng, 1000, 4_000_000 if search == "cone" else 9_000_000), dim=dim, cloud=cloud,
                     search=search, source=rng.choice(["device", "device", "host"]), labels=rng.random() < 0.3)
    if form == "oneshot":
        return _case(n=_log_size(rng, 500, 300_000), dim=dim, cloud=cloud, source="host", call="oneshot")
    if form == "rounds":
        return _case(n=_log_size(rng, 1000, 1_000_000), dim=dim, cloud=cloud, call="rounds",
                     search=rng.choice(["cone", "component"]))
    if form == "terrain":
        return _case(n=_log_size(rng, 2000, 3_000_000), dim=3, cloud=cloud, cone_dim=2)
    if form == "learned":
        return _case(n=_log_size(rng, 20_000, 4_000_000), dim=dim, cloud=rng.choice(["uniform", "gauss", "power"]),
                     learned=True)
    return _case(clouds=rng.randrange(16, 513), lo=100, hi=rng.choice([3000, 10_000, 100_000]),
                 layout=rng.randrange(1, 1000), dim=dim, cloud=rng.choice(["uniform", "gauss8"]), search="component",
                 call="batch", one_launch=rng.random() < 0.4)


def _sizes(case):
    """Points per cloud: log-uniform between lo and hi, a property of the
    case (a service replays batches of one shape with new points)."""
    r = np.random.default_rng(case["layout"])
    return np.rint(np.exp(r.uniform(math.log(case["lo"]), math.log(case["hi"]), case["clouds"]))).astype(np.int64)


def _points(case, n, seed):
    if case["cloud"] == "cities":
        # a map's grid about 12 times as wide as the mean distance between
        # cities: exact ties of distances are common, a few places repeat
        r = np.random.default_rng(seed)
        side = max(2, int(12 * math.sqrt(n)))
        return r.integers(0, side, size=(n, case["dim"])).astype(np.float32)
    return _pkg().synth(KINDS[case["cloud"]], n, case["dim"], seed)


def _cloud(case, seed):
    """All points of the case, host, n x dim float32."""
    if case["call"] == "batch":
        return np.concatenate([_points(case, int(n), seed * 1_000_003 + i) for i, n in enumerate(_sizes(case))])
    return _points(case, case["n"], seed)


def prepare(case, seed):
    pkg = _pkg()
    pts = _cloud(case, seed)
    state = {"case": case, "pkg": pkg, "points": pts}
    if case["source"] == "device":
        state["device"] = torch.from_numpy(pts).to("cuda:0")
        torch.cuda.synchronize()
    if case["call"] == "batch":
        state["sizes"] = _sizes(case)
    if case["call"] != "oneshot":
        ctx = pkg.Calculateur(dim=case["dim"], cone_dim=case["cone_dim"],
                              round_search=1 if case["search"] == "component" else 0,
                              one_launch=1 if case["one_launch"] else 0)
        if case["learned"]:
            ctx.set_radius_model(np.load(os.path.join(os.path.dirname(pkg.__file__), "models",
                                                      f"radius_{case['dim']}d.npy")))
        state["ctx"] = ctx
    return state


def _padded(a, count, fill):
    out = np.full(count, fill, a.dtype)
    out[:len(a)] = a
    return out


def run(state):
    case = state["case"]
    if case["call"] == "oneshot":
        u, v, d2, w = state["pkg"].emst(state["points"])
        return {"u": u, "v": v, "d2": d2, "weight": w}
    ctx = state["ctx"]
    if case["call"] == "batch":
        ctx.initialize_clouds_device(state["device"].data_ptr(), state["sizes"])
        ctx.run()
        w, edges, rounds = ctx.cloud_results()
        u, v, d2 = ctx.getLinks()
        return {"u": u, "v": v, "d2": d2, "weight": w, "edges": edges, "rounds": rounds}
    if case["source"] == "device":
        ctx.initialize_device(state["device"].data_ptr(), case["n"], case["dim"])
    else:
        ctx.initialize(state["points"])
    out = {}
    if case["call"] == "rounds":
        # one row per round, of the 100 that a run has at most
        out["weight"] = np.zeros(100)
        out["size"] = np.zeros(100, np.int64)
        row = 0
        while ctx.activate():
            out["weight"][row], out["size"][row] = ctx.evaluate()
            row += 1
    else:
        ctx.run()
        out["weight"], out["size"] = ctx.evaluate()
    out["u"], out["v"], out["d2"] = ctx.getLinks()
    if case["cone_dim"]:
        # the 2.5D mode may end with a forest: slots of a whole tree
        slots = max(case["n"] - 1, 0)
        out["u"], out["v"] = _padded(out["u"], slots, -1), _padded(out["v"], slots, -1)
        out["d2"] = _padded(out["d2"], slots, 0)
    if case["labels"] or case["call"] == "rounds":
        out["labels"] = ctx.labels()
    return out


def work(case):
    """Points in once, the tree out once; a squared distance and a root per
    edge are the least arithmetic any method does."""
    clouds = 1
    if case["call"] == "batch":
        sizes = _sizes(case)
        n, clouds = int(sizes.sum()), len(sizes)
    else:
        n = case["n"]
    edges = n - clouds
    nbytes = 4 * case["dim"] * n + 12 * edges
    if case["labels"] or case["call"] == "rounds":
        nbytes += 4 * n
    if case["call"] == "batch":
        nbytes += 16 * clouds
    return {"bytes": nbytes, "flops": edges * 3 * case["dim"]}


EXACT_POINTS = 20_000       # Prim over the complete graph: a few seconds


def _unit(p):
    """The rescale factor: (ceil(w) + 1) / width, w = 2 sqrt(n width / height)
    in 2D and (n width^2 / (height depth))^0.333 in 3D."""
    n = len(p)
    ext = [float(e) for e in p.max(axis=0) - p.min(axis=0)]
    width, height = (e if e > 0 else 1.0 for e in ext[:2])
    w = 2 * math.sqrt(n * width / height)
    if len(ext) == 3 and ext[2] > 0:
        w = (n * width * width / (height * ext[2])) ** 0.333
    return (math.ceil(w) + 1) / width


def _tree(p):
    """Minimum spanning tree of the float32 points p over the complete graph,
    by Prim's method, in the framework's order: the float32 squared distance
    of the rescaled points (each square added by a fused multiply-add), then
    the smaller id, then the larger.  Which edges form the tree is a matter of
    that order wherever distances tie.  Rows (u < v), sorted."""
    n = len(p)
    r = ((p - p.min(axis=0)) * np.float32(_unit(p))).astype(np.float32)
    cols = [np.ascontiguousarray(r[:, k]) for k in range(r.shape[1])]
    best = np.full(n, np.inf, np.float32)
    frm = np.zeros(n, np.int64)
    left = np.ones(n, bool)
    cur, edges = 0, []
    for _ in range(n - 1):
        left[cur] = False
        best[cur] = np.inf
        t = cols[0] - cols[0][cur]
        d = t * t
        for c in cols[1:]:
            t = (c - c[cur]).astype(np.float64)
            d = (d + t * t).astype(np.float32)
        take = left & (d < best)
        tie = np.flatnonzero(left & (d == best))
        for j in tie:
            take[j] = (min(cur, j), max(cur, j)) < (min(frm[j], j), max(frm[j], j))
        best[take] = d[take]
        frm[take] = cur
        at = np.flatnonzero(best == best.min())
        at = at[left[at]]
        nxt = min(at, key=lambda j: (min(frm[j], j), max(frm[j], j)))
        edges.append((min(frm[nxt], nxt), max(frm[nxt], nxt)))
        cur = int(nxt)
    e = np.array(edges, np.int64).reshape(-1, 2)
    return e[np.lexsort((e[:, 1], e[:, 0]))]


def exact(case, seed):
    """The weight of the tree and its squared distances in 64 bits: the first
    on the coordinates given, the second on them times the rescale factor."""
    if case["call"] not in ("tree", "oneshot") or case["cone_dim"] or case["n"] > EXACT_POINTS:
        return None
    p = _cloud(case, seed)
    unit = _unit(p)
    e = _tree(p)
    q = p.astype(np.float64)
    d2 = ((q[e[:, 0]] - q[e[:, 1]]) ** 2).sum(axis=1)
    out = {"u": None, "v": None, "d2": d2 * unit * unit, "weight": math.fsum(np.sqrt(d2).tolist())}
    if case["call"] != "oneshot":
        out["size"] = None
    if case["labels"]:
        out["labels"] = None
    return out
