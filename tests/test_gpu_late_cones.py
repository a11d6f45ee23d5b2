"""Late cones (3D, automatic search form, 4096 points and more): the rounds ask
for a point's far cones only when one could hold its component's edge.  Every
run equals the form that makes all cones first (search_split = 1): edges,
per-round forest sizes and labels; and the cone candidates read afterwards are
all of them exact.  The clouds reach each part: few late points in a round (one
wave each), many (a paused round: isolated clusters), points alone within their
first radius, ties on lattices (edges that fail their check restart the run),
and pairs at float distance zero."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def blobs(rng, n, k, spread):
    return (rng.random((k, 3)) * 100)[rng.integers(0, k, n)] + rng.normal(size=(n, 3)) * spread


def make(kind, n, seed):
    rng = np.random.default_rng(seed)
    if kind == "uniform":
        p = rng.random((n, 3))
    elif kind == "clusters":            # round after round of isolated components
        p = blobs(rng, n, 24, 0.4)
    elif kind == "thin":                # a tenth of the points far from any other
        p = blobs(rng, n, 6, 0.2)
        p[rng.random(n) < 0.1] = 0
        z = np.flatnonzero(~p.any(axis=1))
        p[z] = rng.random((len(z), 3)) * 100
    elif kind == "lattice":             # blocks of a cubic lattice: ties on every edge
        m = int(np.ceil((n / 8) ** (1 / 3)))
        g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)
        p = np.concatenate([g + np.array([a, b, c]) * 4.0 * m for a in (0, 1) for b in (0, 1) for c in (0, 1)])
        p = p[rng.permutation(len(p))]
    elif kind == "slab":                # one coordinate for all: a plane in 3D
        p = rng.random((n, 3))
        p[:, 1] = 0.5
    elif kind == "line":
        p = np.zeros((n, 3))
        p[:, 0] = np.cumsum(rng.random(n) ** 3)
    elif kind == "tiny_pairs":          # pairs whose float distance is zero
        p = blobs(rng, n, 5, 0.5)
        p[:40] = 0
        p[:40, 0] = np.arange(40) * 1e-25
    elif kind == "tiny_far":            # such pairs among thin points whose radius reaches a dense cluster
        p = rng.random((n, 3)) * 100
        p[300:] = np.array([12.0, 12.0, 12.0]) + rng.normal(size=(n - 300, 3)) * 0.1
        p[:40] = 0
        p[:40, 0] = np.arange(40) * 1e-25
    return np.ascontiguousarray(p, np.float32)


def run(pkg, pts, split, step=False, trace=False):
    with pkg.Calculateur(dim=3, search_split=split, trace=trace) as c:
        c.initialize(pts)
        sizes = []
        if step:
            while c.activate():
                sizes.append(c.evaluate()[1])
        else:
            c.run()
        u, v, d = c.getLinks()
        w, m = c.evaluate()
        rows = [(r["size"], r["iteration"]) for r in c.trace()] if trace else None
        out = dict(u=u, v=v, d=d.view(np.uint32), labels=c.labels(), m=m, sizes=sizes, rows=rows)
        cand, cd2 = c.candidates()
        return out, w, cand, cd2.view(np.uint32)


CASES = [(k, n) for k in ("uniform", "clusters", "thin", "lattice", "slab", "line", "tiny_pairs")
         for n in (4096, 5000)] + [("clusters", 60_000), ("thin", 120_000), ("uniform", 65_537), ("lattice", 50_000),
                                            ("tiny_far", 30_000)]


@pytest.mark.parametrize("kind,n", CASES)
def test_late_cones_change_nothing(pkg, kind, n):
    pts = make(kind, n, n + 7)
    print("case late", kind, n, flush=True)
    a, wa, ca, da = run(pkg, pts, 1)
    b, wb, cb, db = run(pkg, pts, 0)
    for k in ("u", "v", "d", "labels"):
        assert np.array_equal(a[k], b[k]), k
    assert a["m"] == b["m"] and abs(wa - wb) <= 1e-12 * wa
    assert np.array_equal(ca, cb) and np.array_equal(da, db)


@pytest.mark.parametrize("kind,n", [("clusters", 60_000), ("thin", 5000), ("lattice", 5000), ("tiny_pairs", 5000),
                                    ("tiny_far", 30_000)])
def test_late_cones_round_by_round(pkg, kind, n):
    """Stepped and traced rounds have the forest sizes of the other form."""
    pts = make(kind, n, n + 11)
    print("case late rounds", kind, n, flush=True)
    a = run(pkg, pts, 1, step=True)[0]
    b = run(pkg, pts, 0, step=True)[0]
    t = run(pkg, pts, 0, trace=True)[0]
    assert a["sizes"] == b["sizes"]
    assert [s for s, _ in t["rows"]][:len(a["sizes"])] == [s for s in a["sizes"]][:len(t["rows"])]
    for k in ("u", "v", "d", "labels"):
        assert np.array_equal(a[k], b[k]) and np.array_equal(a[k], t[k]), k


@pytest.mark.parametrize("kind", ["clusters", "thin", "lattice"])
def test_late_cones_against_the_oracle(pkg, oracle_mod, kind):
    pts = make(kind, 3000, 3)
    print("case late oracle", kind, flush=True)
    ref = oracle_mod.emst(pts, mode=0)
    got = run(pkg, pts, 0)[0]
    assert np.array_equal(np.stack([got["u"], got["v"]], 1).astype(np.int64), oracle_mod.canon(ref["u"], ref["v"]))


def test_candidates_between_rounds(pkg):
    """The candidates are completed in the middle of a run; the run goes on."""
    pts = make("clusters", 20_000, 5)
    ref = run(pkg, pts, 1)
    with pkg.Calculateur(dim=3) as c:
        c.initialize(pts)
        for _ in range(3):
            assert c.activate()
        cand, cd2 = c.candidates()
        while c.activate():
            pass
        u, v, _ = c.getLinks()
    assert np.array_equal(cand, ref[2]) and np.array_equal(cd2.view(np.uint32), ref[3])
    assert np.array_equal(u, ref[0]["u"]) and np.array_equal(v, ref[0]["v"])
