"""Late cones (3D) of clusters apart from each other, whose components have no
edge but those that the rounds search for: a point is searched again only when
it can hold its component's edge.  Solid blocks of voxels on a grid of places,
where every gap ties but for rounding, cubes of random points, and blocks at
random places.  The forest is the exact form's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def cloud(kind, n, seed):
    rng = np.random.default_rng(seed)
    if kind == "cubes":
        g = np.argwhere(np.ones((round((n / 1000) ** (1 / 3)),) * 3, bool)) * 3.0
        p = g[rng.integers(0, len(g), n)] + rng.random((n, 3))
    else:
        b = 4 if kind == "blocks4" else 8
        k = round((n / b ** 3) ** (1 / 3))
        g = np.argwhere(np.ones((k,) * 3, bool)) * (b + 8)
        if kind == "scattered":
            g = rng.integers(0, 3 * b * k, (k ** 3, 3))
        q = np.argwhere(np.ones((b,) * 3, bool))
        p = (g[:, None] + q[None]).reshape(-1, 3)
    p = np.unique(np.ascontiguousarray(p, np.float32), axis=0)
    return np.ascontiguousarray(p[rng.permutation(len(p))])


def run(pkg, pts, split):
    with pkg.Calculateur(dim=3, search_split=split, trace=True) as c:
        c.initialize(pts)
        c.run()
        u, v, d = c.getLinks()
        return dict(u=u, v=v, d=d.view(np.uint32), labels=c.labels()), c.trace()


@pytest.mark.parametrize("kind,n", [("blocks4", 30_000), ("blocks4", 110_592), ("blocks8", 175_616), ("cubes", 30_000),
                                    ("cubes", 250_000), ("scattered", 60_000)])
def test_points_are_searched_again_only_for_an_edge(pkg, kind, n):
    pts = cloud(kind, n, n)
    print("case late held", kind, len(pts), flush=True)
    a, ra = run(pkg, pts, 1)
    b, rb = run(pkg, pts, 0)
    assert len(b["u"]) == len(pts) - 1
    for k in ("u", "v", "d", "labels"):
        assert np.array_equal(a[k], b[k]), k
    assert [r["size"] for r in ra] == [r["size"] for r in rb]
    # once while its component has no edge, and once for every tied target that
    # joins: 1.5 of them a point in a block of 4 (24 corner faces, 48 at edges,
    # 24 within faces, of 64 points), fewer elsewhere
    assert sum(r["searched"] for r in rb[1:]) <= 2.5 * len(pts)
