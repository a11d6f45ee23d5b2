"""Late cones (3D) where the first radius could miss: flat leaves (planes and
voxel floors along the axes, whose leaf boxes have no volume) and clouds whose
leaves' spacing is not their points' (rings, a line).  A first pass that
sees next to nothing would leave nearly every point to be searched in every
later round; there the cones are made first.  The forest is the exact form's,
and few points are searched after round 1 (rings apart from each other are
components that the rounds do ask for)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def cloud(kind, n, seed):
    rng = np.random.default_rng(seed)
    if kind == "plane":
        p = rng.random((n, 3))
        p[:, 1] = 0.5
    elif kind == "grid":                # one layer of voxels
        side = int(np.sqrt(n))
        p = np.argwhere(np.ones((side, side, 1), bool))
    elif kind == "floor":               # with boxes on it
        side = int(np.sqrt(n / 1.25))
        full = np.zeros((side, side, 24), bool)
        full[:, :, 0] = True
        for _ in range(side // 4):
            a, b = rng.integers(0, side - 12, 2)
            w, d, h = rng.integers(2, 12, 3)
            full[a:a + w, b:b + d, :h] = True
        p = np.argwhere(full)
    elif kind == "rings":               # circles of points, one for each beam of a scanner
        a = np.tile(np.linspace(0, 2 * np.pi, n // 32, endpoint=False), 32) + rng.random(n // 32 * 32) * 1e-4
        r = np.repeat(1.2 ** np.arange(32) * 2, n // 32)
        p = np.stack([r * np.cos(a), r * np.sin(a), np.repeat(np.zeros(32), n // 32)], 1)
    elif kind == "line":
        p = np.zeros((n, 3))
        p[:, 0] = np.cumsum(rng.random(n) ** 3)
        p = np.unique(p.astype(np.float32), axis=0)
    p = np.ascontiguousarray(p, np.float32)
    return np.ascontiguousarray(p[rng.permutation(len(p))])


def run(pkg, pts, split):
    with pkg.Calculateur(dim=3, search_split=split, trace=True) as c:
        c.initialize(pts)
        c.run()
        u, v, d = c.getLinks()
        rows = c.trace()
        return dict(u=u, v=v, d=d.view(np.uint32), labels=c.labels()), rows


@pytest.mark.parametrize("kind", ["plane", "grid", "floor", "rings", "line"])
@pytest.mark.parametrize("n", [6000, 40_000])
def test_few_points_are_left_to_the_rounds(pkg, kind, n):
    pts = cloud(kind, n, n)
    print("case late blind", kind, len(pts), flush=True)
    a, ra = run(pkg, pts, 1)
    b, rb = run(pkg, pts, 0)
    for k in ("u", "v", "d", "labels"):
        assert np.array_equal(a[k], b[k]), k
    assert [r["size"] for r in ra] == [r["size"] for r in rb]
    if kind != "rings":
        assert sum(r["searched"] for r in rb[1:]) <= len(pts)
