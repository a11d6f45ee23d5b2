"""Late cones (3D, automatic search form) where distances tie and rounds pause.
Voxel surfaces: the points of a floor one voxel thick lie in flat leaves, whose
first radius ends below one voxel, so they are late; the solid boxes on it have
exact cones, and equal distances meet in components that hold both.  A late
point at exactly its component's smallest distance has to be asked in that
round: its ids may make the smaller edge.  And clouds whose rounds pause (more
than 16384 points listed) against the oracle."""
import numpy as np
import pytest

from test_gpu_late_cones import make

pytestmark = pytest.mark.gpu


def voxels(kind, side, seed):
    rng = np.random.default_rng(seed)
    full = np.zeros((side, side, 24), bool)
    full[:, :, 0] = True
    for _ in range(side // 4):
        a, b = rng.integers(0, side - 12, 2)
        w, d, h = rng.integers(2, 12, 3)
        full[a:a + w, b:b + d, :h] = True
    if kind == "walls":                 # two walls one voxel thick, one with gaps
        full[side // 3, :, :] = True
        full[:, side // 2, ::2] = True
    p = np.argwhere(full).astype(np.float32)
    return np.ascontiguousarray(p[rng.permutation(len(p))])


def run(pkg, pts, split, step):
    with pkg.Calculateur(dim=3, search_split=split) as c:
        c.initialize(pts)
        sizes = []
        if step:
            while c.activate():
                sizes.append(c.evaluate()[1])
        else:
            c.run()
        u, v, d = c.getLinks()
        w, m = c.evaluate()
        return dict(u=u, v=v, d=d.view(np.uint32), labels=c.labels()), sizes, w, m


def against_oracle(oracle_mod, pts, got):
    ref = oracle_mod.emst(pts, mode=0)
    assert np.array_equal(np.stack([got["u"], got["v"]], 1).astype(np.int64), oracle_mod.canon(ref["u"], ref["v"]))
    assert np.array_equal(got["labels"], ref["labels"])
    return ref


@pytest.mark.parametrize("kind,side,seed", [("floor", 160, 1), ("walls", 140, 2), ("floor", 256, 3)])
def test_voxel_surfaces(pkg, oracle_mod, kind, side, seed):
    pts = voxels(kind, side, seed)
    print("case late ties", kind, side, len(pts), flush=True)
    a, sa, wa, ma = run(pkg, pts, 1, True)
    b, sb, wb, mb = run(pkg, pts, 0, True)
    c, _, wc, mc = run(pkg, pts, 0, False)
    assert ma == mb == mc == len(pts) - 1
    assert sa == sb and abs(wa - wb) <= 1e-12 * wa and abs(wa - wc) <= 1e-12 * wa
    for k in ("u", "v", "d", "labels"):
        assert np.array_equal(a[k], b[k]) and np.array_equal(a[k], c[k]), k
    if len(pts) < 50_000:
        ref = against_oracle(oracle_mod, pts, b)
        assert sb == ref["cum_edges"][:len(sb)]


@pytest.mark.parametrize("kind,n", [("clusters", 5000), ("thin", 6000), ("lattice", 8000), ("line", 5000),
                                    ("clusters", 30_000), ("thin", 30_000)])
def test_late_cones_against_the_oracle_at_their_sizes(pkg, oracle_mod, kind, n):
    """Sizes that take late cones (4096 points and more); the clusters of
    30000 points are all late once each is one component, so their rounds
    pause."""
    pts = make(kind, n, n + 3)
    print("case late oracle", kind, n, flush=True)
    got, _, _, m = run(pkg, pts, 0, False)
    assert m == len(pts) - 1
    against_oracle(oracle_mod, pts, got)
