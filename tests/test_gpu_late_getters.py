"""Reading the cone candidates or the search's counters in the middle of a run
with late cones (3D) makes a full search beside it: the candidates are exact,
and the rounds that follow go on in the same form (they search the late points
that still matter; how many those are varies with the order in which a round's
edges are found), to the same forest."""
import numpy as np
import pytest

from test_gpu_late_cones import make

pytestmark = pytest.mark.gpu


def run(pkg, pts, read, split=0):
    with pkg.Calculateur(dim=3, trace=True, search_split=split) as c:
        c.initialize(pts)
        cand = stats = None
        while c.activate():
            if read:
                stats = pkg.search_stats(c)
                cand = c.candidates()
        u, v, d = c.getLinks()
        rows = [(r["size"], r["searched"]) for r in c.trace()]
        return dict(u=u, v=v, d=d.view(np.uint32), labels=c.labels()), rows, cand, stats


@pytest.mark.parametrize("kind,n", [("clusters", 60_000), ("thin", 300_000), ("uniform", 5000), ("tiny_far", 30_000)])
def test_getters_leave_the_run_alone(pkg, kind, n):
    pts = make(kind, n, n + 1)
    print("case late getters", kind, n, flush=True)
    a, ra, _, _ = run(pkg, pts, False)
    b, rb, cand, stats = run(pkg, pts, True)
    assert [s for s, _ in ra] == [s for s, _ in rb]
    for (_, x), (_, y) in zip(ra, rb):
        assert 2 * x <= len(pts) or 4 * y > len(pts)
    for k in ("u", "v", "d", "labels"):
        assert np.array_equal(a[k], b[k]), k
    _, _, (full, full_d2), _ = run(pkg, pts, True, 1)
    assert np.array_equal(cand[0], full) and np.array_equal(cand[1].view(np.uint32), full_d2.view(np.uint32))
    assert stats["pairs"] > 0
