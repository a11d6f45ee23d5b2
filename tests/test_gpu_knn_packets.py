"""Neighbour lists with 8, 16, 32 and 64 queries to a packet: sizes at both
sides of each width, and clouds that end inside packets.  The component
search's tree equals the cone search's, which has no lists."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _tree(pkg, pts, dim, search):
    with pkg.Calculateur(dim=dim, round_search=search) as c:
        c.initialize(pts)
        c.run()
        u, v, d = c.getLinks()
        return u, v, d.view(np.uint32), c.evaluate()


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("n", [2, 7, 9, 63_999, 64_001, 127_999, 128_001, 255_999, 256_001])
def test_same_tree_at_every_packet_width(pkg, n, dim):
    print("case packets", n, dim, flush=True)
    pts = pkg.synth(3, n, dim, 17)
    a, b = _tree(pkg, pts, dim, 1), _tree(pkg, pts, dim, 0)
    for x, y in zip(a[:3], b[:3]):
        assert np.array_equal(x, y)
    assert a[3][1] == b[3][1] == n - 1
    assert abs(a[3][0] - b[3][0]) <= 1e-12 * b[3][0]


def test_clouds_that_end_inside_packets(pkg):
    sizes = [1, 5, 8, 13, 2, 64, 3, 1000, 7, 16]
    clouds = [pkg.synth(i % 2, n, 3, 40 + i) for i, n in enumerate(sizes)]
    with pkg.Calculateur(dim=3, round_search=1) as c:
        c.initialize_clouds(clouds)
        c.run()
        w, edges, _ = c.cloud_results()
    for i, pts in enumerate(clouds):
        assert edges[i] == sizes[i] - 1
        if sizes[i] > 1:
            u, v, _, (wi, _) = _tree(pkg, pts, 3, 0)
            assert abs(w[i] - wi) <= 1e-12 * wi
