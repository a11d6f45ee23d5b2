"""The component search where components lie far apart: clusters that become
one component each (every point then searches out to another cluster), clouds
of a batch that finish rounds before the others, and resumed dispatches with
more packets than blocks.  The forests are the cone form's, edge for edge."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(pkg, clouds, dim, round_search):
    with pkg.Calculateur(dim=dim, round_search=round_search) as c:
        c.initialize_clouds(clouds)
        c.run()
        u, v, d = c.getLinks()
        w, e, r = c.cloud_results()
    return u, v, d, w, e, r


@pytest.mark.parametrize("dim,sizes", [
    (3, [150_001]),                                     # one cloud of eight far clusters
    (2, [150_001]),
    (3, [1, 2, 63, 64, 65, 40_000, 129, 7, 8191]),      # clouds done after 0 to 8 rounds
    (2, [3, 64, 30_011, 1, 500, 4097]),
])
def test_far_components_equal_cone_form(pkg, dim, sizes):
    print("case far components", dim, sizes, flush=True)
    clouds = [pkg.synth(3, n, dim, 300 + i) for i, n in enumerate(sizes)]
    a = _run(pkg, clouds, dim, 1)
    b = _run(pkg, clouds, dim, 0)
    for x, y in zip(a, b):
        assert np.array_equal(x.view(np.uint32) if x.dtype == np.float32 else x,
                              y.view(np.uint32) if y.dtype == np.float32 else y)
    assert np.array_equal(a[4], np.array(sizes) - 1)


@pytest.mark.parametrize("dim", [2, 3])
def test_two_far_lattices(pkg, dim):
    """Two lattices with a wide gap: every point of a lattice meets exact ties
    on the way, and the single bridge is as long as many lattice steps."""
    g = np.stack(np.meshgrid(*[np.arange(24 if dim == 3 else 120)] * dim, indexing="ij"), -1).reshape(-1, dim)
    pts = np.concatenate([g, g + np.array([4000] + [0] * (dim - 1))]).astype(np.float32)
    print("case lattices", pts.shape, flush=True)
    a = _run(pkg, [pts], dim, 1)
    b = _run(pkg, [pts], dim, 0)
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
    assert len(a[0]) == len(pts) - 1
