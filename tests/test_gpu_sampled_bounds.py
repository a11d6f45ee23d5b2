"""The component search's sampled bounds (3D, 65536 points and more in the
context, few large components): one cloud and batches of them, leaf sizes of
both kinds, ties on lattices.  The forests are those of the form that makes
every cone first."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _lattices(m, gap):
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)
    return np.concatenate([g + np.array([a, b, 0]) * gap for a in (0, 1, 2) for b in (0, 1)]).astype(np.float32)


def _run(pkg, clouds, bucket, **kw):
    with pkg.Calculateur(dim=3, bucket_size=bucket, **kw) as c:
        c.initialize_clouds(clouds)
        c.run()
        u, v, d = c.getLinks()
        w, e, r = c.cloud_results()
    return u, v, d.view(np.uint32), w, e, r


@pytest.mark.parametrize("bucket", [64, 16])
@pytest.mark.parametrize("case", [[65_535], [65_536], [200_001], [70_000, 1, 500, 40_003], [3000] * 40, "lattices"])
def test_forests_equal(pkg, case, bucket):
    print("case sampled", case if isinstance(case, str) else case[:4], bucket, flush=True)
    if case == "lattices":
        clouds = [_lattices(24, 900)]
    else:
        clouds = [pkg.synth(3, n, 3, 40 + i) for i, n in enumerate(case)]
    a = _run(pkg, clouds, bucket, round_search=1)
    b = _run(pkg, clouds, 0, round_search=0, search_split=1)
    for x, y in zip(a[:3] + a[4:], b[:3] + b[4:]):
        assert np.array_equal(x, y)
    assert np.all(np.abs(a[3] - b[3]) <= 1e-12 * np.abs(b[3]))
