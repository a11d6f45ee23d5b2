"""The sort order: runs sort their points along a Hilbert curve, while
emst_get_radius_samples describes every point on the Morton order.  The sample
features that do not depend on the leaf cell are checked against a numpy
restatement on Morton keys, at sizes around a leaf and a packet."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _morton_order(resc, dim):
    bits = 16 if dim == 3 else 24
    maxq = np.uint64((1 << bits) - 1)
    scale = np.float32(float(maxq) / float(resc.max()))
    q = np.minimum((resc * scale).astype(np.float32).astype(np.uint64), maxq)
    key = np.zeros(len(q), np.uint64)
    for b in range(bits):
        for k in range(dim):
            key |= ((q[:, k] >> np.uint64(b)) & np.uint64(1)) << np.uint64(dim * b + k)
    return np.argsort(key, kind="stable")


@pytest.mark.parametrize("dim,kind,n", [(2, 0, 9), (3, 0, 65), (2, 1, 4097), (3, 1, 20_000), (2, 2, 5000)])
def test_samples_follow_the_morton_order(pkg, dim, kind, n):
    pts = pkg.synth(kind, n, dim, 400 + n)
    print("case samples", dim, kind, n, flush=True)
    with pkg.Calculateur(dim=dim) as c:
        c.initialize(pts)
        c.run()
        u, v, _ = c.getLinks()
        X, T = c.radius_samples()
        resc, _ = c.getAdaptiveMap()
        cand, cd2 = c.candidates()
        u1, v1, _ = c.getLinks()
    assert np.array_equal(u, u1) and np.array_equal(v, v1)          # the forest is left alone
    order = _morton_order(resc, dim)
    p = resc[order].astype(np.float64)
    off = np.zeros((n, dim))
    total = np.zeros(n)
    for o in (-4, -3, -2, -1, 1, 2, 3, 4):
        a, b = max(0, -o), min(n, n - o)
        d = p[a + o:b + o] - p[a:b]
        off[a:b] += d
        total[a:b] += np.linalg.norm(d, axis=1)
    side = np.linalg.norm(off, axis=1) / np.where(total > 0, total, 1)
    # float32 sums of eight offsets: 2^-24 per operation, relative to their total length
    assert np.max(np.abs(X[:, 7] - side)) <= 64 * 2.0 ** -24
    # the targets are the same points': exp(T) / R is the leaf spacing, positive;
    # points without a candidate are marked -20
    far = np.sqrt(np.where(np.isinf(cd2), -1, cd2).max(axis=1).clip(min=0))[order]
    assert np.array_equal(T == -20, far == 0)
