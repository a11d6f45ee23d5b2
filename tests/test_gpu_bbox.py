"""The bounding box of one cloud where its kernel's parts end (four points a
thread, 512 blocks of 256 threads): a non-finite coordinate is found wherever
it stands, and extremes at any place give the box's scale, checked against
numpy through the rescaled coordinates."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [2, 255, 256, 257, 1023, 1024, 1025, 524_287, 524_288, 524_289, 700_001]


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("n", SIZES)
def test_nonfinite_found_anywhere(pkg, dim, n):
    rng = np.random.default_rng(n)
    pts = rng.random((n, dim), dtype=np.float32)
    for at, k, bad in ((0, 0, np.nan), (n // 2, dim - 1, -np.inf), (n - 1, dim - 1, np.inf)):
        q = pts.copy()
        q[at, k] = bad
        print("case box", dim, n, at, bad, flush=True)
        with pkg.Calculateur(dim=dim) as c:
            c.initialize(q)
            with pytest.raises(pkg.EmstError) as ei:
                c.run()
            assert ei.value.code == 4


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("n", SIZES)
def test_extremes_found_anywhere(pkg, oracle_mod, dim, n):
    rng = np.random.default_rng(n + 1)
    pts = rng.random((n, dim), dtype=np.float32)
    for k in range(dim):                # each axis' ends at places of their own
        a, b = rng.choice(n, 2, replace=False) if n > 2 * dim else (0, n - 1)
        pts[a, k], pts[b, k] = -1.5 - k, 4.0 + 3 * k
    if n > 2:
        pts[n - 1] = 9.0                # and the last point outside every other
    print("case box", dim, n, flush=True)
    with pkg.Calculateur(dim=dim) as c:
        c.initialize(pts)
        resc, _ = c.getAdaptiveMap()
    want = oracle_mod.rescale(pts)
    want = want[0] if isinstance(want, tuple) else want
    assert np.array_equal(resc.view(np.uint32), np.asarray(want, np.float32).view(np.uint32))
