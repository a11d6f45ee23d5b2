"""The radix sort at the edges of its forms (one block up to 8192 pairs, tiles
of 4096 above): the cell grid's listing is a stable sort by cell, checked
against numpy, and the links come out in order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1024, 2048, 2049, 4096, 4097, 8191, 8192, 8193, 12_288, 12_289,
                               16_385, 65_537, 300_001])
@pytest.mark.parametrize("kind", ["spread", "one_place"])
def test_cells_listed_in_order(pkg, n, kind):
    rng = np.random.default_rng(n)
    pts = rng.random((n, 2), dtype=np.float32)
    if kind == "one_place":             # one digit value for nearly all keys
        pts[rng.random(n) < 0.95] = pts[0]
    print("case sort", n, kind, flush=True)
    with pkg.Calculateur(dim=2, round_search=1) as c:
        c.initialize(pts)
        c.run()
        u, v, _ = c.getLinks()
        ext, cell_of, start, listed = c.cell_grid(1)
    cell = cell_of[:, 0].astype(np.int64) + int(ext[0]) * cell_of[:, 1]
    assert np.all(cell_of >= 0)
    assert np.array_equal(listed, np.argsort(cell, kind="stable"))
    assert np.array_equal(start, np.searchsorted(cell[listed], np.arange(int(ext[0]) * int(ext[1]) + 1)))
    assert len(u) == n - 1 and np.all(u < v)
    assert np.all(np.diff(u.astype(np.int64) * n + v) > 0)
