"""The hierarchy's build where its blocks end (256 leaf slots a block, the
levels above in a second launch): clouds of one slot up to several blocks, in
one context and in batches, and in runs of one launch.  A wrong box or id
would lose an edge: the forests equal those of single contexts and of the
cone form."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(pkg, clouds, dim, **kw):
    with pkg.Calculateur(dim=dim, **kw) as c:
        c.initialize_clouds(clouds)
        c.run()
        u, v, d = c.getLinks()
    return u, v, d.view(np.uint32)


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("sizes", [[1], [8], [9], [2048], [2049], [4100], [20_000], [65_000],
                                   [1, 2049, 3, 4100, 64, 1, 9000, 2, 700], [300] * 300])
def test_trees_of_all_sizes(pkg, dim, sizes):
    clouds = [pkg.synth(1 + i % 2, n, dim, 70 + i) for i, n in enumerate(sizes)]
    print("case tree", dim, sizes[:5], flush=True)
    want = _run(pkg, clouds, dim, search_split=1)
    for kw in (dict(round_search=1, bucket_size=8), dict(round_search=1), dict(round_search=1, one_launch=1),
               dict(bucket_size=8, search_split=1)):
        got = _run(pkg, clouds, dim, **kw)
        for x, y in zip(want, got):
            assert np.array_equal(x, y), kw
