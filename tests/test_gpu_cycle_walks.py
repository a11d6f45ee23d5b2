"""The 2.5D cycle rule where choices form chains longer than a walk (256
hops): pairs of points on a line with growing gaps, each pair's choice being
the pair before it, beside a cloud whose choices close cycles.  Edges and the
number of withheld hooks equal the oracle's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pairs", [100, 256, 257, 258, 700])
@pytest.mark.parametrize("seed", [1, 2])
def test_chains_around_the_walk_limit(pkg, oracle_mod, pairs, seed):
    rng = np.random.default_rng(seed)
    cloud = rng.random((1500, 3), dtype=np.float32) * np.float32([40, 40, 60])
    # gaps 8.0, 8.01, ...: a pair's points are 1 apart
    at = np.cumsum(8.0 + 0.01 * np.arange(pairs))
    line = np.zeros((2 * pairs, 3), np.float32)
    line[0::2, 0] = 500 + at
    line[1::2, 0] = 500 + at
    line[1::2, 1] = 1.0
    pts = np.concatenate([cloud, line]).astype(np.float32)
    pts = pts[rng.permutation(len(pts))]
    print("case walk", pairs, seed, flush=True)
    ref = oracle_mod.emst(pts, mode=0, cdim=2)
    with pkg.Calculateur(dim=3, cone_dim=2) as c:
        c.initialize(pts)
        c.run()
        u, v, _ = c.getLinks()
        cut = pkg.search_stats(c)["cycles_cut"]
    assert ref["cycles_cut"] > 0
    assert cut == ref["cycles_cut"]
    assert np.array_equal(np.stack([u, v], 1).astype(np.int64), oracle_mod.canon(ref["u"], ref["v"]))
