"""The cone search's first pass with one lane per query (k_cone_first; reached
by search_split 2 and 3 at any size) and the one-launch form's narrow packets
for few queries: cone minima bit for bit against the oracle's exhaustive ones,
at the edges of packets and leaves, on exact ties, with seeds from far too
small to far too large, and across the clouds of a batch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _check(pkg, oracle_mod, pts, **kw):
    with pkg.Calculateur(dim=pts.shape[1], **kw) as c:
        c.initialize(pts)
        cand, cd2 = c.candidates()
        resc, _ = c.getAdaptiveMap()
    ocid, ocd2, _ = oracle_mod.octants(resc, mode=0)
    assert np.array_equal(cand, ocid)
    assert np.array_equal(cd2.view(np.uint32), ocd2.view(np.uint32))


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("n", [1, 2, 9, 63, 64, 65, 129, 2047])
def test_packet_edges(pkg, oracle_mod, dim, n):
    pts = pkg.synth(1, n, dim, 700 + n)
    for split in (3, 1):
        print("case packets", dim, n, split, flush=True)
        _check(pkg, oracle_mod, pts, search_split=split)


@pytest.mark.parametrize("dim,n", [(2, 2500), (2, 2501), (3, 5001), (2, 5001), (3, 10_001)])
def test_narrow_packets(pkg, oracle_mod, dim, n):
    """One launch: 1, 2, 4 and 8 queries to a packet."""
    print("case narrow", dim, n, flush=True)
    _check(pkg, oracle_mod, pkg.synth(0, n, dim, 720), search_split=1)


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("bucket", [8, 16, 32, 64])
@pytest.mark.parametrize("seed_scale", [0.05, 3.0, 40.0])
def test_leaf_sizes_and_seeds(pkg, oracle_mod, dim, bucket, seed_scale):
    print("case leaves", dim, bucket, seed_scale, flush=True)
    _check(pkg, oracle_mod, pkg.synth(1, 1500, dim, 730), search_split=3, bucket_size=bucket, seed_scale=seed_scale)


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("repeats", [1, 3])
def test_lattice_ties(pkg, oracle_mod, dim, repeats):
    """Every offset of a lattice lies on a boundary between cones or ties with
    another, and with repeats in a coincident group."""
    g = np.stack(np.meshgrid(*[np.arange(32 if dim == 2 else 10)] * dim, indexing="ij"), -1).reshape(-1, dim)
    pts = np.random.default_rng(5).permutation(np.repeat(g, repeats, axis=0)).astype(np.float32)
    print("case lattice", pts.shape, flush=True)
    _check(pkg, oracle_mod, pts, search_split=3)


@pytest.mark.parametrize("dim", [2, 3])
def test_batch_packets_straddle_clouds(pkg, dim):
    sizes = [1, 40, 64, 100, 3, 900, 64, 65, 2]
    clouds = [pkg.synth(i % 3, n, dim, 740 + i) for i, n in enumerate(sizes)]
    print("case straddle", dim, flush=True)
    with pkg.Calculateur(dim=dim, search_split=3) as c:
        c.initialize_clouds(clouds)
        cand, cd2 = c.candidates()
        off = c.offsets
    for i, p in enumerate(clouds):
        with pkg.Calculateur(dim=dim) as c:
            c.initialize(p)
            a, b = c.candidates()
        part = cand[off[i]:off[i + 1]]
        assert np.array_equal(np.where(part >= 0, part - off[i], -1), a)
        assert np.array_equal(cd2[off[i]:off[i + 1]].view(np.uint32), b.view(np.uint32))
