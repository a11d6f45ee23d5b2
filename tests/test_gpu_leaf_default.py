"""Leaves of the 2D cone search: 32 points, 16 where a seed model or its samples
describe them, whether the model is set before the points or after."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _model(pkg):
    return np.load(os.path.join(os.path.dirname(pkg.__file__), "models", "radius_2d.npy"))


def _tree(c):
    c.run()
    u, v, d = c.getLinks()
    return u, v, d.view(np.uint32)


@pytest.mark.parametrize("n", [2, 31, 33, 20_000, 600_000])
def test_one_tree_whatever_the_leaves(pkg, n):
    print("case leaf default", n, flush=True)
    pts = pkg.synth(1, n, 2, 23)
    with pkg.Calculateur(dim=2, bucket_size=16, seed_scale=3.0) as c:
        c.initialize(pts)
        ref = _tree(c)
    with pkg.Calculateur(dim=2) as c:
        c.initialize(pts)
        plain = _tree(c)
        c.set_radius_model(_model(pkg))     # after the points
        after = _tree(c)
        c.initialize(pts)                   # before the points
        before = _tree(c)
    for got in (plain, after, before):
        for x, y in zip(got, ref):
            assert np.array_equal(x, y)


@pytest.mark.parametrize("n", [33, 20_000])
def test_samples_describe_leaves_of_16(pkg, n):
    pts = pkg.synth(0, n, 2, 29)
    got = []
    for kw in ({}, {"bucket_size": 16, "seed_scale": 3.0}):
        with pkg.Calculateur(dim=2, **kw) as c:
            c.initialize(pts)
            got.append(c.radius_samples())
    for x, y in zip(*got):
        assert np.array_equal(x.view(np.uint32), y.view(np.uint32))
