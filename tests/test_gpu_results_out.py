"""Results on their way to host memory: small ones in one piece, large ones in
chunks by several threads.  Sizes at the edges of both (64 KB, 1 MB per array,
64 MB in all); every array fetched with the others equals the one fetched
alone, which takes another split."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _alone(pkg, c, which, m):
    a = np.full(m + 2, 7, np.float32 if which == 2 else np.int32)      # two words past the end stay
    args = [None, None, None]
    args[which] = a.ctypes.data_as(ctypes.c_void_p)
    k = ctypes.c_int64(m)
    assert pkg.lib().emst_get_edges(c._c, *args, ctypes.byref(k)) == 0 and k.value == m
    assert a[m] == 7 and a[m + 1] == 7
    return a[:m]


@pytest.mark.parametrize("n", [2, 5462, 5463, 16_385, 16_386, 262_145, 262_146, 500_000, 5_592_500])
def test_links_and_labels_arrive_whole(pkg, n):
    print("case results", n, flush=True)
    pts = pkg.synth(0, n, 2, 7)
    with pkg.Calculateur(dim=2, round_search=1) as c:
        c.initialize(pts)
        c.run()
        u, v, d = c.getLinks()
        assert len(u) == n - 1
        assert np.array_equal(u, _alone(pkg, c, 0, n - 1))
        assert np.array_equal(v, _alone(pkg, c, 1, n - 1))
        assert np.array_equal(d.view(np.uint32), _alone(pkg, c, 2, n - 1).view(np.uint32))
        resc, _ = c.getAdaptiveMap()
        labels = c.labels()
    assert np.array_equal(labels, np.full(n, labels[0]))
    assert np.all(u < v) and np.all(np.diff(u.astype(np.int64) * n + v) > 0)
    # the float32 squared distance of the rescaled ends: two rounded squares,
    # fused or not, differ by less than 2 ulp
    e = resc[u].astype(np.float64) - resc[v]
    ref = (e.astype(np.float32).astype(np.float64) ** 2).sum(axis=1)
    assert np.all(np.abs(d - ref) <= 2.0 ** -22 * ref)


@pytest.mark.parametrize("n", [1000, 300_001])
def test_links_straight_into_pinned_memory(pkg, n):
    """Pinned arrays take their copy without the context's slots, next to a
    pageable one that goes through them."""
    print("case pinned results", n, flush=True)
    hip = pkg.lib()
    hip.hipHostMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t, ctypes.c_uint]
    hip.hipHostFree.argtypes = [ctypes.c_void_p]
    pts = pkg.synth(0, n, 2, 9)
    m = n - 1
    with pkg.Calculateur(dim=2, round_search=1) as c:
        c.initialize(pts)
        c.run()
        u, v, d = c.getLinks()
        pin = ctypes.c_void_p()
        assert hip.hipHostMalloc(ctypes.byref(pin), 8 * (m + 1), 0) == 0
        both = np.ctypeslib.as_array(ctypes.cast(pin, ctypes.POINTER(ctypes.c_int32)), (2, m + 1))
        both[:] = 7
        hv = np.full(m + 1, 7, np.int32)
        k = ctypes.c_int64(m)
        assert hip.emst_get_edges(c._c, pin, hv.ctypes.data_as(ctypes.c_void_p),
                                  ctypes.c_void_p(pin.value + 4 * (m + 1)), ctypes.byref(k)) == 0
        got = both.copy()
        assert hip.hipHostFree(pin) == 0
    assert k.value == m and got[0, m] == 7 and got[1, m] == 7 and hv[m] == 7
    assert np.array_equal(u, got[0, :m]) and np.array_equal(v, hv[:m])
    assert np.array_equal(d.view(np.int32), got[1, :m])
