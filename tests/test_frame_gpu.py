"""The bounding sphere folded on the device (point sets of 8,192 points on) equals the host's, bit
for bit, in a new tree and in a reset one."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
_dp = ctypes.POINTER(ctypes.c_double)


def host_sphere(P):
    from voronoids_amd import _lib
    c, r = np.zeros(3), ctypes.c_double()
    _lib.check(_lib.lib().vo_bounding_sphere(P.shape[1], P.ctypes.data_as(_dp), P.shape[0], c.ctypes.data_as(_dp),
                                             ctypes.byref(r)))
    return c[:P.shape[1]].tolist(), 10.0 * (r.value if r.value > 0 else 1.0)


def sets(n, d):
    rng = np.random.default_rng(n + d)
    u = rng.random((n, d))
    yield "uniform", u
    corners = u.copy()
    corners[n // 2], corners[n - 1] = 0.0, 1.0            # on the sphere through the corners: it grows
    yield "corners", corners
    for name, x in (("equal", 0.25), ("zero", 0.0), ("minus zero", -0.0), ("tiny", u * 1e-170), ("huge", u * 1e160)):
        yield name, np.broadcast_to(np.asarray(x), (n, d)).copy()
    flat = u.copy()
    flat[:, d - 1] = np.where(rng.random(n) < 0.5, 0.0, -0.0)
    yield "flat", flat


@pytest.mark.parametrize("d", [2, 3])
@pytest.mark.parametrize("n", [8191, 8192, 8193, 70001])
def test_frame_is_the_hosts(n, d):
    import voronoids_amd as vo
    t = vo.DelaunayTree(np.zeros((0, d)))
    bits = lambda s: np.array(s[0] + [s[1]]).view(np.int64).tolist()
    for name, P in sets(n, d):
        ref = host_sphere(P)
        t.reset(P)
        assert bits(t._root_sphere) == bits(ref), name
        assert bits(vo.DelaunayTree(P)._root_sphere) == bits(ref), name
    assert vo.DelaunayTree(np.zeros((0, d)))._root_sphere == ([0.0] * d, 10.0)


@pytest.mark.parametrize("n", [100, 8192, 50000])
def test_non_finite_points_are_refused_and_leave_the_tree(n):
    import voronoids_amd as vo
    P = np.random.default_rng(3).random((n, 3))
    t = vo.delaunay(P[:50])
    before = t.canonical()
    for bad in (np.nan, np.inf, -np.inf):
        Q = P.copy()
        Q[n - 1, 2] = bad
        for call in (t.reset, vo.DelaunayTree, t.stage):
            with pytest.raises(vo.VoError) as e:
                call(Q)
            assert e.value.code == -1
    after = t.canonical()
    assert all(np.array_equal(a, b) for a, b in zip(before, after))
