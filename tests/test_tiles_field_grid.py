"""The launch of the magnetostatic field kernel over the whole range of tiles and
points that the entry point takes: a grid holds fewer than 2^32 threads, and the
launches together cover every point (256^3 points of more than 128 tiles are 2^24
blocks of 256 threads).  The plan is host arithmetic and is read from the library
itself; the field over more points than one launch takes equals the field over
parts of them.
"""

import ctypes

import numpy as np
import pytest


class Plan(ctypes.Structure):
    _fields_ = [("width", ctypes.c_int), ("blocks", ctypes.c_int), ("parts", ctypes.c_int)]


def _plan(nt, npt):
    from magtense_amd import _lib

    f = _lib.load()["_ZN2mt16tiles_field_planEii"]  # mt::tiles_field_plan(int, int)
    f.argtypes = [ctypes.c_int, ctypes.c_int]
    f.restype = Plan
    return f(nt, npt)


@pytest.mark.parametrize("nt", [1, 2, 3, 20, 64, 128, 129, 255, 256, 257, 6000, 2 ** 24])
@pytest.mark.parametrize("npt", [1, 255, 5000, 2 ** 24 - 1, 2 ** 24, 2 ** 24 + 1, 10 ** 8, 2 ** 31 - 1])
def test_a_launch_holds_fewer_than_2_32_threads(nt, npt):
    q = _plan(nt, npt)
    assert q.width in (1, 2, 4, 8, 16, 32, 64, 128, 256) and (q.width >= nt or q.width == 256)
    assert 1 <= q.blocks and q.blocks * 256 < 2 ** 32
    assert 1 <= q.parts <= 65535 and (q.parts == 1 or q.blocks * (256 // q.width) >= npt)


@pytest.mark.gpu
def test_field_map_of_256_cubed_points():
    """2^24 + 77 points and 129 prisms: more blocks than one launch holds."""
    from magtense import magstatics as ms

    rng = np.random.default_rng(24)
    t = ms.Tiles(129)
    t.tile_type = [2] * 129
    t.size = rng.uniform(0.05, 0.4, (129, 3))
    t.offset = rng.uniform(-1, 1, (129, 3))
    t.rot = rng.uniform(-3, 3, (129, 3))
    t.M = rng.normal(size=(129, 3)) * 1e5
    n = 2 ** 24 + 77
    pts = rng.uniform(-1.5, 1.5, (n, 3))
    H = ms.get_H_field(t, pts)
    assert H.shape == (n, 3) and np.isfinite(H).all()
    for a in (0, 2 ** 23 - 50, 2 ** 24 - 50, n - 100):  # the ends of launches
        assert np.array_equal(H[a:a + 100], ms.get_H_field(t, pts[a:a + 100]))
