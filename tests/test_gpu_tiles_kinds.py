"""Magnetostatic tiles over the kernels' forms and splits: prisms alone,
tetrahedra alone and both with symmetry, from one (tile, point) pair to more
tiles than a block has threads and more points than a part has blocks; and
points in the planes, on the edges and on the corners of a prism's faces, where
the guards of the formula decide.  A call whose input or output is larger than a
pinned block gives the bits of calls on parts of it, and calls of several threads
at once those of calls one by one.

Tolerances: an entry is a sum over eight corners (four faces) of angles and
logarithms of order one, each rounded to 1e-16, over 4 pi: 1e-13 absolute
leaves a factor of a hundred.  A field is the sum over the tiles in another
order: 1e-12 of the largest component.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _tiles(rng, nt, kind):
    from magtense import magstatics as ms

    t = ms.Tiles(nt)
    types = {"prism": np.full(nt, 2), "tetra": np.full(nt, 5), "any": rng.choice([2, 5], nt)}[kind]
    t.tile_type = types.tolist()
    corner = np.array([[0, 0, 0], [0.4, 0, 0], [0, 0.3, 0], [0, 0, 0.2]])
    t.vertices = np.stack([(corner + rng.uniform(-0.05, 0.05, (4, 3))).T for _ in range(nt)])
    t.size = rng.uniform(0.05, 0.4, (nt, 3))
    t.offset = rng.uniform(-1, 1, (nt, 3))
    t.rot = rng.uniform(-3, 3, (nt, 3))
    t.M = rng.normal(size=(nt, 3)) * 1e5
    if kind == "any":
        t.use_sym[::3] = 1
        t.sym_op[::3] = [1.0, -1.0, 1.0]
    return t


def _check(oracle, t, pts):
    from magtense import magstatics as ms

    args = dict(rot=t.rot, tile_type=t.tile_type, use_sym=t.use_sym, sym_ops=t.sym_op, vertices=t.vertices)
    N = ms.get_demag_tensor(t, pts)
    ref = oracle.tiles_tensor(t.size, t.offset, pts, **args)
    assert np.array_equal(np.isfinite(N), np.isfinite(ref))
    ok = np.isfinite(ref)
    assert np.abs(N - ref)[ok].max() <= 1e-13
    Href = oracle.tiles_field(t.size, t.offset, t.M, pts, **args)
    rows = np.isfinite(Href).all(axis=1)
    for H in (ms.get_H_field(t, pts), ms.get_H_field(t, pts, N)):
        assert np.abs(H - Href)[rows].max() <= 1e-12 * np.abs(Href[rows]).max()


@pytest.mark.parametrize("kind", ["prism", "tetra", "any"])
@pytest.mark.parametrize("nt,npt", [(1, 1), (1, 700), (3, 257), (64, 5), (255, 33), (257, 4), (2100, 1)])
def test_kinds_and_splits(oracle, kind, nt, npt):
    rng = np.random.default_rng(17 * nt + npt)
    _check(oracle, _tiles(rng, nt, kind), rng.uniform(-1.5, 1.5, (npt, 3)))


@pytest.mark.parametrize("scale", [1.0, 2.0 ** -30, 2.0 ** 70])
def test_planes_edges_corners(oracle, scale):
    from magtense import magstatics as ms

    t = ms.Tiles(1)
    t.tile_type = [2]
    t.size = np.array([[1.0, 0.5, 0.25]]) * scale  # halves and offsets exact in binary
    t.M = [[1e5, -2e5, 3e5]]
    s = [np.array([-1.0, -h, -h / 2, 0.0, h / 4, h, 2.0]) for h in (0.5, 0.25, 0.125)]
    pts = np.stack(np.meshgrid(*s, indexing="ij"), axis=-1).reshape(-1, 3) * scale
    _check(oracle, t, pts)


def _part(t, a, b):
    from magtense import magstatics as ms

    u = ms.Tiles(b - a)
    u.tile_type = t.tile_type[a:b].tolist()
    u.vertices, u.size, u.offset, u.rot, u.M = t.vertices[a:b], t.size[a:b], t.offset[a:b], t.rot[a:b], t.M[a:b]
    u.use_sym[:], u.sym_op[:] = t.use_sym[a:b], t.sym_op[a:b]
    return u


@pytest.mark.parametrize("nt,npt", [(130, 300), (14000, 2), (9000, 40)])
def test_larger_than_a_block(nt, npt):
    from magtense import magstatics as ms

    rng = np.random.default_rng(nt)
    t, pts = _tiles(rng, nt, "any"), rng.uniform(-1.5, 1.5, (npt, 3))
    N = ms.get_demag_tensor(t, pts)
    for a in range(0, nt, 1000):
        for p in range(0, npt, 20):
            part = ms.get_demag_tensor(_part(t, a, min(a + 1000, nt)), pts[p:p + 20])
            assert np.array_equal(N[a:a + 1000, p:p + 20], part, equal_nan=True)
    H, Hn = ms.get_H_field(t, pts), ms.get_H_field(t, pts, N)  # evaluated and stored tensor: the same sums
    assert np.array_equal(H, Hn, equal_nan=True)


def test_threads():
    import threading

    from magtense import magstatics as ms

    sets, want, bad = [], [], []
    for k, (nt, npt) in enumerate([(3, 900), (40, 17), (200, 190), (1, 1), (75, 60), (500, 2)]):
        rng = np.random.default_rng(k)
        sets.append((_tiles(rng, nt, ("prism", "tetra", "any")[k % 3]), rng.uniform(-1.5, 1.5, (npt, 3))))
        want.append((ms.get_demag_tensor(*sets[-1]), ms.get_H_field(*sets[-1])))

    def work(k):
        for _ in range(40):
            if not (np.array_equal(ms.get_demag_tensor(*sets[k]), want[k][0], equal_nan=True)
                    and np.array_equal(ms.get_H_field(*sets[k]), want[k][1], equal_nan=True)):
                bad.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(sets))]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not bad
