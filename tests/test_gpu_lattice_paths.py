"""The distinct-entry product (lattice.hip) against the dense one, with the path that
each run took made sure of: what the solver holds on the device at the start of the
run is far less than the dense tensor, or more than it.

* The rule that chooses between them (host arithmetic, read from the library).
* Rows of single columns (n % 4 != 0) that are longer than a wavefront: several
  tiles of 64 receivers to a grid row, runs of columns that start inside a row; several
  planes with rows of whole and of ragged quads, several receiver rows to a wavefront
  and rows longer than one; several planes of single columns, where one state runs on
  the table and two on the dense tensor.  Same bits as the dense rows.
* A state that is not finite in FP32: within a plane the xz and yz entries are +-0
  and their products are left out, unless a packed state held an infinity or a NaN.
  The same fields are then NaN or infinite as in the dense run, and the batch's other
  states keep their bits.  The state comes in by each of the launches that pack one:
  the stage combination, the right-hand side that forms the next stage, and the
  backward pass.
"""

import numpy as np
import pytest

MU0 = 4 * np.pi * 1e-7


@pytest.fixture
def held(monkeypatch):
    """Device bytes that a solver (a gradient) holds when its run starts."""
    import torch
    from magtense_amd import _lib

    L = _lib.lib()
    seen = {}

    def watch(create, run):
        made, ran = getattr(L, create), getattr(L, run)

        def before(*a):
            torch.cuda.synchronize()
            seen["free"] = torch.cuda.mem_get_info()[0]
            return made(*a)

        def at(*a):
            seen["bytes"] = seen["free"] - torch.cuda.mem_get_info()[0]
            return ran(*a)

        monkeypatch.setattr(L, create, before)
        monkeypatch.setattr(L, run, at)

    watch("mt_solver_create", "mt_solver_run")
    watch("mt_rk4_create", "mt_rk4_forward")
    return seen


def _problem(res, m0, path):
    from magtense.micromag import MicromagProblem

    return MicromagProblem(list(res), [4e-9 * res[0], 3.7e-9 * res[1], 3e-9 * res[2]], m0=m0[0], alpha=4.42e3,
                           gamma=2.21e5, tol=1e-5, filename=path)


def _both(res, m0, held, tmp_path):
    """Fields and magnetizations of the batch m0 by the table and by the dense tensor."""
    n, out, used = int(np.prod(res)), [], []
    h = np.linspace(-0.03, 0.03, len(m0))[:, None] * np.array([1.0, 0.3, 0.0]) / MU0
    for path in ("t", str(tmp_path / "tensor.bin")):
        out.append(_problem(res, m0, path).run_simulation_batch(
            2e-13, 2, [lambda t, v=v: np.ones((len(t), 1)) * v for v in h], 4, m0, return_fields=True))
        used.append(held["bytes"])
    assert used[1] >= 24 * n * n and used[0] < used[1] - 12 * n * n, "this grid is not taken by the table"
    return out


def _unit(rng, states, n):
    m0 = rng.normal(size=(states, n, 3))
    return m0 / np.linalg.norm(m0, axis=2, keepdims=True)


# measured with both forms (lattice.hip); the listed lines of the rule
@pytest.mark.parametrize("res,states,pays", [
    ((32, 32, 1), 64, False), ((32, 40, 1), 8, False), ((32, 40, 1), 9, False), ((64, 17, 1), 9, True),
    ((64, 30, 1), 16, True), ((96, 24, 1), 8, True), ((96, 24, 1), 16, False), ((128, 32, 1), 1, True),
    ((128, 32, 1), 64, True), ((32, 33, 2), 4, True), ((32, 33, 2), 8, False), ((32, 33, 2), 12, False), ((64, 12, 3), 9, False), ((64, 16, 4), 12, True),
    ((48, 16, 4), 8, False), ((64, 16, 4), 8, True), ((64, 16, 4), 24, False), ((256, 64, 2), 64, True),
    ((77, 33, 1), 1, False), ((91, 41, 1), 4, True), ((91, 41, 1), 8, False), ((63, 57, 1), 12, True),
    ((63, 57, 1), 24, False), ((45, 41, 2), 1, False), ((67, 19, 3), 2, False), ((65, 49, 3), 1, False),
    ((45, 79, 3), 1, True), ((45, 79, 3), 2, False), ((91, 93, 1), 24, True)])
def test_rule(res, states, pays):
    import ctypes

    from magtense_amd import _lib

    f = _lib.load()["_ZN2mt12lattice_paysEiiii"]  # mt::lattice_pays(int, int, int, int)
    f.argtypes, f.restype = [ctypes.c_int] * 4, ctypes.c_bool
    assert f(*res, states) is pays


@pytest.mark.gpu
@pytest.mark.parametrize("res,states", [([91, 71, 1], 1), ([77, 47, 1], 3), ([99, 37, 1], 2), ([63, 57, 1], 9),
                                        ([90, 30, 1], 5), ([20, 110, 1], 6), ([64, 18, 1], 9), ([32, 33, 2], 3),
                                        ([20, 20, 6], 4), ([16, 9, 16], 2), ([90, 14, 2], 3), ([130, 6, 3], 1),
                                        ([64, 22, 3], 9), ([128, 17, 2], 12)])
def test_table_equals_dense(res, states, held, tmp_path):
    m0 = _unit(np.random.default_rng(4), states, int(np.prod(res)))
    got, ref = _both(res, m0, held, tmp_path)
    for a, b in zip(got, ref):
        assert np.array_equal(a.view(np.int64), b.view(np.int64))


@pytest.mark.gpu
def test_odd_planes_one_state_and_two(held):
    """10665 cells in three planes: one state on the table, two on the dense tensor."""
    res, n = [45, 79, 3], 10665
    m0 = _unit(np.random.default_rng(12), 2, n)
    h = np.array([[2e4, 0.0, 0.0], [-1e4, 5e3, 0.0]])

    def run(k):
        return _problem(res, m0[k], "t").run_simulation_batch(
            2e-13, 2, [lambda t, v=v: np.ones((len(t), 1)) * v for v in h[k]], 4, m0[k], return_fields=True)

    both = run([0, 1])
    assert held["bytes"] >= 24 * n * n
    for k in (0, 1):
        one = run([k])
        assert held["bytes"] < 12 * n * n
        for a, b in zip(both, one):
            assert np.array_equal(a[k].view(np.int64), b[0].view(np.int64))


@pytest.mark.gpu
@pytest.mark.parametrize("res", [[64, 36, 1], [45, 79, 1], [32, 33, 2], [90, 14, 2]])
@pytest.mark.parametrize("component", [0, 2])
def test_state_beyond_fp32_in_a_solver(res, component, held, tmp_path):
    """1e39 in one cell of one state: finite in FP64, an infinity in FP32."""
    n = int(np.prod(res))
    m0 = _unit(np.random.default_rng(9), 3, n)
    m0[1, n // 3, component] = 1e39
    got, ref = _both(res, m0, held, tmp_path)
    for a, b in zip(got, ref):
        assert np.array_equal(a[[0, 2]].view(np.int64), b[[0, 2]].view(np.int64))
        assert np.isfinite(a[[0, 2]]).all()
        assert np.array_equal(a[1], b[1], equal_nan=True)
    demag = got[4][1, 0]  # (t, m, exchange, external, demag, anisotropy) of the state at t = 0
    assert np.isnan(demag[np.arange(n) // (res[0] * res[1]) == n // 3 // (res[0] * res[1])]).any(axis=1).all()


@pytest.mark.gpu
@pytest.mark.parametrize("where", ["m0", "stage", "cotangent"])
@pytest.mark.parametrize("res,states,alone", [([64, 18, 1], 9, "dense"), ([32, 33, 2], 5, "table")])
def test_non_finite_state_in_a_gradient(res, states, alone, where, held):
    """A state of the batch and the state alone, one of them on the table and one on the
    dense tensor.  m0: 1e39; stage: finite in FP32 at first, beyond it in the second
    stage's argument; cotangent: finite states, an infinite dL/dm(T)."""
    import torch
    from magtense_amd.adjoint import ll_rk4

    n, bad = int(np.prod(res)), 2
    rng = np.random.default_rng(6)
    m0 = _unit(rng, states, n)
    w = rng.normal(size=m0.shape)
    if where == "m0":
        m0[bad, n // 2, 2] = 1e39
    elif where == "stage":
        m0[bad, n // 2, 2] = 1e24
    else:
        w[bad, n // 2, 2] = np.inf
    h = torch.tensor(rng.normal(size=(states, 3)) * 1e4, requires_grad=True)
    ms = torch.tensor(rng.uniform(7e5, 9e5, n))
    m0, w = torch.tensor(m0, requires_grad=True), torch.tensor(w)
    args = (ms, res, [4e-9 * res[0], 4e-9 * res[1], 3e-9 * res[2]], 2e-14, 2)
    mT = ll_rk4(m0, h, *args, checkpoint_every=2)
    g = torch.autograd.grad(mT, [m0, h], w)
    batch = held["bytes"]
    for b in (0, bad, states - 1):
        one = ll_rk4(m0[b:b + 1], h[b:b + 1], *args, checkpoint_every=2)
        gb = torch.autograd.grad(one, [m0, h], w[b:b + 1])
        if alone == "dense":
            assert held["bytes"] >= 24 * n * n and batch < held["bytes"]
        else:
            assert batch >= 24 * n * n and held["bytes"] < batch - 12 * n * n
        for x, y in ((mT[b], one[0]), (g[0][b], gb[0][b]), (g[1][b], gb[1][b])):
            x, y = x.detach().numpy(), y.detach().numpy()
            assert np.array_equal(x, y, equal_nan=True)
            assert np.isfinite(x).all() or b == bad
    assert not torch.isfinite(g[0][bad]).all()
