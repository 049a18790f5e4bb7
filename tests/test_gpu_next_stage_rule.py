"""FP32 dense rows: which launches form the next stage argument as well.

The rule's lines, read from the library (host arithmetic): one state above 1024
cells, where the longer kernel costs more than the launch that it saves, gets a
vector launch per stage.  Runs on both sides of a line have the same bits: a state
of a batch and the state alone.
"""

import numpy as np
import pytest

MU0 = 4 * np.pi * 1e-7


@pytest.mark.parametrize("n,states,pays", [
    (256, 1, True), (1024, 1, True), (1024, 64, True), (1025, 1, False), (1080, 1, False), (1530, 1, False),
    (3465, 1, False), (16425, 1, False), (1080, 2, True), (1760, 4, True), (2304, 2, False), (2541, 4, False),
    (1760, 8, False), (1530, 8, False), (1530, 12, True), (3465, 9, True), (2304, 12, False), (1530, 24, False)])
def test_rule(n, states, pays):
    import ctypes

    from magtense_amd import _lib

    f = _lib.load()["_ZN2mt23next_stage_in_rows_paysEii"]  # mt::next_stage_in_rows_pays(int, int)
    f.argtypes, f.restype = [ctypes.c_int, ctypes.c_int], ctypes.c_bool
    assert f(n, states) is pays


@pytest.mark.gpu
@pytest.mark.parametrize("res,states", [([36, 30, 1], 3), ([45, 17, 2], 12), ([45, 25, 1], 2), ([11, 33, 5], 4),
                                        ([12, 14, 13], 9), ([9, 41, 9], 12), ([12, 14, 13], 17),
                                        ([8, 8, 8], 30), ([33, 31, 1], 13), ([2, 2, 1], 10)])
def test_batch_equals_single_states(res, states):
    from magtense.micromag import MicromagProblem

    n = int(np.prod(res))
    rng = np.random.default_rng(n)
    m0 = rng.normal(size=(states, n, 3))
    m0 /= np.linalg.norm(m0, axis=2, keepdims=True)
    h = np.linspace(-0.03, 0.03, states)[:, None] * np.array([1.0, 0.3, 0.0]) / MU0

    def run(k):
        p = MicromagProblem(res, [4e-9 * res[0], 3.7e-9 * res[1], 3e-9 * res[2]], m0=m0[k[0]], alpha=4.42e3,
                            gamma=2.21e5, tol=1e-5, K0=2e4)
        p.u_ea = np.tile([0.0, 0.6, 0.8], (n, 1))
        return p.run_simulation_batch(4e-13, 2, [lambda t, v=v: np.ones((len(t), 1)) * v for v in h[k]], 4, m0[k],
                                      return_fields=True)

    whole = run(list(range(states)))
    for k in (0, states - 1):
        for a, b in zip(whole, run([k])):
            assert np.array_equal(a[k].view(np.int64), b[0].view(np.int64))
