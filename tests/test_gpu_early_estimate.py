"""RKSUITE's early error estimate (stage 7) goes with the reductions after stage 8
in one launch where it is read with them.  MT_DEFER_EARLY=0 forms it before stage
8 and waits for it: the same sums over the same operands and the same
decisions, so trajectories, fields and counts agree to the bit.  By value for up
to two states in one launch, three and four in two, more from device memory; one
or several blocks a state; results through host lines and, past their number,
through the copy."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("res, B, t_end", [
    ([8, 4, 1], 1, 2e-11), ([8, 4, 1], 2, 2e-11), ([8, 4, 1], 3, 2e-11), ([8, 4, 1], 4, 2e-11),
    ([8, 4, 1], 5, 2e-11), ([8, 4, 1], 70, 5e-12), ([45, 17, 2], 2, 2e-12), ([45, 17, 2], 12, 2e-12),
    ([64, 40, 1], 1, 2e-12), ([64, 40, 1], 3, 2e-12), ([80, 70, 1], 64, 2e-13)])
def test_early_estimate_with_the_final_one(monkeypatch, res, B, t_end):
    from magtense.micromag import MicromagProblem

    n = int(np.prod(res))
    rng = np.random.default_rng(81)
    m0 = rng.normal(size=(B, n, 3))
    m0 /= np.linalg.norm(m0, axis=2, keepdims=True)
    fields = np.stack([np.linspace(-3e4, 3e4, B), 5e3 * np.ones(B), np.zeros(B)], axis=1)
    rows = np.repeat(fields[:, None, :], 4, axis=1)
    out = {}
    for v in ("0", "1"):
        monkeypatch.setenv("MT_DEFER_EARLY", v)
        p = MicromagProblem(res, [r * 4e-9 for r in res], alpha=4.42e3, gamma=2.21e5, tol=1e-6, precision="fp32")
        y = p.run_simulation_batch(t_end, 4, rows, 4, m0, return_fields=True)
        out[v] = y, [(s["steps"], s["f_calls"]) for s in p.last_stats]
    print(res, B, out["1"][1][:3])
    assert out["0"][1] == out["1"][1]
    for a, b in zip(out["0"][0], out["1"][0]):
        assert np.array_equal(a, b)
