"""FP32 runs on uniform grids take the demag product from the distinct tensor
entries (lattice.hip); a run that writes the tensor to a file holds the dense
tensor instead.  Same entries, same sums in the same order: trajectories and
fields are equal bit for bit, for one state and for batches of every width the
kernel has, on grids with whole and ragged column quads, rows shorter and longer
than a wavefront, one plane and several, and odd cell counts.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MU0 = 4 * np.pi * 1e-7


def _run(res, states, path, seed=3):
    from magtense.micromag import MicromagProblem

    n = int(np.prod(res))
    rng = np.random.default_rng(seed)
    m0 = rng.normal(size=(states, n, 3))
    m0[0, :, 2] = 0.0  # exact zeros among the products
    m0 /= np.linalg.norm(m0, axis=2, keepdims=True)
    p = MicromagProblem(list(res), [4e-9 * res[0], 3.7e-9 * res[1], 3e-9 * res[2]], m0=m0[0], alpha=4.42e3,
                        gamma=2.21e5, tol=1e-5, K0=2e4, filename=path)
    p.u_ea = np.tile([0.0, 0.6, 0.8], (n, 1))
    h = np.linspace(-0.03, 0.03, states)[:, None] * np.array([1.0, 0.3, 0.0]) / MU0
    return p.run_simulation_batch(4e-13, 2, [lambda t, v=v: np.ones((len(t), 1)) * v for v in h], 4, m0,
                                  return_fields=True)


# n % 4 == 0, nx % 4 == 0: 128 (two rows a step), 256 (one), 64, 32, 20 and 16 (several receiver rows a wave);
# 90 (quads that end in the next row), 300 (rows longer than a step); n % 4 != 0 (single columns): 45, 33, 513, 130
@pytest.mark.parametrize("res,states", [([128, 16, 1], 1), ([256, 8, 1], 2), ([64, 33, 1], 3), ([32, 33, 2], 5),
                                        ([20, 20, 4], 9), ([90, 14, 1], 9), ([90, 6, 2], 10), ([45, 41, 2], 3),
                                        ([45, 79, 1], 2), ([33, 107, 1], 1), ([300, 8, 1], 5), ([513, 7, 1], 1),
                                        ([16, 9, 8], 9), ([130, 3, 9], 4)])
def test_lattice_equals_dense(res, states, tmp_path):
    got = _run(res, states, "t")
    ref = _run(res, states, str(tmp_path / "tensor.bin"))
    assert (tmp_path / "tensor.bin").exists()
    for a, b in zip(got, ref):
        assert np.array_equal(a.view(np.int64), b.view(np.int64))


@pytest.mark.parametrize("res", [[64, 20, 1], [60, 11, 2], [32, 11, 3], [45, 79, 1], [64, 36, 1]])
def test_rk4_batch_equals_single_states(res):
    """Of 1025 to 2000 cells a gradient of one state runs on the dense tensor and
    one of nine states on the distinct entries, above both on the entries: the
    same m(T) and gradients."""
    import torch
    from magtense_amd.adjoint import ll_rk4

    n = int(np.prod(res))
    rng = np.random.default_rng(8)
    m0 = rng.normal(size=(9, n, 3))
    m0 /= np.linalg.norm(m0, axis=2, keepdims=True)
    h = torch.tensor(rng.normal(size=(9, 3)) * 1e4, requires_grad=True)
    ms = torch.tensor(rng.uniform(7e5, 9e5, n))
    w = torch.tensor(rng.normal(size=m0.shape))
    m0 = torch.tensor(m0, requires_grad=True)
    L = [4e-9 * res[0], 4e-9 * res[1], 3e-9 * res[2]]
    args = (ms, res, L, 2e-14, 5)
    mT = ll_rk4(m0, h, *args, checkpoint_every=2)
    g = torch.autograd.grad(mT, [m0, h], w)
    for b in (0, 3, 8):
        one = ll_rk4(m0[b:b + 1], h[b:b + 1], *args, checkpoint_every=2)
        gb = torch.autograd.grad(one, [m0, h], w[b:b + 1])
        assert torch.equal(mT[b].view(torch.int64), one[0].view(torch.int64))
        assert torch.equal(g[0][b].view(torch.int64), gb[0][b].view(torch.int64))
        assert torch.equal(g[1][b].view(torch.int64), gb[1][b].view(torch.int64))


@pytest.mark.parametrize("n", [1, 255, 1021, 1024, 2050])
def test_states_per_pass_equal_single_states(n):
    """mt_demag_apply_f32 reads the tensor once for up to eight states; each of
    them has the bits of its own call (whole and partly idle groups, several)."""
    import torch
    from magtense_amd import _lib

    lib = _lib.lib()
    g = torch.Generator(device="cuda").manual_seed(n)
    K = torch.randn(6 * n * n, generator=g, device="cuda")
    m = torch.randn(19, 3, n, generator=g, device="cuda")
    one = torch.empty_like(m)
    for s in range(19):
        _lib.check(lib.mt_demag_apply_f32(K.data_ptr(), n, m[s].data_ptr(), one[s].data_ptr(), 1, -0.7))
    for S in (2, 3, 4, 5, 7, 8, 9, 16, 19):
        h = torch.full_like(m, 7.0)
        _lib.check(lib.mt_demag_apply_f32(K.data_ptr(), n, m.data_ptr(), h.data_ptr(), S, -0.7))
        assert torch.equal(h[:S].view(torch.int32), one[:S].view(torch.int32))
        assert (h[S:] == 7.0).all()
