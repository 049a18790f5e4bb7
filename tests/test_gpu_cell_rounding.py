"""The Landau-Lifshitz right-hand side of a cell, bit for bit.

Several kernels evaluate the cell (the LL kernel, the FP32 demag rows, the
near-band kernel), and a batch has the bits of its single runs only if all of them
round alike.  Which products are fused into the following sum is written in
llg_cell.h; here it is restated with the C library's fma and compared with the LL
kernel: exchange and anisotropy fields from m, and dm/dt from m and the fields.
"""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

_fma = ctypes.CDLL("libm.so.6").fma
_fma.restype = ctypes.c_double
_fma.argtypes = [ctypes.c_double] * 3
MU0 = 4.0 * 3.141592653589793 * 1e-7


def fma(a, b, c):
    a, b, c = np.broadcast_arrays(a, b, c)
    return np.array([_fma(x, y, z) for x, y, z in zip(a.ravel(), b.ravel(), c.ravel())]).reshape(a.shape)


def _row(v, axis):
    """Second difference along an axis with the boundary rows (-1, 1) and (1, -1)."""
    v = np.moveaxis(v, axis, 0)
    out = np.empty_like(v)
    out[1:-1] = (v[:-2] - 2.0 * v[1:-1]) + v[2:]  # the product by two is exact
    out[0], out[-1] = v[1] - v[0], v[-2] - v[-1]
    return np.moveaxis(out, 0, axis)


@pytest.mark.parametrize("res,K0", [((5, 4, 3), 3e4), ((6, 5, 1), 0.0), ((2, 2, 2), 1e5)])
def test_cell_rounds_as_written(res, K0):
    import torch
    from magtense_amd import _lib

    nx, ny, nz = res
    n = nx * ny * nz
    rng = np.random.default_rng(n)
    L = [nx * 4.1e-9, ny * 3.7e-9, nz * 2.9e-9]
    m = rng.normal(size=(3, n))
    ms = rng.uniform(6e5, 9e5, n)
    k0 = np.full(n, K0) * rng.uniform(0.5, 1.5, n)
    u = rng.normal(size=(n, 3))
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    hext = np.array([1.3e4, -2.7e4, 5.1e3])
    A0, gamma, alpha = 1.3e-11, 2.21e5, 4.42e3
    K = torch.tensor(rng.normal(size=6 * n * n) * 0.1, dtype=torch.float32, device="cuda")
    dm, dout = torch.tensor(m, device="cuda"), torch.empty((3, n), dtype=torch.float64, device="cuda")
    dF = torch.empty((4, 3, n), dtype=torch.float64, device="cuda")
    lib = _lib.lib()
    _lib.check(lib.mt_ll_rhs(nx, ny, nz, L[0], L[1], L[2], ms.ctypes.data, k0.ctypes.data, u.ctypes.data, A0, gamma,
                             alpha, K.data_ptr(), dm.data_ptr(), hext.ctypes.data, 1, dout.data_ptr(), dF.data_ptr()))
    got, F = dout.cpu().numpy(), dF.cpu().numpy()

    d = [L[0] / nx, L[1] / ny, L[2] / nz if nz > 1 else L[2]]
    w = [1.0 / (s * s) for s in d]
    hj = np.empty((3, n))
    for c in range(3):
        v = m[c].reshape(nz, ny, nx)
        lap = fma(_row(v, 2), w[0], _row(v, 1) * w[1])
        if nz > 1:
            lap = fma(_row(v, 0), w[2], lap)
        hj[c] = (-2.0 * lap).ravel() * (A0 / (MU0 * ms))
    assert np.array_equal(F[0], hj)
    assert np.array_equal(F[1], np.repeat(-hext[:, None], n, axis=1))
    hk = np.zeros((3, n))
    if K0:
        f = -2.0 * (k0 / (MU0 * ms))
        A = [u[:, a] * u[:, b] for a, b in ((0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2))]
        for c, (x, y, z) in enumerate(((0, 1, 2), (1, 3, 4), (2, 4, 5))):
            hk[c] = f * fma(A[z], m[2], fma(A[y], m[1], A[x] * m[0]))
    assert np.array_equal(F[3], hk)

    H = F[1] + F[0] + F[2] + F[3]
    t = [fma(m[(c + 1) % 3], H[(c + 2) % 3], -(m[(c + 2) % 3] * H[(c + 1) % 3])) for c in range(3)]
    x = [fma(m[(c + 2) % 3], t[(c + 1) % 3], -(m[(c + 1) % 3] * t[(c + 2) % 3])) for c in range(3)]
    for c in range(3):
        assert np.array_equal(got[c], fma(gamma, t[c], -(alpha * x[c])))
