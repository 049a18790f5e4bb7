"""The threshold-sparse product's column types and state groups.

* 16-bit columns up to 65536 cells, 32-bit above: host CSR components of five
  entries a row over the whole column range at 65535, 65536 and 65537 cells,
  against the FP64 product.  A field is a sum of 45 products at most, each rounded
  once and added in FP32: 46 * 2^-24 < 3e-6 of the sum of their sizes.
* Any number of states up to 16 (interleaved by one, two or four, one group or
  two) gives every state the bits of its own one-state product, with one handle
  shared by two threads.
"""

import ctypes as C
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

COMP = [[0, 1, 2], [1, 3, 4], [2, 4, 5]]


@pytest.mark.parametrize("n", [65535, 65536, 65537])
def test_column_range(n):
    import scipy.sparse as sp
    from magtense_amd import _lib

    lib = _lib.lib()
    rng = np.random.default_rng(n)
    K, keep = [], []
    for c in range(6):
        col = np.sort(rng.integers(0, n, size=(n, 5)), axis=1)
        col[0, -1] = col[-1, -1] = n - 1
        col[1, 0] = 0
        val = rng.normal(size=(n, 5)).astype(np.float32)
        K.append(sp.csr_matrix((val.ravel().astype(np.float64), col.ravel(), np.arange(0, 5 * n + 1, 5)), shape=(n, n)))
        cols = np.ascontiguousarray(col.ravel() + 1, dtype=np.int32)
        rows = np.arange(1, 5 * n + 2, 5, dtype=np.int32)
        vals = np.ascontiguousarray(val.ravel())
        keep += [cols, rows, vals]
        lib.icl_initDemagMatrices_sparse(C.byref(C.c_int(n)), C.byref(C.c_int(5 * n)), C.byref(C.c_int(c + 1)),
                                         vals.ctypes.data, cols.ctypes.data, rows.ctypes.data)
    m = rng.normal(size=(3, n)).astype(np.float32)
    h = np.zeros((3, n), np.float32)
    lib.icl_MVMult_GetH_sparse(m[0].ctypes.data, m[1].ctypes.data, m[2].ctypes.data, h[0].ctypes.data,
                               h[1].ctypes.data, h[2].ctypes.data, C.byref(C.c_int(n)), C.byref(C.c_float(-1.0)))
    lib.icl_destroy()
    m64 = m.astype(np.float64)
    for a in range(3):
        ref = -sum(K[COMP[a][b]] @ m64[b] for b in range(3))
        size = sum(abs(K[COMP[a][b]]) @ abs(m64[b]) for b in range(3))
        assert np.all(np.abs(h[a] - ref) <= 3e-6 * size + 1e-30)


@pytest.mark.parametrize("n", [1, 63, 500, 1027])
def test_states_share_nothing(n):
    import torch
    from magtense_amd import _lib

    lib = _lib.lib()
    g = torch.Generator(device="cuda").manual_seed(n)
    K = torch.randn(6 * n * n, generator=g, device="cuda")
    m = torch.randn(16, 3, n, generator=g, device="cuda")
    hd = C.c_void_p()
    _lib.check(lib.mt_demag_sparse_create(K.data_ptr(), n, 2, 0.8, C.byref(hd)))
    try:
        one = torch.empty_like(m)
        for s in range(16):
            _lib.check(lib.mt_demag_apply_sparse(hd, m[s].data_ptr(), one[s].data_ptr(), 1, 0.5))
        for S in range(2, 17):
            h = torch.full_like(m, 7.0)
            _lib.check(lib.mt_demag_apply_sparse(hd, m.data_ptr(), h.data_ptr(), S, 0.5))
            assert torch.equal(h[:S].view(torch.int32), one[:S].view(torch.int32)), S
            assert (h[S:] == 7.0).all()
        bad = []

        def work(first, S):
            h = torch.empty_like(m)
            for _ in range(50):
                _lib.check(lib.mt_demag_apply_sparse(hd, m[first:].data_ptr(), h.data_ptr(), S, 0.5))
                if not torch.equal(h[:S].view(torch.int32), one[first:first + S].view(torch.int32)):
                    bad.append((first, S))

        t = [threading.Thread(target=work, args=a) for a in ((0, 3), (5, 8))]
        [x.start() for x in t]
        [x.join() for x in t]
        assert not bad
    finally:
        lib.mt_demag_sparse_destroy(hd)
