"""Row lengths of the threshold-sparse product: a lane takes four of its entries at a
time and the up to three left over under a mask.  Rows of 0 to 700 entries, so every
remainder, with another length in each component, against the FP64 product.  A field
is a chain of 3 * 11 fused products a lane, six additions over the lanes and the
factor: 40 roundings, 42 * 2^-24 of the sum of the products' sizes; an entry
counted twice or left out is a few 1e-4 of it or more."""

import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

COMP = [[0, 1, 2], [1, 3, 4], [2, 4, 5]]


def test_row_lengths():
    import scipy.sparse as sp
    from magtense_amd import _lib

    lib, n = _lib.lib(), 700
    rng = np.random.default_rng(9)
    K, keep = [], []
    for c in range(6):
        count = (np.arange(n) + 117 * c) % (n + 1)
        cols = np.concatenate([np.sort(rng.permutation(n)[:k]) for k in count])
        rows = np.concatenate([[0], np.cumsum(count)])
        vals = rng.normal(size=len(cols)).astype(np.float32)
        K.append(sp.csr_matrix((vals.astype(np.float64), cols, rows), shape=(n, n)))
        cols1, rows1 = (cols + 1).astype(np.int32), (rows + 1).astype(np.int32)
        keep += [cols1, rows1, vals]
        lib.icl_initDemagMatrices_sparse(C.byref(C.c_int(n)), C.byref(C.c_int(len(cols))), C.byref(C.c_int(c + 1)),
                                         vals.ctypes.data, cols1.ctypes.data, rows1.ctypes.data)
    m = rng.normal(size=(3, n)).astype(np.float32)
    h = np.zeros((3, n), np.float32)
    lib.icl_MVMult_GetH_sparse(m[0].ctypes.data, m[1].ctypes.data, m[2].ctypes.data, h[0].ctypes.data,
                               h[1].ctypes.data, h[2].ctypes.data, C.byref(C.c_int(n)), C.byref(C.c_float(-1.0)))
    lib.icl_destroy()
    m64 = m.astype(np.float64)
    for a in range(3):
        ref = -sum(K[COMP[a][b]] @ m64[b] for b in range(3))
        size = sum(abs(K[COMP[a][b]]) @ abs(m64[b]) for b in range(3))
        assert np.all(np.abs(h[a] - ref) <= 42 * 2.0 ** -24 * size)
