"""Threshold-sparse products of two to four states, which small matrices gather one
by one and larger ones interleaved: on both sides of the line every state has the
bits of its own call, and what lies behind the last state is left alone.
"""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# entries x (states - 1) against 1.5 M and 2200 a row: all below, two states below and
# three or four above, all above; rows of no entries, of one, of a few per lane
@pytest.mark.parametrize("n,kept", [(1, 1.0), (7, 0.5), (255, 0.02), (256, 0.7), (512, 0.7), (1000, 0.03),
                                    (1000, 0.4), (1501, 0.1)])
def test_states_equal_their_own_calls(n, kept):
    import torch
    from magtense_amd import _lib

    lib = _lib.lib()
    g = torch.Generator(device="cuda").manual_seed(n)
    K = torch.randn(6 * n * n, generator=g, device="cuda")
    K.view(6, n, n)[:, n // 2] *= 1e-3  # a row that the threshold empties
    thr = float(np.quantile(K.abs().cpu().numpy(), 1.0 - kept)) if kept < 1.0 else 0.0
    sp = ctypes.c_void_p()
    _lib.check(lib.mt_demag_sparse_create(K.data_ptr(), n, 2, ctypes.c_double(thr), ctypes.byref(sp)))
    try:
        m = torch.randn(5, 3, n, generator=g, device="cuda")
        one = torch.empty_like(m)
        for s in range(5):
            _lib.check(lib.mt_demag_apply_sparse(sp, m[s].data_ptr(), one[s].data_ptr(), 1, ctypes.c_float(-0.7)))
        for S in (2, 3, 4, 5):
            h = torch.full_like(m, 7.0)
            _lib.check(lib.mt_demag_apply_sparse(sp, m.data_ptr(), h.data_ptr(), S, ctypes.c_float(-0.7)))
            assert torch.equal(h[:S].view(torch.int32), one[:S].view(torch.int32))
            assert (h[S:] == 7.0).all()
    finally:
        lib.mt_demag_sparse_destroy(sp)
