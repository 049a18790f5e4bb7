"""The order of the dense FP32 product's sums, by a numpy restatement: thread T of
256 takes column quads 4 T + 1024 k (n % 4 == 0; columns T + 256 k otherwise),
adds up each quad and then the quads; the 64 threads of a wave join by xor 32, 16,
8, 4, 2, 1 and the four waves in order.  States of a single +1 component make
every product exact, so that FP32 additions alone restate the sums: all bits are
compared, for every group width and with idle states and rows."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _row_sums(K):
    """K (rows, n) float32 -> (rows,)."""
    rows, n = K.shape
    q = 4 if n % 4 == 0 else 1
    pad = -n % (256 * q)
    k = np.pad(K, ((0, 0), (0, pad))).reshape(rows, -1, 256, q)
    t = k[..., 0]
    for c in range(1, q):
        t = t + k[..., c]
    acc = np.zeros((rows, 256), np.float32)
    for s in range(t.shape[1]):
        acc = acc + t[:, s]
    w = acc.reshape(rows, 4, 64)
    for bit in (32, 16, 8, 4, 2, 1):
        w = w + w[..., np.arange(64) ^ bit]
    w = w[..., 0]
    return ((w[:, 0] + w[:, 1]) + w[:, 2]) + w[:, 3]


@pytest.mark.parametrize("n", [1, 3, 64, 255, 260, 1021, 1024, 1534, 2052])
def test_sums_in_order(n):
    import torch
    from magtense_amd import _lib

    lib = _lib.lib()
    rng = np.random.default_rng(n)
    K = rng.normal(size=(6, n, n)).astype(np.float32)
    plane = ((0, 1, 2), (1, 3, 4), (2, 4, 5))
    want = np.stack([[_row_sums(K[plane[a][b]]) for a in range(3)] for b in range(3)])  # component b -> field a
    dK = torch.as_tensor(K).cuda()
    for S in (1, 2, 3, 6, 8, 11, 12, 21, 27):
        m = np.zeros((S, 3, n), np.float32)
        m[np.arange(S), np.arange(S) % 3] = 1.0
        dm = torch.as_tensor(m).cuda()
        h = torch.empty_like(dm)
        _lib.check(lib.mt_demag_apply_f32(dK.data_ptr(), n, dm.data_ptr(), h.data_ptr(), S, 1.0))
        got = h.cpu().numpy()
        for s in range(S):
            assert np.array_equal(got[s] + 0.0, want[s % 3] + 0.0), (n, S, s)  # + 0.0: the sign of a zero
