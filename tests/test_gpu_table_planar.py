"""The table products leave out the xz and yz blocks between cells of one plane,
which are exactly zero there, unless a packed state is not finite.

* Finite states give the same bits with and without those products (a fourth
  state holding a NaN brings them all back for every column of the call).
* A NaN or an infinity reaches the same outputs as in the dense product.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _table(res):
    import torch
    from magtense_amd import _lib

    lib = _lib.lib()
    box = [2e-9 * res[0], 2.5e-9 * res[1], 1.5e-9 * res[2]]
    K = torch.empty(lib.mt_toeplitz_tensor_bytes(*res), dtype=torch.uint8, device="cuda")
    _lib.check(lib.mt_toeplitz_tensor(*res, *box, K.data_ptr()))
    return lib, K, box


def _apply(lib, K, res, m):
    import torch
    from magtense_amd import _lib

    dm = torch.as_tensor(m).cuda()
    h = torch.full_like(dm, 7.0)
    _lib.check(lib.mt_demag_apply_bf16x2_toeplitz(K.data_ptr(), *res, dm.data_ptr(), h.data_ptr(), m.shape[0], -1.0))
    return h.cpu().numpy()


# entry-reuse kernel (nx % 128 == 0) and four-tile kernel: one plane, k-splits
# that end inside a plane, more planes than k-splits, groups spanning planes
@pytest.mark.parametrize("res", [[128, 2, 1], [128, 3, 3], [256, 6, 2], [384, 5, 1], [32, 2, 1], [32, 7, 5],
                                 [96, 9, 1], [160, 16, 2], [64, 30, 4]])
def test_planar_steps_same_bits(res):
    lib, K, _ = _table(res)
    rng = np.random.default_rng(5)
    m = rng.normal(size=(4, 3, int(np.prod(res)))).astype(np.float32)
    without = _apply(lib, K, res, m)
    bad = m.copy()
    bad[3, 2, -1] = np.nan
    every = _apply(lib, K, res, bad)
    assert np.array_equal(without[:3].view(np.int32), every[:3].view(np.int32))
    assert np.isnan(every[3]).all()  # 0 x NaN in the in-plane components too


@pytest.mark.parametrize("value", [np.inf, -np.inf, 3.4e38])
def test_infinite_state_reaches_every_component(value):
    """3.4e38 is finite in FP32 and packs to an infinity in BF16."""
    res = [128, 4, 1]
    lib, K, _ = _table(res)
    m = np.zeros((2, 3, 512), dtype=np.float32)
    m[:, 0] = 1.0
    m[1, 2, 7] = value
    h = _apply(lib, K, res, m)
    assert np.isfinite(h[0]).all()
    assert not np.isfinite(h[1]).any()
