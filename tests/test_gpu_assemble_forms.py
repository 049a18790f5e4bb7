"""The two assembly kernels (a pair to a thread for the receiver-major planes,
eight columns to a thread where the split fragments are asked for too) are one
formula: their FP32 and FP64 planes agree bit for bit, over the remainders of
both splits, with one size or a size per source, rotated or not, with points in
the planes of faces, and in whatever unit of length."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_src,n_pts", [(1, 1), (1, 300), (7, 33), (255, 3), (257, 32), (520, 65)])
@pytest.mark.parametrize("rotated,sizes,unit", [(False, False, 1e-9), (True, True, 1.0), (False, True, 1e12)])
def test_planes_and_split_kernels_agree(n_src, n_pts, rotated, sizes, unit):
    import torch
    from magtense_amd import _lib

    L = _lib.lib()
    rng = np.random.default_rng(n_src + 7 * n_pts)
    src = rng.integers(-6, 7, (n_src, 3)) * 0.5 * unit
    abc = (rng.integers(1, 4, (n_src, 3)) if sizes else np.ones((1, 3))) * 0.5 * unit
    pts = rng.integers(-6, 7, (n_pts, 3)) * 0.25 * unit
    rot = None
    if rotated:
        rot = torch.as_tensor(np.linalg.qr(rng.normal(size=(n_src, 3, 3)))[0].copy()).cuda()
    src, abc, pts = (torch.as_tensor(a).cuda() for a in (src, abc, pts))
    pad = -(-n_src // 32) * 32
    rows = -(-n_pts // 32) * 32
    out = []
    for with_split in (False, True):
        K32 = torch.full((6 * n_src * n_pts,), float("nan"), device="cuda")
        K64 = torch.full((6 * n_src * n_pts,), float("nan"), dtype=torch.float64, device="cuda")
        split = torch.zeros(rows * pad * 24, dtype=torch.uint8, device="cuda") if with_split else None
        _lib.check(L.mt_prism_tensor(src.data_ptr(), abc.data_ptr(), 3 if sizes else 0,
                                     None if rot is None else rot.data_ptr(), pts.data_ptr(), n_src, n_pts,
                                     K32.data_ptr(), K64.data_ptr(), None if split is None else split.data_ptr()))
        out.append((K32.view(torch.int32), K64.view(torch.int64)))
    assert torch.equal(out[0][0], out[1][0])
    assert torch.equal(out[0][1], out[1][1])
