"""The register-ring GEMM holds one column half of 32 states or two, with rings of
four and three chunks: a state has the same bits beside 31 others, 32 or 63, for
the dense split-BF16 and FP32 fragments and both block-sparse forms, over chunk
counts below, at and past the rings and the chunks between two flushes (8 and
128)."""

import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [5, 40, 60, 97, 255, 900, 2100, 4130])
@pytest.mark.parametrize("form", ["bf16x2", "f32", "sparse_bf16x2", "sparse_f32"])
def test_one_half_equals_two(n, form):
    import torch
    from magtense_amd import _lib

    lib = _lib.lib()
    rng = np.random.default_rng(n)
    pts = torch.as_tensor(rng.uniform(0, n ** (1 / 3), (n, 3))).cuda()
    d = torch.ones(3, dtype=torch.float64, device="cuda")
    K = torch.empty(6 * n * n, dtype=torch.float32, device="cuda")
    _lib.check(lib.mt_prism_tensor(pts.data_ptr(), d.data_ptr(), 0, None, pts.data_ptr(), n, n, K.data_ptr(), None,
                                   None))
    frags = torch.empty(lib.mt_split_tensor_bytes(n), dtype=torch.uint8, device="cuda")
    h = C.c_void_p()
    if form == "bf16x2":
        _lib.check(lib.mt_split_tensor(K.data_ptr(), n, frags.data_ptr()))
    elif form == "f32":
        _lib.check(lib.mt_f32_mfma_tensor(K.data_ptr(), n, frags.data_ptr()))
    else:
        create = lib.mt_demag_sparse_create_bf16x2 if form == "sparse_bf16x2" else lib.mt_demag_sparse_create_f32_tiles
        _lib.check(create(K.data_ptr(), n, 2, 1e-3, 0, C.byref(h)))
    m = torch.as_tensor(rng.normal(size=(64, 3, n)).astype(np.float32)).cuda()

    def product(S):
        out = torch.full_like(m, 7.0)
        if form == "bf16x2":
            rc = lib.mt_demag_apply_bf16x2(frags.data_ptr(), n, m.data_ptr(), out.data_ptr(), S, -1.0)
        elif form == "f32":
            rc = lib.mt_demag_apply_f32_mfma(frags.data_ptr(), n, m.data_ptr(), out.data_ptr(), S, -1.0)
        else:
            rc = lib.mt_demag_apply_sparse(h, m.data_ptr(), out.data_ptr(), S, -1.0)
        _lib.check(rc)
        assert (out[S:] == 7.0).all()
        return out[:S].view(torch.int32)

    try:
        one, two, full = product(32), product(33), product(64)
        assert torch.equal(one, two[:32]) and torch.equal(two, full[:33])
        K64 = K.cpu().numpy().reshape(6, n, n).astype(np.float64)
        if h:
            K64[np.abs(K64) <= np.float32(1e-3)] = 0.0
        m64 = m[40].cpu().numpy().astype(np.float64)
        ref = -np.stack([sum(K64[[[0, 1, 2], [1, 3, 4], [2, 4, 5]][a][b]] @ m64[b] for b in range(3)) for a in range(3)])
        got = full[40].view(torch.float32).cpu().numpy()
        # split products keep 2^-16 of an entry and of a value, FP32 sums add less
        assert np.linalg.norm(got - ref) <= 2e-5 * np.linalg.norm(ref)
    finally:
        if h:
            lib.mt_demag_sparse_destroy(h)
