"""Performance cases: the work that users of this framework have it do, through its public entry points.

Kinds of work (``case["kind"]``):

* ``film``     ``MicromagProblem.run_simulation`` of one film, creation to returned fields, in the default
               FP32 arithmetic; uniform grids, or a graded film of unstructured prisms (``graded``).
* ``batch``    ``MicromagProblem.run_simulation_batch``: many independent states in one call.
* ``grad``     ``ll_rk4`` forward and backward: the gradient of a fixed-step integration.
* ``product``  one demag product of the C ABI on device arrays, with a tensor that the program laid out once.
* ``assemble`` one prism tensor of the C ABI on a jittered lattice.
* ``field``    ``get_H_field`` of magnetostatic tiles at points (host arrays in and out).
* ``tensor``   ``get_demag_tensor`` of magnetostatic tiles at points (host arrays in and out).

``exact`` restates the same mathematics in 64 bits with plain torch: the closed-form prism tensor, its
product by FFT convolution (or densely where the cells are no lattice), the Landau-Lifshitz right-hand side,
and RK4 at a step far below the solver's.
"""

import ctypes as C
import math

import numpy as np
import torch

MU0 = 4e-7 * math.pi
GAMMA, ALPHA, A0, MS = 2.21e5, 4.42e3, 1.3e-11, 8e5
F64 = torch.float64


def listed():
    return [
        # the smallest film of the tests and the benchmark: a right-hand side is a few microseconds, so launches,
        # latency and the controller's round trips are all there is
        dict(name="film-32x8x1", kind="film", nx=32, ny=8, nz=1, cx=15.625e-9, cy=15.625e-9, cz=3e-9, t_end=2e-10,
             nt=11, K0=0.0, graded=False),
        # the standard-problem-4 film at the benchmark's resolution, the ordinary single run
        dict(name="film-128x32x1", kind="film", nx=128, ny=32, nz=1, cx=3.90625e-9, cy=3.90625e-9, cz=3e-9,
             t_end=3e-11, nt=6, K0=0.0, graded=False),
        # a small parameter sweep in the default arithmetic on an odd, ragged grid with anisotropy
        dict(name="batch-fp32-45x17x2", kind="batch", nx=45, ny=17, nz=2, cx=4e-9, cy=4e-9, cz=3e-9, t_end=5e-12, nt=3,
             K0=1e4, states=12, precision="fp32"),
        # the headline batch: 64 states of the 32768-cell film, split BF16, from creation to results
        dict(name="batch-bf16x2-256x64x2", kind="batch", nx=256, ny=64, nz=2, cx=2e-9, cy=2e-9, cz=1.5e-9,
             t_end=2e-13, nt=2, K0=0.0, states=64, precision="bf16x2"),
        # the differentiation configuration's film with fewer steps
        dict(name="grad-128x32x1", kind="grad", nx=128, ny=32, nz=1, cx=3.90625e-9, cy=3.90625e-9, cz=3e-9, states=1,
             steps=40, every=20, dt=1e-13, precision="fp32"),
        # the product of the headline metric on the dense tensor (25.8 GB)
        dict(name="product-bf16x2-n32768", kind="product", form="bf16x2", nx=256, ny=64, nz=2, cx=2e-9, cy=2e-9,
             cz=1.5e-9, states=64),
        # the FP32 product for a handful of states, a cell count that is no multiple of anything large
        dict(name="product-fp32-n6300", kind="product", form="fp32", nx=90, ny=70, nz=1, cx=4e-9, cy=4e-9, cz=3e-9,
             states=8),
        # the batched FP32 product on the matrix cores, a ragged batch
        dict(name="product-fp32_mfma-n8192", kind="product", form="fp32_mfma", nx=64, ny=64, nz=2, cx=4e-9, cy=4e-9,
             cz=3e-9, states=33),
        # the threshold-sparse product in the reference's per-state form, for a few states
        dict(name="product-csr-n8192", kind="product", form="csr", nx=128, ny=64, nz=1, cx=4e-9, cy=4e-9, cz=3e-9,
             states=3),
        # tensor assembly on the 16384-prism jittered lattice
        dict(name="assemble-n16384", kind="assemble", points=16384, sources=16384, out="fp32"),
        # the field of several thousand rotated magnets at as many points
        dict(name="field-6000x5000", kind="field", tiles=6000, points=5000, rotated=True, shape="prism"),
        # a handful of magnets on the default 20 x 20 grid of evaluation points, the everyday magnetostatic call
        dict(name="tensor-20x400", kind="tensor", tiles=20, points=400, rotated=False, shape="prism"),
    ]


# ---- drawn cases ------------------------------------------------------------------------------------


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, lo, hi):
    """A film or block of lo to hi cells: odd sides among them, one to four layers."""
    n = _log(rng, lo, hi)
    nz = rng.choice([1, 1, 1, 2, 3, 4])
    ratio = rng.choice([1, 2, 4])
    ny = max(2, int(round(math.sqrt(n / nz / ratio))))
    nx = max(2, int(round(n / nz / ny)))
    if rng.random() < 0.4 and nx >= 32:
        nx = nx // 32 * 32
    elif rng.random() < 0.5:
        nx |= 1
    cx = rng.choice([2e-9, 3.90625e-9, 4e-9, 5e-9])
    return dict(nx=nx, ny=ny, nz=nz, cx=cx, cy=cx, cz=rng.choice([1.5e-9, 3e-9, cx]))


def draw(rng):
    kind = rng.choice(["film", "film", "batch", "batch", "grad", "product", "product", "assemble", "field", "tensor"])
    if kind == "film":
        graded = rng.random() < 0.25
        c = dict(kind=kind, **_grid(rng, 200, 1200 if graded else 6000), nt=rng.randint(2, 12),
                 K0=rng.choice([0.0, 0.0, 2e4]), graded=graded)
        if graded:
            c["ny"], c["nx"], c["nz"] = c["ny"] * c["nz"], c["nx"], 1
        # about the same number of solver steps whatever the cell
        c["t_end"] = 2e-11 * (min(c["cx"], c["cz"] if c["nz"] > 1 else c["cx"]) / 3.90625e-9) ** 2
        return c
    if kind == "batch":
        precision = rng.choice(["fp32", "bf16x2", "fp32_mfma"])
        c = dict(kind=kind, **_grid(rng, 300, 8000), nt=2, K0=rng.choice([0.0, 2e4]), states=_log(rng, 2, 64),
                 precision=precision)
        c["t_end"] = 4e-12 * (min(c["cx"], c["cz"] if c["nz"] > 1 else c["cx"]) / 3.90625e-9) ** 2
        return c
    if kind == "grad":
        g = _grid(rng, 200, 5000)
        return dict(kind=kind, **g, states=rng.randint(1, 4), steps=rng.randint(8, 40), every=rng.choice([7, 10, 20]),
                    dt=1e-13 * min(1.0, (min(g["cx"], g["cz"] if g["nz"] > 1 else g["cx"]) / 3.90625e-9) ** 2),
                    precision=rng.choice(["fp32", "fp32", "fp64"]))
    if kind == "product":
        form = rng.choice(["fp32", "bf16x2", "table", "fp32_mfma", "csr", "tiles_fp32", "tiles_bf16x2"])
        c = dict(kind=kind, form=form, **_grid(rng, 400, 9000), states=_log(rng, 1, 64))
        if form == "table":  # the translation-invariant table is for rows of a multiple of 32 cells
            c["nx"] = max(32, (c["nx"] + 16) // 32 * 32)
        return c
    if kind == "assemble":
        return dict(kind=kind, points=_log(rng, 300, 12000), sources=_log(rng, 300, 12000),
                    out=rng.choice(["fp32", "split", "fp64"]))
    shape = rng.choice(["prism", "prism", "tetra"])
    if kind == "field":
        t = _log(rng, 4, 6000 if shape == "prism" else 1500)
        return dict(kind=kind, tiles=t, points=_log(rng, 50, 5000 if shape == "prism" else 1500),
                    rotated=rng.random() < 0.5, shape=shape)
    return dict(kind=kind, tiles=_log(rng, 4, 1500), points=_log(rng, 50, 1500 if shape == "prism" else 700),
                rotated=rng.random() < 0.5, shape=shape)


# ---- inputs -------------------------------------------------------------------------------------------


def _gen(seed, salt=0):
    return torch.Generator().manual_seed(int(seed) * 7919 + salt)


def _unit(v):
    return v / v.norm(dim=-1, keepdim=True)


def _cells(case):
    return case["nx"] * case["ny"] * case["nz"]


def _res(case):
    return [case["nx"], case["ny"], case["nz"]]


def _box(case):
    return [case["nx"] * case["cx"], case["ny"] * case["cy"], case["nz"] * case["cz"]]


def _widths(case):
    """Column widths of the graded film (10 % steps)."""
    return case["cx"] * (1 + 0.1 * (np.arange(case["nx"]) % 4))


def _smooth(case, g, states):
    """Smooth magnetizations, as relaxed films have them: +-x with a few long waves on top; (states, N, 3)."""
    nx, ny, nz = _res(case)
    z, y, x = torch.meshgrid(torch.arange(nz) / nz, torch.arange(ny) / ny, torch.arange(nx) / nx, indexing="ij")
    m = torch.zeros(states, 3, nz, ny, nx, dtype=F64)
    amp = 0.25 * torch.randn(states, 3, 3, 3, generator=g, dtype=F64)
    for p in range(3):
        for q in range(3):
            wave = torch.cos(math.pi * (p * x + q * y) + 0.3 * z).to(F64)
            m += amp[:, :, p, q, None, None, None] * wave
    m[:, 0] += torch.where(torch.rand(states, generator=g) < 0.5, -1.0, 1.0).to(F64)[:, None, None, None]
    m = m.reshape(states, 3, -1).transpose(1, 2)
    return _unit(m).contiguous()


def _random(case, g, states):
    """Independent random directions in every cell (the batch benchmark's start)."""
    return _unit(torch.randn(states, _cells(case), 3, generator=g, dtype=F64))


def _field(g, states):
    """In-plane applied fields of up to 50 mT, in A/m."""
    h = (torch.rand(states, 3, generator=g, dtype=F64) - 0.5) * 0.1 / MU0
    h[:, 2] = 0
    return h


def _axes(case):
    """Easy axes, one tilted direction for the whole film."""
    return np.tile(np.array([0.6, 0.0, 0.8]), (_cells(case), 1))


def _start(case, seed):
    """(m0, applied field) of a film, batch or gradient case."""
    g = _gen(seed)
    states = case.get("states", 1)
    m0 = _random(case, g, states) if case["kind"] == "batch" and case["precision"] != "fp32" else _smooth(case, g, states)
    return m0, _field(g, states)


def _graded(case):
    """Points, edges and finite-volume exchange operator (dense) of the graded film."""
    nx, ny, w = case["nx"], case["ny"], _widths(case)
    edge = np.concatenate([[0.0], np.cumsum(w)])
    n = nx * ny
    j, i = np.divmod(np.arange(n), nx)
    pts = np.stack([((edge[:-1] + edge[1:]) / 2)[i], (j + 0.5) * case["cy"], np.zeros(n)], axis=1)
    abc = np.stack([w[i], np.full(n, case["cy"]), np.full(n, case["cz"])], axis=1)
    A = np.zeros((n, n))
    for di, dj in ((-1, 0), (1, 0), (0, -1), (0, 1)):
        ok = (i + di >= 0) & (i + di < nx) & (j + dj >= 0) & (j + dj < ny)
        r = np.nonzero(ok)[0]
        k = r + di + dj * nx
        c = 1.0 / (0.5 * (w[i[r]] + w[i[k]]) * w[i[r]]) if di else np.full(len(r), 1.0 / case["cy"] ** 2)
        np.add.at(A, (r, k), c)
        np.add.at(A, (r, r), -c)
    return pts, abc, A


def _lattice(case):
    """Cell centres (host, float64), x fastest, and the cell's edges."""
    res, box = _res(case), _box(case)
    d = [box[k] / res[k] for k in range(3)]
    ax = [np.array([-box[k] / 2 + i * d[k] + d[k] / 2 for i in range(res[k])]) if res[k] > 1 else np.zeros(1)
          for k in range(3)]
    z, y, x = np.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    return np.stack([x.ravel(), y.ravel(), z.ravel()], axis=1), np.array(d)


def _threshold(case):
    """Absolute threshold that drops the far field: the size of an in-plane entry a few cells away."""
    d = 0.18 * math.sqrt(_cells(case)) * case["cx"]
    return case["cx"] * case["cy"] * case["cz"] / (4 * math.pi * d ** 3)


def _prisms(case, seed):
    """Sources, their edges and receivers of the jittered lattice, on the GPU."""
    g = _gen(seed, 3)
    n = max(case["points"], case["sources"])
    side = int(math.ceil(math.sqrt(n)))
    k = torch.arange(n)
    c = torch.stack([k % side, k // side, torch.zeros_like(k)], dim=1).to(F64) * 5e-9
    c[:, :2] += (torch.rand(n, 2, generator=g, dtype=F64) - 0.5) * 1e-9
    abc = (0.8 + 0.4 * torch.rand(n, 3, generator=g, dtype=F64)) * torch.tensor([5e-9, 5e-9, 2e-9], dtype=F64)
    ns, npt = case["sources"], case["points"]
    return c[:ns].contiguous().cuda(), abc[:ns].contiguous().cuda(), c[:npt].contiguous().cuda()


def _tile_arrays(case, seed):
    """Magnets in a decimetre-sized cube and evaluation points around them."""
    rng = np.random.default_rng([int(seed), 11])
    t, p = case["tiles"], case["points"]
    a = dict(size=rng.uniform(0.002, 0.01, (t, 3)), offset=rng.uniform(-0.05, 0.05, (t, 3)),
             rot=rng.uniform(-1.0, 1.0, (t, 3)) if case["rotated"] else np.zeros((t, 3)),
             M=rng.normal(size=(t, 3)) * 6e5, pts=rng.uniform(-0.07, 0.07, (p, 3)))
    base = np.array([[0, 0, 0], [0.008, 0, 0], [0, 0.006, 0], [0, 0, 0.007]])
    a["vertices"] = (base[None] + rng.uniform(-0.001, 0.001, (t, 4, 3))).transpose(0, 2, 1)
    return a


class _Sparse:
    """A threshold-sparse tensor handle, destroyed with the state that holds it."""

    def __init__(self, lib, K, n, form, thr, nx):
        from magtense_amd import _lib

        self.lib, self.h = lib, C.c_void_p()
        if form == "csr":
            rc = lib.mt_demag_sparse_create(K.data_ptr(), n, _lib.DEMAG_THRESHOLD, thr, C.byref(self.h))
        else:
            make = lib.mt_demag_sparse_create_f32_tiles if form == "tiles_fp32" else lib.mt_demag_sparse_create_bf16x2
            rc = make(K.data_ptr(), n, _lib.DEMAG_THRESHOLD, thr, nx if nx % 32 == 0 else 0, C.byref(self.h))
        _lib.check(rc)

    def __del__(self):
        if self.h:
            self.lib.mt_demag_sparse_destroy(self.h)


def prepare(case, seed):
    torch.zeros(1, device="cuda")
    from magtense_amd import _lib

    kind, s = case["kind"], {"case": case}
    if kind in ("film", "batch"):
        from magtense.micromag import MicromagProblem

        m0, h = _start(case, seed)
        n = _cells(case)
        kw = dict(alpha=ALPHA, gamma=GAMMA, tol=1e-6, A0=A0, Ms=MS, K0=case["K0"], m0=m0[0].numpy())
        if case.get("graded"):
            p = MicromagProblem([n, 1, 1], grid_type="unstructuredPrisms", **kw)
            p.grid_pts, p.grid_abc, A = _graded(case)
            p.set_exchange_matrix(A)
        else:
            p = MicromagProblem(_res(case), _box(case), precision=case.get("precision", False), **kw)
        if case["K0"]:
            p.u_ea = _axes(case)
        s.update(problem=p, m0=m0.numpy(), h=h.numpy())
    elif kind == "grad":
        m0, h = _start(case, seed)
        g = _gen(seed, 5)
        ms = MS * (0.9 + 0.2 * torch.rand(_cells(case), generator=g, dtype=F64))
        w = torch.randn(m0.shape, generator=g, dtype=F64) / math.sqrt(m0.numel())
        s.update(m0=m0.requires_grad_(), h=h.requires_grad_(), ms=ms.requires_grad_(), w=w)
    elif kind == "product":
        lib, n, form, S = _lib.lib(), _cells(case), case["form"], case["states"]
        g = torch.Generator(device="cuda").manual_seed(int(seed))
        m = _unit(torch.randn(S, n, 3, generator=g, device="cuda")).transpose(1, 2).contiguous()
        s.update(lib=lib, m=m, h=torch.empty_like(m))
        if form == "table":
            s["K"] = torch.empty(lib.mt_toeplitz_tensor_bytes(*_res(case)), dtype=torch.uint8, device="cuda")
            _lib.check(lib.mt_toeplitz_tensor(*_res(case), *_box(case), s["K"].data_ptr()))
            return s
        pts, d = (torch.as_tensor(a).cuda() for a in _lattice(case))
        split = torch.empty(lib.mt_split_tensor_bytes(n), dtype=torch.uint8, device="cuda") if form == "bf16x2" else None
        K = torch.empty(6 * n * n, dtype=torch.float32, device="cuda") if split is None else None
        _lib.check(lib.mt_prism_tensor(pts.data_ptr(), d.data_ptr(), 0, None, pts.data_ptr(), n, n,
                                       None if K is None else K.data_ptr(), None,
                                       None if split is None else split.data_ptr()))
        if form == "fp32_mfma":
            s["K"] = torch.empty(lib.mt_split_tensor_bytes(n), dtype=torch.uint8, device="cuda")
            _lib.check(lib.mt_f32_mfma_tensor(K.data_ptr(), n, s["K"].data_ptr()))
        elif form in ("csr", "tiles_fp32", "tiles_bf16x2"):
            s["K"] = _Sparse(lib, K, n, form, _threshold(case), case["nx"])
        else:
            s["K"] = K if split is None else split
    elif kind == "assemble":
        src, abc, pts = _prisms(case, seed)
        lib, ns, npt = _lib.lib(), case["sources"], case["points"]
        up = lambda v: (v + 31) // 32 * 32  # noqa: E731
        out = (torch.empty(up(ns) * up(npt) * 24, dtype=torch.uint8, device="cuda") if case["out"] == "split" else
               torch.empty(6, npt, ns, dtype=F64 if case["out"] == "fp64" else torch.float32, device="cuda"))
        s.update(lib=lib, src=src, abc=abc, pts=pts, out=out)
    else:
        from magtense import magstatics

        a = _tile_arrays(case, seed)
        t = magstatics.Tiles(case["tiles"])
        t.tile_type = 5 if case["shape"] == "tetra" else 2
        t.size, t.offset, t.rot, t.M, t.vertices = a["size"], a["offset"], list(a["rot"]), a["M"], a["vertices"]
        s.update(tiles=t, pts=a["pts"])
    return s


# ---- one pass -----------------------------------------------------------------------------------------


def _constant(h):
    return lambda t: np.ones((len(t), 1)) * h


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind == "film":
        return state["problem"].run_simulation(case["t_end"], case["nt"], _constant(state["h"][0]), 10)
    if kind == "batch":
        return state["problem"].run_simulation_batch(case["t_end"], case["nt"], [_constant(h) for h in state["h"]], 10,
                                                     state["m0"])
    if kind == "grad":
        from magtense_amd.adjoint import ll_rk4

        leaves = [state["m0"], state["h"], state["ms"]]
        mT = ll_rk4(*leaves, _res(case), _box(case), case["dt"], case["steps"], checkpoint_every=case["every"], A0=A0,
                    alpha=ALPHA, gamma=GAMMA, demag_precision=case["precision"])
        return [mT.detach(), *torch.autograd.grad(mT, leaves, state["w"])]
    if kind in ("field", "tensor"):
        from magtense import magstatics

        return (magstatics.get_H_field if kind == "field" else magstatics.get_demag_tensor)(state["tiles"], state["pts"])
    from magtense_amd import _lib

    lib = state["lib"]
    if kind == "assemble":
        ptr = {k: None for k in ("fp32", "fp64", "split")} | {case["out"]: state["out"].data_ptr()}
        _lib.check(lib.mt_prism_tensor(state["src"].data_ptr(), state["abc"].data_ptr(), 3, None, state["pts"].data_ptr(),
                                       case["sources"], case["points"], ptr["fp32"], ptr["fp64"], ptr["split"]))
        return state["out"]
    K, m, h, n, S = state["K"], state["m"].data_ptr(), state["h"].data_ptr(), _cells(case), case["states"]
    pref, form = C.c_float(-1.0), case["form"]
    if form == "fp32":
        rc = lib.mt_demag_apply_f32(K.data_ptr(), n, m, h, S, pref)
    elif form == "bf16x2":
        rc = lib.mt_demag_apply_bf16x2(K.data_ptr(), n, m, h, S, pref)
    elif form == "table":
        rc = lib.mt_demag_apply_bf16x2_toeplitz(K.data_ptr(), *_res(case), m, h, S, pref)
    elif form == "fp32_mfma":
        rc = lib.mt_demag_apply_f32_mfma(K.data_ptr(), n, m, h, S, pref)
    else:
        rc = lib.mt_demag_apply_sparse(K.h, m, h, S, pref)
    _lib.check(rc)
    return state["h"]


def work(case):
    """What a pass cannot do without.  A solver or gradient case counts its tensor once per call, and for each
    right-hand side the state read, dm/dt written and the product's operations."""
    kind = case["kind"]
    if kind == "assemble":
        pairs = float(case["points"]) * case["sources"]
        return {"bytes": pairs * (48 if case["out"] == "fp64" else 24), "flops": pairs * 500}
    if kind in ("field", "tensor"):
        pairs = float(case["points"]) * case["tiles"]
        per = 500 if case["shape"] == "prism" else 2000
        return {"bytes": 72 * pairs if kind == "tensor" else 24.0 * case["points"] + 96 * case["tiles"],
                "flops": pairs * per}
    n, S = float(_cells(case)), case.get("states", 1)
    if kind == "product":
        per = 4 if case["form"] != "csr" else 8
        share = 1.0
        if case["form"] in ("csr", "tiles_fp32", "tiles_bf16x2"):  # entries within the threshold's distance
            share = min(1.0, math.pi * 0.18 ** 2)
        tensor = 6 * n * n * per * share
        if case["form"] == "table":  # one entry per cell offset
            tensor = 24.0 * (2 * case["nx"] - 1) * (2 * case["ny"] - 1) * (2 * case["nz"] - 1)
        return {"bytes": tensor + 24 * n * S, "flops": 18 * n * n * S * share}
    if kind == "grad":
        evals = 12.0 * case["steps"]
    else:  # right-hand sides of the solver: eight to a step, a step of about 0.15 ps on 3.9 nm cells
        d2 = (min(case["cx"], case["cz"] if case["nz"] > 1 else case["cx"]) / 3.90625e-9) ** 2
        evals = 8.0 * max(4.0, case["t_end"] / (0.15e-12 * d2))
    tensor = 24 * n * n  # once; on a uniform grid one entry per cell offset
    if not case.get("graded"):
        tensor = 24.0 * (2 * case["nx"] - 1) * (2 * case["ny"] - 1) * (2 * case["nz"] - 1)
    return {"bytes": tensor + evals * S * n * 48, "flops": evals * 18 * n * n * S}


# ---- the same in 64 bits --------------------------------------------------------------------------------


def _prism(a, b, c, x, y, z):
    """Point tensor of a prism with full edges (a, b, c) at offset (x, y, z): minus the demagnetization tensor,
    components xx xy xz yy yz zz (Smith et al. 2010)."""
    hx, hy, hz = (a / 2 - x, a / 2 + x), (b / 2 - y, b / 2 + y), (c / 2 - z, c / 2 + z)
    r = {(i, j, k): torch.sqrt(hx[i] ** 2 + hy[j] ** 2 + hz[k] ** 2) for i in (0, 1) for j in (0, 1) for k in (0, 1)}
    f = 1 / (4 * math.pi)
    diag = [0.0, 0.0, 0.0]
    for (i, j, k), q in r.items():
        diag[0] = diag[0] + torch.atan(hy[j] * hz[k] / (hx[i] * q))
        diag[1] = diag[1] + torch.atan(hx[i] * hz[k] / (hy[j] * q))
        diag[2] = diag[2] + torch.atan(hx[i] * hy[j] / (hz[k] * q))

    def off(h, pick):
        # log of the ratio of (s h + r) over the corners of either parity, s the side along the third axis
        up = down = 1.0
        for key, q in r.items():
            side = pick(key)
            v = (-h[1] if side else h[0]) + q
            if sum(key) % 2 == 0:
                up = up * v
            else:
                down = down * v
        return torch.log(up / down)

    xy, yz, xz = off(hz, lambda q: q[2]), off(hx, lambda q: q[0]), off(hy, lambda q: q[1])
    return [-f * diag[0], f * xy, f * xz, -f * diag[1], f * yz, -f * diag[2]]


_AB = ((0, 1, 2), (1, 3, 4), (2, 4, 5))


class _Lattice64:
    """K m on a uniform grid by FFT convolution; m (S, 3, N) float64 on the GPU."""

    def __init__(self, case):
        self.res = _res(case)
        d = [b / r for b, r in zip(_box(case), self.res)]
        self.pad = [2 * r if r > 1 else 1 for r in self.res]
        ax = []
        for r, p, c in zip(self.res, self.pad, d):
            o = torch.arange(p, device="cuda", dtype=F64)
            ax.append(torch.where(o >= r, o - p, o) * c)
        z, y, x = torch.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
        K = torch.stack(_prism(d[0], d[1], d[2], x, y, z))
        self.K = torch.fft.rfftn(K, dim=(1, 2, 3))

    def __call__(self, m):
        nx, ny, nz = self.res
        shape = self.pad[::-1]
        out = []
        for s in range(0, m.shape[0], 16):
            f = torch.fft.rfftn(m[s:s + 16].reshape(-1, 3, nz, ny, nx), s=shape, dim=(2, 3, 4))
            h = torch.stack([sum(self.K[_AB[a][b]] * f[:, b] for b in range(3)) for a in range(3)], dim=1)
            h = torch.fft.irfftn(h, s=shape, dim=(2, 3, 4))[:, :, :nz, :ny, :nx]
            out.append(h.reshape(h.shape[0], 3, -1))
        return torch.cat(out)


def _dense(K, m):
    out = [sum(m[:, b] @ K[_AB[a][b]].T for b in range(3)) for a in range(3)]
    return torch.stack(out, dim=1)


class _Film64:
    """The four negated effective fields and dm/dt of a film in 64 bits; m (S, 3, N)."""

    def __init__(self, case, h, ms):
        self.case, self.h, self.ms = case, h[:, :, None], ms
        if case.get("graded"):
            pts, abc, A = (torch.as_tensor(a).cuda() for a in _graded(case))
            d = pts[:, None] - pts[None]
            K = torch.stack(_prism(abc[:, 0], abc[:, 1], abc[:, 2], d[..., 0], d[..., 1], d[..., 2]))
            self.K, self.A = (lambda m: _dense(K, m)), A
        else:
            self.K = _Lattice64(case)

    def lap(self, m):
        if self.case.get("graded"):
            return m @ self.A.T
        nx, ny, nz = _res(self.case)
        v = m.reshape(*m.shape[:2], nz, ny, nx)
        out = torch.zeros_like(v)
        for dim, n, c in ((4, nx, self.case["cx"]), (3, ny, self.case["cy"]), (2, nz, self.case["cz"])):
            if n > 1:  # second differences, the outer neighbour missing at the walls
                step = (v.narrow(dim, 1, n - 1) - v.narrow(dim, 0, n - 1)) / c ** 2
                zero = torch.zeros_like(step.narrow(dim, 0, 1))
                out = out + torch.cat([step, zero], dim) - torch.cat([zero, step], dim)
        return out.reshape(m.shape)

    def fields(self, m):
        exc = -2 * self.lap(m) * (A0 / (MU0 * self.ms))
        dem = -self.K(m) * self.ms
        ani = torch.zeros_like(m)
        if self.case.get("K0"):
            u = torch.as_tensor(_axes(self.case)).cuda().T[None]
            ani = -2 * self.case["K0"] / (MU0 * self.ms) * u * (u * m).sum(1, keepdim=True)
        return exc, -self.h.expand_as(m), dem, ani

    def rhs(self, m):
        H = sum(self.fields(m))
        c = torch.linalg.cross(H, m, dim=1)
        return -GAMMA * c - ALPHA * torch.linalg.cross(m, c, dim=1)

    def step(self, m, dt):
        k1 = self.rhs(m)
        k2 = self.rhs(m + dt / 2 * k1)
        k3 = self.rhs(m + dt / 2 * k2)
        k4 = self.rhs(m + dt * k3)
        return m + dt / 6 * (k1 + 2 * k2 + 2 * k3 + k4)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("film", "batch"):
        m0, h = _start(case, seed)
        ms = torch.tensor(MS, dtype=F64, device="cuda")
        f = _Film64(case, h.cuda(), ms)
        m = m0.transpose(1, 2).contiguous().cuda()
        cell = min(case["cx"], case["cz"] if case["nz"] > 1 else case["cx"])
        t = np.linspace(0, case["t_end"], case["nt"])
        steps = int(math.ceil(t[1] / (5e-14 * (cell / 3.90625e-9) ** 2)))
        seen = [m]
        for _ in range(case["nt"] - 1):
            for _ in range(steps):
                m = f.step(m, t[1] / steps)
            seen.append(m)
        if kind == "batch":
            return np.tile(t, (m.shape[0], 1)), torch.stack(seen, 1).transpose(2, 3).contiguous().cpu()
        out = torch.stack(seen)  # (nt, 1, 3, N) -> (nt, N, 1, 3)
        H = [torch.stack(q) for q in zip(*(f.fields(v) for v in seen))]
        M, *H = [v.permute(0, 3, 1, 2).cpu() for v in (out, *H)]
        pts = _graded(case)[0] if case["graded"] else _lattice(case)[0]
        return t, M, pts, *H
    if kind == "grad":
        s = prepare(case, seed)
        m0, h, ms = (s[k].detach().cuda().requires_grad_() for k in ("m0", "h", "ms"))
        f = _Film64(case, h, ms)
        m = m0.transpose(1, 2)
        for _ in range(case["steps"]):
            m = f.step(m, case["dt"])
        m = m.transpose(1, 2)
        return [m.detach(), *torch.autograd.grad(m, [m0, h, ms], s["w"].cuda())]
    if kind == "product":
        g = torch.Generator(device="cuda").manual_seed(int(seed))
        m = _unit(torch.randn(case["states"], _cells(case), 3, generator=g, device="cuda")).transpose(1, 2).to(F64)
        if case["form"] not in ("csr", "tiles_fp32", "tiles_bf16x2"):
            return -_Lattice64(case)(m)
        pts, d = (torch.as_tensor(a).cuda() for a in _lattice(case))
        h = torch.zeros_like(m)
        for r in range(0, len(pts), 512):
            o = pts[r:r + 512, None] - pts[None]
            K = torch.stack(_prism(d[0], d[1], d[2], o[..., 0], o[..., 1], o[..., 2]))
            K = torch.where(K.float().abs() > _threshold(case), K, 0.0)
            h[:, :, r:r + 512] = _dense(K, m)
        return -h
    if kind == "assemble":
        if case["out"] == "split":
            return None  # bytes of a storage order: they have to stay as they are
        src, abc, pts = _prisms(case, seed)
        out = torch.empty(6, len(pts), len(src), dtype=F64, device="cuda")
        for r in range(0, len(pts), 256):
            o = pts[r:r + 256, None] - src[None]
            for k, v in enumerate(_prism(abc[:, 0], abc[:, 1], abc[:, 2], o[..., 0], o[..., 1], o[..., 2])):
                out[k, r:r + 256] = v
        return out
    if case["shape"] == "tetra":
        return None  # the face integrals have no restatement here
    a = {k: torch.as_tensor(np.ascontiguousarray(v)).cuda() for k, v in _tile_arrays(case, seed).items()}
    R = _rotations(-a["rot"])
    N = torch.empty(case["tiles"], case["points"], 3, 3, dtype=F64, device="cuda") if kind == "tensor" else None
    H = torch.zeros(case["points"], 3, dtype=F64, device="cuda")
    for r in range(0, case["tiles"], 256):
        q = slice(r, r + 256)
        o = torch.einsum("tab,tpb->tpa", R[q], a["pts"][None] - a["offset"][q, None])
        e = a["size"][q, :, None]
        k = _prism(e[:, 0], e[:, 1], e[:, 2], o[..., 0], o[..., 1], o[..., 2])
        full = torch.stack([torch.stack([k[_AB[i][j]] for j in range(3)], -1) for i in range(3)], -2)
        if N is not None:
            N[q] = full
        else:
            RM = torch.einsum("tab,tb->ta", R[q], a["M"][q])
            H += torch.einsum("tba,tpbc,tc->pa", R[q], full, RM)
    return H if N is None else N


def _rotations(angles):
    """Row-major Rz Ry Rx of the (negated) tile angles: the tile frame's rotation."""
    c, s = torch.cos(angles), torch.sin(angles)
    one, nil = torch.ones_like(c[:, 0]), torch.zeros_like(c[:, 0])

    def mat(*v):
        return torch.stack(v, dim=1).reshape(-1, 3, 3)

    rx = mat(one, nil, nil, nil, c[:, 0], -s[:, 0], nil, s[:, 0], c[:, 0])
    ry = mat(c[:, 1], nil, s[:, 1], nil, one, nil, -s[:, 1], nil, c[:, 1])
    rz = mat(c[:, 2], -s[:, 2], nil, s[:, 2], c[:, 2], nil, nil, nil, one)
    return rz @ ry @ rx
