"""
Performance cases: what a program that uses this framework has it do.

Every case is a dict with a ``kind`` and sizes.  The kinds, and what each one
is in real use:

``regrid``
    the drop-in one-call regrid of host arrays (conservative, 2-D grids).
``from_weights``
    the drop-in apply of host values to weights made once: new images of one
    pair of grids, frame after frame.
``build``
    device-resident grids whose relation changes each time: weights built,
    then applied to a stack of FP64 images.
``batch``
    many independent, uneven pairs of grids built and applied together.
``apply``
    kept weights applied to device-resident images, forward or adjoint.
``train``
    a differentiable step through kept weights: forward, then the gradient.
``views``
    an inversion step: one unknown image against several observation grids,
    forward and gradient.
``find``
    point location: the vertices of one grid in the cells of another.
``fill``
    missing pixels of an image stack relaxed from their neighbours.
``line``
    1-D conservative weights of many spectra, each with its own wavelength
    solution and weighting, onto a common axis.

Vertex counts are along (x, y); a grid of n vertices has n - 1 cells along an
axis.  Grids are smooth warps of rotated rectangles, images Poisson counts.
"""

from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import regridding_amd as rg
from regridding_amd._conservative import PackedPairs, build_2d_batched, build_2d_device
from regridding_amd._lib import DeviceArray, check, lib, rg_apply_job
from regridding_amd.torch_ops import regrid_apply, regrid_apply_views

DEVICE = "cuda"

# ---- the cases -------------------------------------------------------------


def listed() -> list[dict]:
    return [
        # one small call from start to end: the host path and launch latency
        dict(name="regrid_small", kind="regrid", nxi=129, nyi=129, nxo=101, nyo=101, images=4),
        # a detector's frames through weights made once, values on the host
        dict(name="from_weights_frames", kind="from_weights", nxi=513, nyi=513, nxo=385,
             nyo=385, images=8),
        # a small, uneven pair on the device: launches and host waits count
        dict(name="build_small", kind="build", nxi=67, nyi=190, nxo=81, nyo=125, images=1),
        # the headline configuration: a full detector, 16 images
        dict(name="build_large", kind="build", nxi=2049, nyi=2049, nxo=1537, nyo=1537,
             images=16),
        # a mixed batch: sizes over two orders of magnitude, 1-8 images each
        dict(name="batch_mixed", kind="batch", pairs=64, n_min=33, n_max=1025),
        # one image through small weights: the smallest device call
        dict(name="apply_f64_small", kind="apply", nxi=129, nyi=129, nxo=101, nyo=101,
             images=1, dtype="float64", transpose=False),
        # a stack of full detector images
        dict(name="apply_f64_large", kind="apply", nxi=2049, nyi=2049, nxo=1537, nyo=1537,
             images=16, dtype="float64", transpose=False),
        # a learning step in single precision, odd sizes, a ragged batch
        dict(name="train_f32_ragged", kind="train", nxi=1202, nyi=1501, nxo=1000, nyo=1334,
             images=5, dtype="float32"),
        # eight views of one image: one step of an iterative inversion
        dict(name="views_f64", kind="views", nxi=1025, nyi=1025, nxo=769, nyo=769, views=8,
             dtype="float64"),
        # every vertex of a large grid located in a warped one
        dict(name="find_cells", kind="find", nxi=1025, nyi=1025, nxo=1537, nyo=1537),
        # bad pixels and dropped blocks of an image stack, odd width
        dict(name="fill_stack", kind="fill", images=4, ny=768, nx=1001, iterations=100),
        # a spectrograph's rows onto a common wavelength axis
        dict(name="line_spectra", kind="line", rows=2048, n=2049, m=1537, reverse=False),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _pair_sizes(rng, lo: int, hi: int) -> dict:
    """An uneven pair: axes within a factor of two of each other, output to
    input spacing between a half and two."""
    nx = _log_int(rng, lo, hi)
    ny = min(hi, max(lo, int(round(nx * rng.uniform(0.6, 1.6)))))
    r = rng.uniform(0.5, 2.0)
    return dict(nxi=nx, nyi=ny, nxo=min(hi, max(9, int(nx / r))),
                nyo=min(hi, max(9, int(ny / r))))


def draw(rng) -> dict:
    """One more case of the ranges the listed ones stand for."""
    kind = rng.choice(["regrid", "from_weights", "build", "build", "batch", "apply", "apply",
                       "train", "views", "find", "fill", "fill", "line"])
    if kind == "regrid":
        return dict(kind=kind, **_pair_sizes(rng, 17, 400), images=rng.randint(1, 8))
    if kind == "from_weights":
        return dict(kind=kind, **_pair_sizes(rng, 65, 800), images=rng.randint(1, 8))
    if kind == "build":
        return dict(kind=kind, **_pair_sizes(rng, 17, 1537), images=rng.randint(1, 16))
    if kind == "batch":
        return dict(kind=kind, pairs=_log_int(rng, 2, 48), n_min=33,
                    n_max=_log_int(rng, 129, 900))
    if kind == "apply":
        return dict(kind=kind, **_pair_sizes(rng, 33, 1537), images=rng.randint(1, 16),
                    dtype=rng.choice(["float64", "float32"]),
                    transpose=rng.random() < 0.5)
    if kind == "train":
        return dict(kind=kind, **_pair_sizes(rng, 33, 1537), images=rng.randint(1, 12),
                    dtype=rng.choice(["float64", "float32"]))
    if kind == "views":
        return dict(kind=kind, **_pair_sizes(rng, 65, 1025), views=rng.randint(2, 8),
                    dtype=rng.choice(["float64", "float32"]))
    if kind == "find":
        return dict(kind=kind, **_pair_sizes(rng, 33, 1537))
    if kind == "fill":
        return dict(kind=kind, images=rng.randint(1, 8), ny=_log_int(rng, 24, 1100),
                    nx=_log_int(rng, 24, 1100), iterations=rng.choice([50, 100, 100, 200]))
    n = _log_int(rng, 65, 2500)
    return dict(kind="line", rows=_log_int(rng, 16, 2048), n=n,
                m=max(33, int(n * rng.uniform(0.5, 1.5))), reverse=rng.random() < 0.25)


# ---- inputs ----------------------------------------------------------------


def _grid(nx: int, ny: int, theta: float, ax: float, ay: float, lo: float, hi: float):
    """A rotated rectangle of vertices with a smooth warp."""
    X, Y = np.meshgrid(np.linspace(lo, hi, nx), np.linspace(lo, hi, ny), indexing="ij")
    c, s = math.cos(theta), math.sin(theta)
    xr, yr = X * c - Y * s, X * s + Y * c
    return xr + ax * np.sin(3 * yr), yr + ay * np.cos(2 * xr)


OUT_LO, OUT_HI = -0.9, 0.9


def _pair(case: dict, rng):
    """Warped input grid, rotated output grid, and the output's rotation."""
    ax, ay = rng.uniform(0.01, 0.08, 2)
    t_in, t_out = rng.uniform(0, math.pi / 4, 2)
    gi = _grid(case["nxi"], case["nyi"], t_in, ax, ay, -1.0, 1.0)
    go = _grid(case["nxo"], case["nyo"], t_out, 0.0, 0.0, OUT_LO, OUT_HI)
    return gi, go, t_out


def _cells(nx: int, ny: int) -> int:
    return (nx - 1) * (ny - 1)


def _images(rng, batch: int, cells: int, dtype=torch.float64) -> torch.Tensor:
    """Poisson counts on the device, one lognormal rate per image."""
    gen = torch.Generator(device=DEVICE).manual_seed(int(rng.integers(1 << 60)))
    rate = torch.as_tensor(rng.lognormal(3, 1, batch), dtype=torch.float32, device=DEVICE)
    counts = torch.poisson(rate[:, None].expand(batch, cells).contiguous(), generator=gen)
    return counts.to(dtype)


def _device_grid(g):
    return [DeviceArray.from_host(a) for a in g]


def _build(gi, go):
    (xi, yi), (xo, yo) = _device_grid(gi), _device_grid(go)
    return build_2d_device(xi, yi, gi[0].shape, xo, yo, go[0].shape)


def _batch_pairs(case: dict, rng):
    """Uneven pairs: per-axis vertex counts log-uniform in [n_min, n_max]
    (the sizes are the case's, the grids and values the seed's)."""
    sizes = np.random.default_rng(3)
    pairs = []
    for _ in range(case["pairs"]):
        nx, ny = np.round(np.exp(sizes.uniform(math.log(case["n_min"]), math.log(case["n_max"]),
                                               2))).astype(int)
        r = sizes.uniform(0.5, 2.0)
        c = dict(nxi=int(nx), nyi=int(ny), nxo=max(2, int(round((nx - 1) / r)) + 1),
                 nyo=max(2, int(round((ny - 1) / r)) + 1))
        pairs.append((c, *_pair(c, rng), int(sizes.integers(1, 9))))
    return pairs


def _batch_values(pairs, rng):
    return [_images(rng, b, _cells(c["nxi"], c["nyi"])) for c, _, _, _, b in pairs]


def _views(case: dict, rng):
    truth = _grid(case["nxi"], case["nyi"], 0.0, 0.0, 0.0, -1.0, 1.0)
    obs, thetas = [], []
    for _ in range(case["views"]):
        t = rng.uniform(0.02, math.pi / 4)
        thetas.append(t)
        obs.append(_grid(case["nxo"], case["nyo"], t, 0.0, 0.0, OUT_LO, OUT_HI))
    return truth, obs, thetas


def _mask(rng, T: int, ny: int, nx: int) -> np.ndarray:
    """Scattered bad pixels (2 %) and a few dropped blocks per image."""
    where = rng.random((T, ny, nx)) < 0.02
    for t in range(T):
        for _ in range(6):
            h = int(rng.integers(1, max(2, ny // 8)))
            w = int(rng.integers(1, max(2, nx // 8)))
            j, i = int(rng.integers(0, ny)), int(rng.integers(0, nx))
            where[t, j:j + h, i:i + w] = True
    return where


def _fill_inputs(case: dict, rng):
    T, ny, nx = case["images"], case["ny"], case["nx"]
    where = _mask(rng, T, ny, nx)
    y, x = np.mgrid[0:ny, 0:nx]
    base = 100 + 50 * np.sin(6.0 * x / nx) * np.cos(4.0 * y / ny)
    a = rng.poisson(np.broadcast_to(base, (T, ny, nx))).astype(np.float64)
    for t in range(T):
        good = a[t][~where[t]]
        a[t][where[t]] = np.median(good) if good.size else 0.0
    return a, where


def _spectra(case: dict, rng):
    """Per-row wavelength solutions (offset, dispersion, curvature), a common
    output axis inside their mean range and a cell weighting.  The solutions
    are the instrument's (the sizes alone set them, and with them the number
    of weights); which row has which, and the weighting, are the seed's."""
    D, n, m = case["rows"], case["n"], case["m"]
    made = np.random.default_rng(7)
    u = np.linspace(0, 1, n)
    off = made.uniform(-0.02, 0.02, (D, 1))
    disp = made.uniform(0.95, 1.05, (D, 1))
    curve = made.uniform(-0.05, 0.05, (D, 1))
    x = (500 + 100 * (off + disp * u + curve * u * (1 - u)))[rng.permutation(D)]
    axis = np.linspace(500 + made.uniform(1, 4), 600 - made.uniform(1, 4), m)
    if case["reverse"]:  # a frequency axis: descending
        axis = axis[::-1]
    return x, np.ascontiguousarray(np.broadcast_to(axis, (D, m))), rng.uniform(0.8, 1.2,
                                                                               (D, n - 1))


def prepare(case: dict, seed: int) -> dict:
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    s = dict(case=case)
    if kind in ("regrid", "from_weights"):
        gi, go, _ = _pair(case, rng)
        shape = (case["images"], case["nxi"] - 1, case["nyi"] - 1)
        rate = rng.lognormal(3, 1, case["images"])
        s["values"] = rng.poisson(rate[:, None, None], shape).astype(np.float64)
        if kind == "regrid":
            s.update(gi=gi, go=go)
        else:
            s["weights"] = rg.weights(gi, go, method="conservative")
    elif kind == "build":
        gi, go, _ = _pair(case, rng)
        s.update(gi=_device_grid(gi), go=_device_grid(go), si=gi[0].shape, so=go[0].shape,
                 x=_images(rng, case["images"], _cells(case["nxi"], case["nyi"])))
    elif kind == "batch":
        pairs = _batch_pairs(case, rng)
        s["packed"] = PackedPairs([(gi, go) for _, gi, go, _, _ in pairs])
        s["x"] = _batch_values(pairs, rng)
        s["n_out"] = [_cells(c["nxo"], c["nyo"]) for c, *_ in pairs]
    elif kind in ("apply", "train"):
        gi, go, _ = _pair(case, rng)
        dtype = getattr(torch, case["dtype"])
        n_in, n_out = _cells(case["nxi"], case["nyi"]), _cells(case["nxo"], case["nyo"])
        s["w"] = _build(gi, go)
        if kind == "apply":
            s["x"] = _images(rng, case["images"], n_out if case["transpose"] else n_in, dtype)
        else:
            s["x"] = _images(rng, case["images"], n_in, dtype).requires_grad_()
            s["g"] = _images(rng, case["images"], n_out, dtype)
    elif kind == "views":
        truth, obs, _ = _views(case, rng)
        dtype = getattr(torch, case["dtype"])
        s["w"] = tuple(build_2d_batched([(truth, o) for o in obs]))
        s["x"] = _images(rng, 1, _cells(case["nxi"], case["nyi"]), dtype)[0].requires_grad_()
        s["g"] = _images(rng, 1, case["views"] * _cells(case["nxo"], case["nyo"]), dtype)[0]
    elif kind == "find":
        gi, go, _ = _pair(case, rng)
        s["grid"] = [torch.as_tensor(a, device=DEVICE) for a in gi]
        s["points"] = [torch.as_tensor(a.ravel(), device=DEVICE) for a in go]
    elif kind == "fill":
        a, where = _fill_inputs(case, rng)
        s["a"] = torch.as_tensor(a, device=DEVICE)
        s["where"] = torch.as_tensor(where.astype(np.uint8), device=DEVICE)
    elif kind == "line":
        s["x"], s["axis"], s["wi"] = (torch.as_tensor(a, device=DEVICE)
                                      for a in _spectra(case, rng))
    else:
        raise ValueError(kind)
    return s


# ---- one pass --------------------------------------------------------------


def _stream() -> int:
    return torch.cuda.current_stream().cuda_stream


def run(s: dict):
    case = s["case"]
    kind = case["kind"]
    if kind == "regrid":
        return rg.regrid(s["gi"], s["go"], s["values"], axis_input=(-2, -1),
                         axis_output=(-2, -1), method="conservative")
    if kind == "from_weights":
        w, shape_in, shape_out = s["weights"]
        return rg.regrid_from_weights(w, shape_in, shape_out, s["values"],
                                      axis_input=(-2, -1), axis_output=(-2, -1))
    if kind == "build":
        w = build_2d_device(*s["gi"], s["si"], *s["go"], s["so"], stream=_stream())
        return regrid_apply(w, s["x"])
    if kind == "batch":
        handles = build_2d_batched(s["packed"], stream=_stream())
        y = torch.empty(sum(x.shape[0] * n for x, n in zip(s["x"], s["n_out"])),
                        dtype=torch.float64, device=DEVICE)
        jobs = (rg_apply_job * len(handles))()
        at = 0
        for job, h, x, n in zip(jobs, handles, s["x"], s["n_out"]):
            job.weights, job.transpose, job.batch = h.ptr, 0, x.shape[0]
            job.values_input, job.values_output = x.data_ptr(), y.data_ptr() + 8 * at
            at += x.shape[0] * n
        check(lib().rg_apply_batched_f64(jobs, len(handles), _stream()))
        return y
    if kind == "apply":
        return regrid_apply(s["w"], s["x"], transpose=case["transpose"])
    if kind in ("train", "views"):
        f = regrid_apply if kind == "train" else regrid_apply_views
        y = f(s["w"], s["x"])
        (grad,) = torch.autograd.grad(y, s["x"], s["g"])
        return y.detach(), grad
    if kind == "find":
        (x, y), (px, py) = s["grid"], s["points"]
        ij = torch.empty((px.numel(), 2), dtype=torch.int64, device=DEVICE)
        check(lib().rg_find_cells_2d(x.data_ptr(), y.data_ptr(), x.shape[0], x.shape[1],
                                     px.data_ptr(), py.data_ptr(), px.numel(), ij.data_ptr(),
                                     _stream()))
        return ij
    if kind == "fill":
        a = s["a"].clone()
        T, ny, nx = a.shape
        check(lib().rg_fill_gauss_seidel_2d(a.data_ptr(), s["where"].data_ptr(), T, ny, nx,
                                            case["iterations"], _stream()))
        return a
    if kind == "line":
        x, axis, wi = s["x"], s["axis"], s["wi"]
        (D, n), m = x.shape, axis.shape[1]
        counts = torch.empty(D * (n - 1), dtype=torch.int32, device=DEVICE)
        offsets = torch.empty(D * (n - 1) + 1, dtype=torch.int64, device=DEVICE)
        total = ctypes.c_int64()
        check(lib().rg_conservative_1d_count(x.data_ptr(), n, axis.data_ptr(), m, D,
                                             counts.data_ptr(), offsets.data_ptr(),
                                             ctypes.byref(total), _stream()))
        i = torch.empty(total.value, dtype=torch.int64, device=DEVICE)
        j = torch.empty_like(i)
        w = torch.empty(total.value, dtype=torch.float64, device=DEVICE)
        check(lib().rg_conservative_1d_emit(x.data_ptr(), n, axis.data_ptr(), m, D,
                                            wi.data_ptr(), counts.data_ptr(),
                                            offsets.data_ptr(), i.data_ptr(), j.data_ptr(),
                                            w.data_ptr(), _stream()))
        return i, j, w
    raise ValueError(kind)


# ---- the work a pass cannot do without ---------------------------------------


def _pair_nnz(c: dict, cells_in=None) -> float:
    """Overlapping pairs of two grids over the output's area: the faces of
    two crossed lattices at an angle of about pi / 12."""
    n_out = _cells(c["nxo"], c["nyo"])
    n_in = 0.81 * _cells(c["nxi"], c["nyi"])
    turn = math.sin(math.pi / 12) + math.cos(math.pi / 12)
    return n_in + n_out + 2 * turn * math.sqrt(n_in * n_out)


def _apply_work(c: dict, batch: int, size: int) -> tuple[float, float]:
    n_in, n_out, nnz = _cells(c["nxi"], c["nyi"]), _cells(c["nxo"], c["nyo"]), _pair_nnz(c)
    return batch * (n_in + n_out) * size + nnz * (4 + size) + 4 * n_out, 2 * nnz * batch


def _build_work(c: dict) -> tuple[float, float]:
    """Both grids read once, the weights (column, value, row starts) written
    once; about 64 operations a crossing segment, two segments a pair."""
    nnz = _pair_nnz(c)
    grids = 16 * (c["nxi"] * c["nyi"] + c["nxo"] * c["nyo"])
    return grids + 12 * nnz + 4 * _cells(c["nxi"], c["nyi"]), 128 * nnz


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind in ("regrid", "build"):
        parts = [_build_work(case), _apply_work(case, case["images"], 8)]
    elif kind == "from_weights":
        parts = [_apply_work(case, case["images"], 8)]
    elif kind == "batch":
        # the mean pair of the declared distribution
        a, b = math.log(case["n_min"]), math.log(case["n_max"])
        mean = (math.exp(b) - math.exp(a)) / (b - a)
        n = int(mean)
        c = dict(nxi=n, nyi=n, nxo=n, nyo=n)
        parts = [tuple(case["pairs"] * v for v in w)
                 for w in (_build_work(c), _apply_work(c, 4.5, 8))]
    elif kind == "apply":
        parts = [_apply_work(case, case["images"], 8 if case["dtype"] == "float64" else 4)]
    elif kind == "train":
        parts = 2 * [_apply_work(case, case["images"], 8 if case["dtype"] == "float64" else 4)]
    elif kind == "views":
        size = 8 if case["dtype"] == "float64" else 4
        n_in = _cells(case["nxi"], case["nyi"])
        # x is read once and the gradient written once for all views
        parts = 2 * case["views"] * [_apply_work(case, 1, size)]
        parts.append((-2.0 * (case["views"] - 1) * n_in * size, 0.0))
    elif kind == "find":
        n = case["nxo"] * case["nyo"]
        parts = [(16 * case["nxi"] * case["nyi"] + 32 * n, 200 * n)]
    elif kind == "fill":
        cells = case["images"] * case["ny"] * case["nx"]
        parts = [(17 * cells, 0.05 * cells * 6 * case["iterations"])]
    else:
        D, n, m = case["rows"], case["n"], case["m"]
        nnz = D * (n + m)
        parts = [(8 * D * (2 * n + m) + 24 * nnz + 12 * D * n, 4 * nnz)]
    return dict(bytes=float(sum(p[0] for p in parts)), flops=float(sum(p[1] for p in parts)))


# ---- plain 64-bit results ------------------------------------------------------


def _overlaps(gi, go, theta: float):
    """(input cell, output cell, overlap / input area) of a grid of
    quadrilaterals against a rotated regular grid, in plain torch: in the
    output's index space its cells are unit squares, and a polygon's area
    inside a square is the sum over its edges of the integral of the edge's
    height, clamped to the square, over the edge's clamped x range."""
    nxo, nyo = go[0].shape
    c, s = math.cos(theta), math.sin(theta)
    x = torch.as_tensor(gi[0], device=DEVICE)
    y = torch.as_tensor(gi[1], device=DEVICE)
    u = ((x * c + y * s) - OUT_LO) / (OUT_HI - OUT_LO) * (nxo - 1)
    v = ((-x * s + y * c) - OUT_LO) / (OUT_HI - OUT_LO) * (nyo - 1)
    corners = lambda a: torch.stack(  # noqa: E731
        [a[:-1, :-1], a[1:, :-1], a[1:, 1:], a[:-1, 1:]], -1).reshape(-1, 4)
    U, V = corners(u), corners(v)
    lo_u, lo_v = U.min(1).values.floor(), V.min(1).values.floor()
    ku = int((U.max(1).values.ceil() - lo_u).max())
    kv = int((V.max(1).values.ceil() - lo_v).max())
    U1, V1 = U.roll(-1, 1), V.roll(-1, 1)
    area = 0.5 * (U * V1 - U1 * V).sum(1)
    found = []
    step = max(1, 4_000_000 // (ku * kv))
    for at in range(0, U.shape[0], step):
        sl = slice(at, at + step)
        a = lo_u[sl, None, None, None] + torch.arange(ku, device=DEVICE)[None, :, None, None]
        b = lo_v[sl, None, None, None] + torch.arange(kv, device=DEVICE)[None, None, :, None]
        p, q = U[sl, None, None, :] - a, U1[sl, None, None, :] - a
        h0, h1 = V[sl, None, None, :] - b, V1[sl, None, None, :] - b
        d = q - p
        flat = d == 0
        d1 = torch.where(flat, torch.ones_like(d), d)
        t0 = ((p.clamp(0, 1) - p) / d1).clamp(0, 1)
        t1 = ((q.clamp(0, 1) - p) / d1).clamp(0, 1)
        dh = h1 - h0
        dh1 = torch.where(dh == 0, torch.ones_like(dh), dh)
        cut = torch.stack([(0 - h0) / dh1, (1 - h0) / dh1])  # where it crosses the square's sides
        ta, tb = torch.minimum(t0, t1), torch.maximum(t0, t1)
        e1 = torch.minimum(torch.maximum(cut.min(0).values, ta), tb)
        e2 = torch.minimum(torch.maximum(cut.max(0).values, ta), tb)
        total = torch.zeros_like(d)
        for f, t in ((ta, e1), (e1, e2), (e2, tb)):
            mid = (h0 + dh * (0.5 * (f + t))).clamp(0, 1)
            total = total + mid * (t - f)
        total = torch.where(flat, torch.zeros_like(d), total * d)
        part = -total.sum(-1) / area[sl, None, None]
        a, b = a[..., 0].expand_as(part), b[..., 0].expand_as(part)
        keep = (part > 1e-15) & (a >= 0) & (a < nxo - 1) & (b >= 0) & (b < nyo - 1)
        cell = torch.arange(at, at + part.shape[0], device=DEVICE)[:, None, None]
        found.append((cell.expand_as(part)[keep], (a * (nyo - 1) + b)[keep].long(), part[keep]))
    return [torch.cat(z) for z in zip(*found)]


def _plain_apply(src, dst, w, x: torch.Tensor, n: int) -> torch.Tensor:
    x = x.detach().double().reshape(-1, x.shape[-1])
    y = torch.zeros((x.shape[0], n), dtype=torch.float64, device=x.device)
    for k in range(x.shape[0]):
        y[k].index_add_(0, dst, w * x[k, src])
    return y


def _plain_fill(a, where, iterations: int):
    """Red-black Gauss-Seidel with periodic neighbours, cells updated row by
    row within a colour: of two same-colour neighbours across an odd edge the
    one in the last column or row comes second, the corner last of all."""
    T, ny, nx = a.shape
    j, i = torch.meshgrid(torch.arange(ny, device=a.device), torch.arange(nx, device=a.device),
                          indexing="ij")
    late = ((i == nx - 1) & (nx % 2 == 1)).long() + ((j == ny - 1) & (ny % 2 == 1)).long()
    cx, cy = ((nx - 1) / 2) ** 2, ((ny - 1) / 2) ** 2
    for _ in range(iterations):
        for colour in (0, 1):
            for rank in range(1 + nx % 2 + ny % 2):
                now = where & ((i + j) % 2 == colour) & (late == rank)
                new = (cx * (a.roll(1, 2) + a.roll(-1, 2)) + cy * (a.roll(1, 1) + a.roll(-1, 1)))
                a = torch.where(now, new / (2 * (cx + cy)), a)
    return a


def exact(case: dict, seed: int):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind in ("regrid", "from_weights"):
        s = prepare(dict(case, kind="regrid"), seed)
        gi, go, theta = _pair(case, rng)
        i, o, w = _overlaps(gi, go, theta)
        x = torch.as_tensor(s["values"], device=DEVICE).reshape(case["images"], -1)
        y = _plain_apply(i, o, w, x, _cells(case["nxo"], case["nyo"]))
        return y.reshape(case["images"], case["nxo"] - 1, case["nyo"] - 1).cpu().numpy()
    if kind in ("build", "apply", "train"):
        gi, go, theta = _pair(case, rng)
        i, o, w = _overlaps(gi, go, theta)
        n_in, n_out = _cells(case["nxi"], case["nyi"]), _cells(case["nxo"], case["nyo"])
        dtype = getattr(torch, case.get("dtype", "float64"))
        if case.get("transpose"):
            return _plain_apply(o, i, w, _images(rng, case["images"], n_out, dtype), n_in)
        y = _plain_apply(i, o, w, _images(rng, case["images"], n_in, dtype), n_out)
        if kind != "train":
            return y
        return y, _plain_apply(o, i, w, _images(rng, case["images"], n_out, dtype), n_in)
    if kind == "batch":
        pairs = _batch_pairs(case, rng)
        out = []
        for (c, gi, go, theta, _), x in zip(pairs, _batch_values(pairs, rng)):
            out.append(_plain_apply(*_overlaps(gi, go, theta), x,
                                    _cells(c["nxo"], c["nyo"])).reshape(-1))
        return torch.cat(out)
    if kind == "views":
        truth, obs, thetas = _views(case, rng)
        n_in, n_out = _cells(case["nxi"], case["nyi"]), _cells(case["nxo"], case["nyo"])
        dtype = getattr(torch, case["dtype"])
        x = _images(rng, 1, n_in, dtype)
        g = _images(rng, 1, case["views"] * n_out, dtype)[0].reshape(-1, n_out)
        y, grad = [], torch.zeros(n_in, dtype=torch.float64, device=DEVICE)
        for k, (go, theta) in enumerate(zip(obs, thetas)):
            i, o, w = _overlaps(truth, go, theta)
            y.append(_plain_apply(i, o, w, x, n_out)[0])
            grad += _plain_apply(o, i, w, g[k:k + 1], n_in)[0]
        return torch.cat(y), grad
    if kind == "fill":
        a, where = _fill_inputs(case, rng)
        return _plain_fill(torch.as_tensor(a, device=DEVICE),
                           torch.as_tensor(where, device=DEVICE), case["iterations"])
    if kind == "line" and not case["reverse"]:
        x, axis, wi = (torch.as_tensor(a, device=DEVICE) for a in _spectra(case, rng))
        cuts = torch.cat([x, axis], 1).sort(1).values
        mid, length = 0.5 * (cuts[:, 1:] + cuts[:, :-1]), cuts[:, 1:] - cuts[:, :-1]
        i = torch.searchsorted(x, mid) - 1
        j = torch.searchsorted(axis, mid) - 1
        keep = ((i >= 0) & (i < x.shape[1] - 1) & (j >= 0) & (j < axis.shape[1] - 1)
                & (length > 0))
        cell = x[:, 1:] - x[:, :-1]
        at = i.clamp(0, cell.shape[1] - 1)
        w = length / cell.gather(1, at) * wi.gather(1, at)
        return i[keep], j[keep], w[keep]
    return None  # cell indices; descending axes
