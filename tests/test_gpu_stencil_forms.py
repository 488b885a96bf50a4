"""The stencil's forms against each other and their partial sums: windows of one
and of two wavefronts per row (widths just below and above where a row needs a
window more), and the form with per-workgroup sums of out * y, for one, two and
four 64-column parts of a row, ragged rows, slabs that do not divide and columns
taller than 64 planes.

Tolerance: each form adds 6R + 3 products per point, so two of them differ by at
most 2 (6R + 6) u times the sum of the terms' absolute values (u = 2^-24 or
2^-53).  The sums add n products in FP64: 2 n 2^-53 of the sum of their absolute
values."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# nx, ny, nz, radius
SHAPES = [(64, 5, 9, 4), (65, 7, 70, 2), (128, 9, 11, 4), (128, 21, 5, 6), (128, 6, 70, 1), (121, 17, 6, 4),
          (120, 17, 6, 4), (117, 9, 8, 6), (116, 9, 8, 6), (127, 11, 7, 1), (126, 10, 7, 2), (123, 8, 9, 3),
          (129, 6, 5, 4), (200, 3, 6, 6), (113, 8, 9, 2), (116, 16, 5, 3), (112, 9, 6, 3)]


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("ragged", [False, True])
@pytest.mark.parametrize("nx,ny,nz,radius", SHAPES)
def test_stencil_forms_and_partial_sums(gpu, nx, ny, nz, radius, ragged, dtype):
    import torch
    from parsec_python_amd import _lib
    from parsec_python_amd.device import ptr, stream
    from parsec_python_amd.grid import DeviceGrid, Grid
    from parsec_python_amd.hamiltonian import leading_dim
    print(f"stencil forms {nx}x{ny}x{nz} r={radius} ragged={ragged} {dtype}", flush=True)
    rng = np.random.default_rng(nx + 3 * ny + 7 * nz + radius)
    mask = np.ones((nz, ny, nx), bool)
    if ragged:   # wide rows with a few short and empty ones
        lo = rng.integers(0, 5, (nz, ny))
        hi = nx - rng.integers(0, 5, (nz, ny))
        short = rng.random((nz, ny)) < 0.2
        hi[short] = lo[short] + rng.integers(0, 6, (nz, ny))[short]
        i = np.arange(nx)
        mask = (i >= lo[..., None]) & (i < hi[..., None])
    g = Grid(nx=nx, ny=ny, nz=nz, h=0.4, rad=0.2 * (nx - 1), mask=mask.reshape(-1), kind="cube")
    dg = DeviceGrid(g, radius)
    n, ld = g.npts, leading_dim(g.npts)
    tdt, u = (torch.float64, 2.0 ** -53) if dtype == "f64" else (torch.float32, 2.0 ** -24)
    a, b, c, scale = 0.7, -0.3, -1.1, 0.5
    V = torch.randn(n, dtype=tdt, device="cuda")
    for nvec in (1, 5):
        Y = torch.full((nvec, ld), float("nan"), dtype=tdt, device="cuda")
        X = torch.full((nvec, ld), float("nan"), dtype=tdt, device="cuda")
        Y[:, :n] = torch.randn((nvec, n), dtype=tdt, device="cuda")
        X[:, :n] = torch.randn((nvec, n), dtype=tdt, device="cuda")
        absY = torch.nan_to_num(Y).abs()

        def run(y, x, out, v, sc, part):
            _lib.call(f"pc_stencil_{dtype}", dg.handle, ptr(y), ptr(x) if x is not None else None, ptr(out), ptr(v),
                      nvec, ld, sc, a, b, c, ptr(part) if part is not None else None, stream())
        # the terms' absolute values, up to the signs that the weights' alternation cancels: sum |w| is below
        # 3 |w_0| + 6 sum |w_d| < 24 for every radius
        mag = 24 * scale * absY.amax() + (abs(a) * V.abs().amax() + abs(b)) * absY.amax() + abs(c) * X[:, :n].abs().amax()
        count, per = C.c_int(), C.c_int()
        _lib.call("pc_stencil_num_partials", dg.handle, tdt.itemsize, nvec, C.byref(count), C.byref(per))
        for x in (None, X):
            plain = torch.full_like(Y, 7.0) if x is None else X.clone()
            dots = torch.full_like(Y, 7.0) if x is None else X.clone()
            part = torch.full((count.value + 8,), 7.0, dtype=torch.float64, device="cuda")
            run(Y, None if x is None else plain, plain, V, scale, None)
            run(Y, None if x is None else dots, dots, V, scale, part)
            assert bool(((plain - dots)[:, :n].abs().double() <= 2 * (6 * radius + 6) * u * mag).all())
            if x is None:
                assert bool((plain[:, n:] == 7.0).all()) and bool((dots[:, n:] == 7.0).all())
            else:
                assert bool(torch.isnan(plain[:, n:]).all()) and bool(torch.isnan(dots[:, n:]).all())
            assert bool((part[count.value:] == 7.0).all())
            terms = dots[:, :n].double() * Y[:, :n].double()
            got = part[:count.value].view(nvec, per.value).sum(1)
            assert bool(((got - terms.sum(1)).abs() <= 2 * n * 2.0 ** -53 * terms.abs().sum(1)).all())
    dg.close()


@pytest.mark.parametrize("dtype,nvec", [("f64", 23), ("f32", 49)])
def test_stencil_time_per_point_of_wide_cubes(gpu, dtype, nvec):
    """Radius 4: 126 columns cost no more per point than 118, which fit two
    windows of 64 (three windows for 126: 18 and 20 % more)."""
    import torch
    from parsec_python_amd import _lib
    from parsec_python_amd.device import ptr, stream
    from parsec_python_amd.grid import DeviceGrid, make_grid
    from parsec_python_amd.hamiltonian import leading_dim
    tdt = torch.float64 if dtype == "f64" else torch.float32
    steps, times = [], [[], []]
    for nx in (118, 126):
        print(f"stencil time {nx}^3 {dtype} nvec={nvec}", flush=True)
        g = make_grid(nx, 0.4, 0.2 * (nx - 1), "cube")
        dg, ld = DeviceGrid(g, 4), leading_dim(g.npts)
        Y, X = (torch.zeros((nvec, ld), dtype=tdt, device="cuda") for _ in range(2))
        V = torch.zeros(g.npts, dtype=tdt, device="cuda")

        def step(dg=dg, ld=ld, Y=Y, X=X, V=V):
            _lib.call(f"pc_stencil_{dtype}", dg.handle, ptr(Y), ptr(X), ptr(X), ptr(V), nvec, ld, 0.5, 1.0, 0.0, 0.5,
                      None, stream())
        steps.append((step, g.npts, dg))
    for _ in range(9):
        for i, (step, npts, _dg) in enumerate(steps):
            e0, e1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            step()
            e0.record()
            for _ in range(4):
                step()
            e1.record()
            torch.cuda.synchronize()
            times[i].append(e0.elapsed_time(e1) / npts)
    narrow, wide = (sorted(t)[4] for t in times)
    print(f"{1e6 * narrow:.3f} and {1e6 * wide:.3f} ns", flush=True)
    assert wide <= 1.1 * narrow
    for _step, _npts, dg in steps:
        dg.close()


def test_stencil_time_per_point_of_full_rows(gpu):
    """Radius 2, 23 vectors, FP32: rows of 120 columns cost no more per point than
    rows of 126 (as two windows of 60 with inner edges 1.2 times)."""
    import torch
    from parsec_python_amd import _lib
    from parsec_python_amd.device import ptr, stream
    from parsec_python_amd.grid import DeviceGrid, make_grid
    from parsec_python_amd.hamiltonian import leading_dim
    steps, times = [], [[], []]
    for nx in (120, 126):
        print(f"stencil time {nx}^3", flush=True)
        g = make_grid(nx, 0.4, 0.2 * (nx - 1), "cube")
        dg, ld = DeviceGrid(g, 2), leading_dim(g.npts)
        Y, X = (torch.zeros((23, ld), device="cuda") for _ in range(2))
        V = torch.zeros(g.npts, device="cuda")

        def step(dg=dg, ld=ld, Y=Y, X=X, V=V):
            _lib.call("pc_stencil_f32", dg.handle, ptr(Y), ptr(X), ptr(X), ptr(V), 23, ld, 0.5, 1.0, 0.0, 0.5, None, stream())
        steps.append((step, g.npts, dg))
    for _ in range(9):
        for i, (step, npts, _dg) in enumerate(steps):
            e0, e1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            step()
            e0.record()
            for _ in range(4):
                step()
            e1.record()
            torch.cuda.synchronize()
            times[i].append(e0.elapsed_time(e1) / npts)
    full, wide = (sorted(t)[4] for t in times)
    print(f"{1e6 * full:.3f} and {1e6 * wide:.3f} ns", flush=True)
    assert full <= 1.1 * wide
    for _step, _npts, dg in steps:
        dg.close()
