"""Edges of the windowed stencil: slabs whose columns just fit one, two or three
windows of 64 lanes and one more, rows that begin and end anywhere (also empty
ones), slabs and z-chunks that do not divide the grid, columns taller than the
row table's 64 planes, 8 vectors and enough of them to go without z-chunks.

Tolerance, per point: a sum of 6R + 3 products, each rounded with its addition,
errs by at most (6R + 6) u times the sum of the terms' absolute values; the
oracle's FP64 sum adds the same with its own u."""
import numpy as np
import pytest

from oracle import fd as ofd

pytestmark = pytest.mark.gpu

# nx, ny, nz, radius: 64, 128 - 2R and 192 - 4R columns fill one, two and three windows
SHAPES = [(64, 9, 13, 4), (65, 17, 7, 6), (116, 13, 9, 6), (117, 8, 21, 6), (120, 7, 11, 4), (121, 9, 6, 4),
          (176, 5, 9, 4), (177, 16, 5, 4), (256, 4, 5, 6), (126, 3, 4, 1), (127, 3, 5, 1), (180, 9, 5, 3),
          (33, 24, 150, 2), (7, 8, 9, 1), (1, 3, 70, 3), (20, 25, 66, 6)]


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("ragged", [False, True])
@pytest.mark.parametrize("nx,ny,nz,radius", SHAPES)
def test_stencil_edges(gpu, nx, ny, nz, radius, ragged, dtype):
    import torch
    from parsec_python_amd.grid import Grid
    from parsec_python_amd.hamiltonian import Hamiltonian, leading_dim
    print(f"stencil edge case {nx}x{ny}x{nz} r={radius} ragged={ragged} {dtype}", flush=True)
    h, a, b, c = 0.4, 0.7, -0.3, -1.1
    rng = np.random.default_rng(nx + 3 * ny + 7 * nz + radius)
    mask = np.ones((nz, ny, nx), bool)
    if ragged:
        lo = rng.integers(0, nx, (nz, ny))
        hi = lo + rng.integers(0, nx + 1, (nz, ny))
        i = np.arange(nx)
        mask = (i >= lo[..., None]) & (i < hi[..., None])
    g = Grid(nx=nx, ny=ny, nz=nz, h=h, rad=0.5 * h * (nx - 1), mask=mask.reshape(-1), kind="cube")
    n = g.npts
    tdt, u = (torch.float64, 2.0 ** -53) if dtype == "f64" else (torch.float32, 2.0 ** -24)
    A = (ofd.laplacian_masked(nx, ny, nz, radius, g.mask) * (0.5 / h ** 2)).tocsr()
    pot = rng.standard_normal(n)
    H = Hamiltonian(g, radius, None, torch.tensor(pot, device="cuda"), tdt)
    ld = leading_dim(n)
    for nvec in (8, 37):
        Y = torch.full((nvec, ld), float("nan"), dtype=tdt, device="cuda")   # the padding must not be read
        X = torch.full((nvec, ld), float("nan"), dtype=tdt, device="cuda")
        Y[:, :n] = torch.tensor(rng.standard_normal((nvec, n)), dtype=tdt)
        X[:, :n] = torch.tensor(rng.standard_normal((nvec, n)), dtype=tdt)
        y, x = Y[:, :n].double().cpu().numpy().T, X[:, :n].double().cpu().numpy().T
        ref0 = a * (A @ y + pot[:, None] * y) + b * y
        mag0 = abs(a) * (abs(A) @ abs(y) + abs(pot[:, None] * y)) + abs(b * y)
        O = torch.full_like(X, float("nan"))
        H.step(Y, None, O, nvec, a, b, 0.0)
        H.step(Y, X, X, nvec, a, b, c)              # in place
        for out, ref, mag in ((O, ref0, mag0), (X, ref0 + c * x, mag0 + abs(c * x))):
            got = out[:, :n].double().cpu().numpy().T
            assert np.all(np.abs(got - ref) <= (6 * radius + 6) * (u + 2.0 ** -53) * mag)
            assert torch.isnan(out[:, n:]).all()    # nor written
    H.close()
