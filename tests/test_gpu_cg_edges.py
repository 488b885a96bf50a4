"""Edges of the Hartree passes: rows of one and two x-chunks and wider, slabs and
z-chunks that do not divide the grid, columns so tall that a chunk holds more
than 6 planes, and multigrid hierarchies of 1, 2 and more levels in LDS.

Plain CG: 6 iterations against the oracle's loop; every operation differs by
rounding only, and 6 steps of a well-scaled residual amplify it by less than
1e4: 1e-11 of the largest value.  Multigrid: the residual against the oracle's
operator meets the tolerance asked for (5 % for the rounding of the recurrence)."""
import numpy as np
import pytest

from oracle import fd as ofd
from oracle.pcg import pcg as opcg
from tests.test_gpu_kernels import _grid

pytestmark = pytest.mark.gpu

SHAPES = [(5, 4, 3, "cube", 1), (64, 9, 13, "cube", 4), (65, 17, 7, "cube", 6), (128, 10, 9, "cube", 3),
          (129, 11, 8, "cube", 4), (16, 16, 16, "cube", 4), (30, 30, 30, "sphere", 4), (33, 31, 29, "cube", 2),
          (75, 75, 75, "sphere", 4), (4, 120, 420, "cube", 2), (68, 120, 424, "cube", 1)]


@pytest.mark.parametrize("nx,ny,nz,kind,radius", SHAPES)
def test_cg_edges(gpu, nx, ny, nz, kind, radius):
    import torch
    from parsec_python_amd.grid import DeviceGrid
    from parsec_python_amd.hartree import HartreeSolver
    print(f"cg edge case {nx}x{ny}x{nz} {kind} r={radius}", flush=True)
    h = 0.35
    g = _grid(nx, ny, nz, h, kind)
    A = ((1.0 / h ** 2) * ofd.laplacian_masked(g.nx, g.ny, g.nz, radius, g.mask)).tocsr()
    rng = np.random.default_rng(nx + 3 * ny + 7 * nz)
    rhs = rng.standard_normal(g.npts)
    b = torch.tensor(rhs, device="cuda")
    dg = DeviceGrid(g, radius)
    for alias in (True, False):
        xr, _ = opcg(A, rhs, np.zeros(g.npts), 6, 0.0, reference_aliasing=alias)
        hs = HartreeSolver(dg, h, reference_aliasing=alias)
        x = torch.zeros_like(b)
        assert hs.solve(b, x, 6, 0.0) == 6
        assert np.max(np.abs(x.cpu().numpy() - xr)) <= 1e-11 * np.abs(xr).max()
    hm = HartreeSolver(dg, h, prec="mg")
    for tol in (1e-5, 1e-9):
        x = torch.zeros_like(b)
        its = hm.solve(b, x, 300, tol)
        assert its < 300
        assert np.linalg.norm(rhs - A @ x.cpu().numpy()) <= 1.05 * tol * np.linalg.norm(rhs)
    hm.close()
    dg.close()


@pytest.mark.parametrize("nx,ny,nz,radius", [(70, 12, 9, 4), (64, 7, 130, 6), (130, 9, 7, 3), (1, 5, 5, 2)])
def test_single_vector_step_edges(gpu, nx, ny, nz, radius):
    """One FP64 vector (the Lanczos H v) in place: 1e-13 of the operands' scale."""
    import torch
    from parsec_python_amd.hamiltonian import Hamiltonian, leading_dim
    print(f"single edge case {nx}x{ny}x{nz} r={radius}", flush=True)
    h = 0.4
    g = _grid(nx, ny, nz, h, "cube")
    rng = np.random.default_rng(nx + ny)
    V, y, x = (rng.standard_normal(g.npts) for _ in range(3))
    H = Hamiltonian(g, radius, None, torch.tensor(V, device="cuda"), torch.float64)
    Y, X = (torch.zeros((1, leading_dim(g.npts)), dtype=torch.float64, device="cuda") for _ in range(2))
    Y[0, :g.npts] = torch.tensor(y)
    X[0, :g.npts] = torch.tensor(x)
    H.step(Y, X, X, 1, 0.7, -0.3, -1.1)
    lap = ofd.laplacian_masked(nx, ny, nz, radius, g.mask)
    want = 0.7 * (0.5 / h ** 2 * (lap @ y) + V * y) - 0.3 * y - 1.1 * x
    assert np.max(np.abs(X[0, :g.npts].cpu().numpy() - want)) <= 1e-13 * (np.abs(want).max() + 30 / h ** 2)
    H.close()
