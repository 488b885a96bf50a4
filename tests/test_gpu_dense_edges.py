"""Edges of the dense stage's own kernels: orders around the multiples of the
32-column Cholesky blocks and of the 64 lanes that hold a column's rows, the
orders where the tridiagonalization changes kernels, and pencils whose
reflectors vanish (a diagonal matrix: no column has anything to annihilate).

Against scipy's generalised eigensolver.  Both are backward stable: eigenvalues
within 1e-11 k of the pencil's scale (some 1e4 units of rounding per order), the
eigenvectors' residuals likewise."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ORDERS = [1, 2, 3, 8, 9, 31, 33, 63, 64, 65, 71, 96, 97, 127, 128, 129, 191, 192, 193, 255, 257, 288, 319, 320]


@pytest.mark.parametrize("kind", ["full", "diagonal"])
@pytest.mark.parametrize("k", ORDERS)
def test_dense_rr_edges(gpu, k, kind):
    import ctypes as C
    import torch
    from scipy.linalg import eigh
    from parsec_python_amd import _lib
    from parsec_python_amd.hamiltonian import BlockLinalg
    print(f"dense edge case k={k} {kind}", flush=True)
    rng = np.random.default_rng(7 * k + len(kind))
    if kind == "full":
        B = rng.standard_normal((2 * k, k))
        S = B.T @ B / B.shape[0] + 0.5 * np.eye(k)
        M = rng.standard_normal((k, k))
        G = M + M.T
    else:
        S = np.diag(rng.uniform(0.5, 2.0, k))
        G = np.diag(rng.standard_normal(k))
    ref = eigh(G, S, eigvals_only=True)
    scale = max(1.0, np.abs(ref).max())
    la = BlockLinalg(10, k)
    for rep in range(2):                    # the second call reuses the first one's workspace
        Sd = torch.tensor(S.T.copy(), device="cuda").view(-1)
        Gd = torch.tensor(G.T.copy(), device="cuda").view(-1)
        T, lam = la.dense_rr(Sd, Gd, k)
        assert np.allclose(lam, ref, rtol=0, atol=1e-11 * scale * k)
        Tm = T.cpu().numpy()[:k * k].reshape(k, k).T
        assert np.abs(Tm.T @ S @ Tm - np.eye(k)).max() < 1e-10 * k
        assert np.abs(Tm.T @ G @ Tm - np.diag(lam)).max() < 1e-10 * scale * k
    aborts = C.c_int(-1)
    _lib.call("pc_dense_trd_control", la.dense, 0, 0, C.byref(aborts))
    assert aborts.value == 0
    la.close()
