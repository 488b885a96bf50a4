"""Edges of the aligned Gram and rotation kernels: tile widths (32, 64, 96
columns), column blocks of the rotation, partial point stages, and the general
form for unaligned columns, against FP64 NumPy.

Tolerances (absolute values of the products summed, eps = 2^-53, u = 2^-24):
FP64 products and sums over n points err by at most (n + 2) eps each; the FP32
Gram sums 16 products in FP32 (17 u) and the rest in FP64; the FP32 rotation
rounds Q once and adds k products in order ((k + 2) u)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 1), (15, 3, 2), (16, 16, 17), (33, 32, 33), (257, 64, 65), (1000, 96, 97), (4099, 17, 129),
         (2053, 128, 128), (777, 275, 275), (1024, 288, 289), (513, 300, 320), (130, 577, 20), (95, 20, 577)]


@pytest.mark.parametrize("n,kx,ky", SIZES)
@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("aligned", [True, False])
def test_gram_rotate_edges(gpu, n, kx, ky, dtype, aligned):
    import torch
    from parsec_python_amd.hamiltonian import BlockLinalg
    print(f"gemm edge case n={n} kx={kx} ky={ky} {dtype} aligned={aligned}", flush=True)
    tdt = torch.float64 if dtype == "f64" else torch.float32
    rng = np.random.default_rng(n * 7 + kx)
    ld = (n + 15) // 16 * 16 if aligned else n + (1 if n % 2 == 0 else 0)   # odd: no 16-byte columns
    X = torch.full((kx, ld), float("nan"), dtype=tdt, device="cuda")   # the padding must not reach a result
    Y = torch.full((ky, ld), float("nan"), dtype=tdt, device="cuda")
    X[:, :n] = torch.tensor(rng.standard_normal((kx, n)), dtype=tdt)
    Y[:, :n] = torch.tensor(rng.standard_normal((ky, n)), dtype=tdt)
    Q = torch.tensor(rng.standard_normal((ky, kx)), device="cuda")      # row j: column j of Q
    Xh, Yh, Qh = X[:, :n].double().cpu().numpy(), Y[:, :n].double().cpu().numpy(), Q.cpu().numpy()
    la = BlockLinalg(n, max(kx, ky))
    eps, u = 2.0 ** -53, 2.0 ** -24
    gram_tol = (n + 2) * eps if dtype == "f64" else 17 * u + n * eps
    G = torch.empty(ky, kx, dtype=torch.float64, device="cuda")
    la.gram(X, Y, kx, ky, G.view(-1), sym=False)
    S = torch.empty(kx, kx, dtype=torch.float64, device="cuda")
    la.gram(X, X, kx, kx, S.view(-1), sym=True)
    for got, A, B in ((G, Yh, Xh), (S, Xh, Xh)):
        err = np.abs(got.cpu().numpy() - A @ B.T)
        assert np.all(err <= 2 * gram_tol * (np.abs(A) @ np.abs(B).T)), err.max()
    Z = torch.full((ky, ld), 7.0, dtype=tdt, device="cuda")
    la.rotate(X, Q.view(-1), kx, ky, Z)
    rot_tol = (kx + 2) * (eps if dtype == "f64" else u)
    err = np.abs(Z[:, :n].double().cpu().numpy() - Qh @ Xh)
    assert np.all(err <= 2 * rot_tol * (np.abs(Qh) @ np.abs(Xh))), err.max()
    assert bool((Z[:, n:] == 7.0).all())
    la.close()
