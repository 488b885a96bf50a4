"""Gram products in the smallest workspaces that they take."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _smallest_gram_workspace(n, kx, ky, sym):
    """Bytes of the partial sums in tiles of 64 x 64, chunks of 1024 points and up, 2048 tiles at most."""
    ti, tj = -(-kx // 64), -(-ky // 64)
    ntile = ti * (ti + 1) // 2 if sym else ti * tj
    nchunk = min(max(1, 2048 // ntile), max(1, -(-n // 1024)))
    chunk = -(-(-(-n // nchunk)) // 32) * 32
    return -(-n // chunk) * ntile * 4096 * 8


@pytest.mark.parametrize("n,kx,ky,sym", [(5, 3, 2, False), (40, 64, 64, True), (250, 97, 97, True), (999, 275, 275, True),
                                         (1000, 20, 100, False), (1023, 96, 96, False), (4099, 300, 40, False),
                                         (65541, 100, 100, True)])
@pytest.mark.parametrize("dtype", ["f64", "f32"])
def test_gram_smallest_workspace(gpu, n, kx, ky, sym, dtype):
    """Tolerance: n products in FP64 ((n + 2) eps), in FP32 16 of them at a time (17 u)."""
    import torch
    from parsec_python_amd import _lib
    from parsec_python_amd.device import ptr, stream
    print(f"gram workspace case n={n} kx={kx} ky={ky} sym={sym} {dtype}", flush=True)
    tdt = torch.float64 if dtype == "f64" else torch.float32
    ld = (n + 15) // 16 * 16
    g = torch.Generator(device="cuda").manual_seed(n + kx)
    X = torch.full((kx, ld), float("nan"), dtype=tdt, device="cuda")
    X[:, :n] = torch.randn((kx, n), generator=g, dtype=tdt, device="cuda")
    Y = X
    if not sym:
        Y = torch.full((ky, ld), float("nan"), dtype=tdt, device="cuda")
        Y[:, :n] = torch.randn((ky, n), generator=g, dtype=tdt, device="cuda")
    nbytes = _smallest_gram_workspace(n, kx, ky, sym)
    work = torch.full((nbytes // 8 + 64,), 7.0, dtype=torch.float64, device="cuda")
    S = torch.full((ky, kx), float("nan"), dtype=torch.float64, device="cuda")
    _lib.call(f"pc_gram_{dtype}", ptr(X), ld, ptr(Y), ld, n, kx, ky, ptr(S), kx, int(sym), ptr(work), nbytes, stream())
    x, y = X[:, :n].double().cpu().numpy(), Y[:, :n].double().cpu().numpy()
    tol = (n + 2) * 2.0 ** -53 if dtype == "f64" else 17 * 2.0 ** -24 + n * 2.0 ** -53
    assert np.all(np.abs(S.cpu().numpy() - y @ x.T) <= 2 * tol * (np.abs(y) @ np.abs(x).T))
    assert bool((work[nbytes // 8:] == 7.0).all())
