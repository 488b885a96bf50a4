"""Gram and rotation at the limits of their arguments: the smallest workspaces
that the Gram product takes, and columns beyond 2^24 points."""
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


def _rotate(X, n, Q, dtype, ldz, Z=None):
    """Z = X Q through pc_rotate_*; X: (kx, ldx), Q: (ky, kx) with row j = column j."""
    import ctypes as C
    import torch
    from parsec_python_amd import _lib
    from parsec_python_amd.device import ptr, stream
    ky, kx = Q.shape
    nbytes = C.c_size_t()
    _lib.call("pc_rotate_workspace", kx, ky, int(dtype == "f32"), C.byref(nbytes))
    work = torch.empty(nbytes.value, dtype=torch.uint8, device="cuda")
    if Z is None:
        Z = torch.full((ky, ldz), 7.0, dtype=X.dtype, device="cuda")
    _lib.call(f"pc_rotate_{dtype}", ptr(X), X.shape[1], ptr(Q), kx, ptr(Z), ldz, n, kx, ky, ptr(work), nbytes.value,
              stream())
    return Z


# columns just beyond 2^24 points; columns whose 16 exceed 32-bit byte offsets
@pytest.mark.parametrize("dtype,n,ldx,kx,ky", [("f32", 2 ** 24 + 21, 2 ** 24 + 32, 3, 2), ("f64", 2 ** 24 + 21, 2 ** 24 + 32, 3, 2),
                                               ("f32", 1003, 72_000_000, 17, 20), ("f64", 1003, 36_000_000, 17, 20)])
def test_rotate_long_columns(gpu, dtype, n, ldx, kx, ky):
    """Tolerance: kx products added in order, ((kx + 2) u), Q rounded once in FP32."""
    import torch
    print(f"long columns {dtype} n={n} ldx={ldx} kx={kx} ky={ky}", flush=True)
    tdt, u = (torch.float64, 2.0 ** -53) if dtype == "f64" else (torch.float32, 2.0 ** -24)
    g = torch.Generator(device="cuda").manual_seed(kx)
    X = torch.empty((kx, ldx), dtype=tdt, device="cuda")
    X[:, :n] = torch.randn((kx, n), generator=g, dtype=tdt, device="cuda")
    X[:, n:n + 64] = float("nan")
    Q = torch.randn((ky, kx), generator=g, dtype=torch.float64, device="cuda")
    Z = _rotate(X, n, Q, dtype, (n + 15) // 16 * 16)
    for j in range(ky):
        ref = (Q[j, :, None] * X[:, :n].double()).sum(0)
        mag = (Q[j, :, None] * X[:, :n].double()).abs().sum(0)
        assert bool(((Z[j, :n].double() - ref).abs() <= 2 * (kx + 2) * u * mag).all())
    assert bool((Z[:, n:] == 7.0).all())


def test_rotate_long_columns_split_bf16(gpu):
    """The optional split form serves long columns too: the bits of the same block in short ones."""
    import torch
    from parsec_python_amd import _lib
    n, kx, ky = 1003, 17, 20
    print("long columns, split form", flush=True)
    g = torch.Generator(device="cuda").manual_seed(5)
    short = torch.randn((kx, 1008), generator=g, device="cuda")
    long = torch.empty((kx, 2 ** 24 + 32), device="cuda")
    long[:, :n] = short[:, :n]
    Q = torch.randn((ky, kx), generator=g, dtype=torch.float64, device="cuda")
    plain = _rotate(short, n, Q, "f32", 1008)
    try:
        _lib.call("pc_rotate_set_split_bf16", 1)
        a, b = _rotate(short, n, Q, "f32", 1008), _rotate(long, n, Q, "f32", 1008)
    finally:
        _lib.call("pc_rotate_set_split_bf16", 0)
    assert not torch.equal(a, plain)
    assert torch.equal(a, b)


@pytest.mark.parametrize("dtype", ["f32", "f64"])
def test_rotate_long_columns_keep_their_speed(gpu, dtype):
    """Columns on either side of 2^24 points take the same kernel (96 columns of
    400,000 points: 93 us in FP32 and 165 in FP64, 150 and 350 with the general one)."""
    import torch
    print(f"long columns' time {dtype}", flush=True)
    n, k = 400_000, 96
    tdt = torch.float64 if dtype == "f64" else torch.float32
    Q = torch.ones((k, k), dtype=torch.float64, device="cuda")
    blocks = [torch.zeros((k, 2 ** 24 + d), dtype=tdt, device="cuda") for d in (-1040, 1040)]
    times = [[], []]
    for _ in range(9):
        for i, X in enumerate(blocks):
            torch.cuda.synchronize()
            e0, e1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            Z = _rotate(X, n, Q, dtype, n)
            e0.record()
            for _ in range(4):
                _rotate(X, n, Q, dtype, n, Z)
            e1.record()
            torch.cuda.synchronize()
            times[i].append(e0.elapsed_time(e1))
    short, long = (sorted(t)[4] for t in times)
    print(f"{250 * short:.1f} and {250 * long:.1f} us", flush=True)
    assert long <= 1.25 * short


@pytest.mark.parametrize("n,k", [(16, 33), (100, 100), (128, 275), (255, 289), (257, 520), (1000, 300), (2001, 577)])
@pytest.mark.parametrize("dtype", ["f64", "f32"])
def test_short_columns(gpu, n, k, dtype):
    """Narrower Gram tiles and rotation blocks, few chunks: against FP64 (tolerances as above)."""
    import torch
    from parsec_python_amd import _lib
    from parsec_python_amd.device import ptr, stream
    import ctypes as C
    print(f"short columns n={n} k={k} {dtype}", flush=True)
    tdt, u = (torch.float64, 2.0 ** -53) if dtype == "f64" else (torch.float32, 2.0 ** -24)
    ld = (n + 15) // 16 * 16
    g = torch.Generator(device="cuda").manual_seed(n + k)
    X = torch.full((k, ld), float("nan"), dtype=tdt, device="cuda")
    Y = torch.full((k + 3, ld), float("nan"), dtype=tdt, device="cuda")
    X[:, :n] = torch.randn((k, n), generator=g, dtype=tdt, device="cuda")
    Y[:, :n] = torch.randn((k + 3, n), generator=g, dtype=tdt, device="cuda")
    x, y = X[:, :n].double().cpu().numpy(), Y[:, :n].double().cpu().numpy()
    tol = (n + 2) * 2.0 ** -53 if dtype == "f64" else 17 * 2.0 ** -24 + n * 2.0 ** -53
    for ky, other, sym in ((k, X, 1), (k + 3, Y, 0)):
        nb = C.c_size_t()
        _lib.call("pc_gram_workspace", n, k, ky, sym, C.byref(nb))
        work = torch.full((nb.value // 8 + 64,), 7.0, dtype=torch.float64, device="cuda")
        S = torch.full((ky, k), float("nan"), dtype=torch.float64, device="cuda")
        _lib.call(f"pc_gram_{dtype}", ptr(X), ld, ptr(other), ld, n, k, ky, ptr(S), k, sym, ptr(work), nb.value, stream())
        b = x if sym else y
        assert np.all(np.abs(S.cpu().numpy() - b @ x.T) <= 2 * tol * (np.abs(b) @ np.abs(x).T))
        assert bool((work[nb.value // 8:] == 7.0).all())
    Q = torch.randn((k + 3, k), generator=g, dtype=torch.float64, device="cuda")
    Z = _rotate(X, n, Q, dtype, ld)
    q = Q.cpu().numpy()
    assert np.all(np.abs(Z[:, :n].double().cpu().numpy() - q @ x) <= 2 * (k + 2) * u * (np.abs(q) @ np.abs(x)))
    assert bool((Z[:, n:] == 7.0).all())
