"""Edges of the network's layer kernels: box remainders, every staged channel
count and the general form beyond them, unaligned channel strides, one-channel
tensors, and workspaces of the smallest accepted size, against FP64.

Tolerances: K products and sums in FP32 err by at most (K + 2) 2^-24 of the sum
of their absolute values; a BF16 result by 2^-8 of itself besides."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

U = 2.0 ** -24
SLOPE = 0.1


def _shift(t, k, dims):
    """Volume (V, c) moved so that row v holds tap k's neighbour (zero outside)."""
    d, h, w = dims
    p = np.pad(t.reshape(d, h, w, -1), ((1, 1), (1, 1), (1, 1), (0, 0)))
    return p[k // 9:k // 9 + d, k // 3 % 3:k // 3 % 3 + h, k % 3:k % 3 + w].reshape(d * h * w, -1)


CONV = [(1, 16, (5, 7, 9), 0), (1, 1, (4, 4, 4), 0), (16, 16, (9, 10, 17), 0), (16, 48, (64, 32, 33), 0), (32, 32, (6, 9, 8), 0),
        (32, 17, (40, 40, 16), 0), (48, 16, (20, 36, 50), 0), (48, 16, (3, 3, 70), 4), (64, 64, (7, 7, 7), 0),
        (80, 32, (6, 5, 4), 0), (96, 5, (4, 4, 9), 8), (112, 48, (14, 10, 12), 0), (128, 16, (5, 5, 5), 0),
        (16, 1, (12, 8, 8), 0), (16, 16, (48, 48, 56), 0)]


@pytest.mark.parametrize("cin,cout,dims,pad", CONV)
@pytest.mark.parametrize("mode", [0, 1, 2])
def test_conv_edges(gpu, cin, cout, dims, pad, mode):
    import torch
    from parsec_python_amd import _lib
    from parsec_python_amd.device import ptr, stream
    print(f"conv edge cin={cin} cout={cout} dims={dims} pad={pad} mode={mode}", flush=True)
    d, h, w = dims
    V = d * h * w
    g = torch.Generator().manual_seed(cin * 7 + cout)
    ldx, ldy = cin + pad, cout + pad
    X = torch.full((V, ldx), float("nan"), dtype=torch.bfloat16)
    X[:, :cin] = torch.randn(V, cin, generator=g).to(torch.bfloat16)
    W = (torch.randn(cout, 27, cin, generator=g) / 9).to(torch.bfloat16)
    b = torch.randn(cout, generator=g)
    Y = torch.full((V, ldy), 7.0, dtype=torch.bfloat16 if mode == 1 else torch.float32, device="cuda")
    Xd, Wd, bd = X.cuda(), W.cuda(), b.cuda()
    _lib.call("pc_unet_conv3d_fwd", ptr(Xd), ldx, cin, ptr(Wd), ptr(bd) if mode < 2 else None, cout, d, h, w, mode,
              SLOPE, ptr(Y), ldy, stream())
    x, wt = X[:, :cin].double().numpy(), W.double().numpy()
    ref, mag = np.zeros((V, cout)), np.zeros((V, cout))
    for k in range(27):
        s = _shift(x, k, dims)
        ref += s @ wt[:, k].T
        mag += np.abs(s) @ np.abs(wt[:, k]).T
    if mode < 2:
        ref += b.double().numpy()
        mag += np.abs(b.double().numpy())
    tol = (27 * cin + 4) * U * mag
    if mode == 1:
        ref = np.where(ref > 0, ref, SLOPE * ref)
        tol = tol + 2.0 ** -8 * np.abs(ref)
    got = Y.double().cpu().numpy()
    assert np.all(np.abs(got[:, :cout] - ref) <= tol)
    assert np.all(got[:, cout:] == 7.0)


@pytest.mark.parametrize("cin,cout,dims,pad", [c for c in CONV if c[0] <= 112])
@pytest.mark.parametrize("small", [True, False])
def test_layer_backward_edges(gpu, cin, cout, dims, pad, small):
    """Activation backward with the bias gradient, and the weight gradient."""
    import torch
    from parsec_python_amd import _lib
    from parsec_python_amd.device import ptr, stream
    print(f"layer backward edge cin={cin} cout={cout} dims={dims} pad={pad} small={small}", flush=True)
    d, h, w = dims
    V = d * h * w
    g = torch.Generator().manual_seed(cin + 5 * cout)
    dA = torch.randn(V, cout + pad, generator=g)
    a = torch.randn(V, cout + pad, generator=g).to(torch.bfloat16)
    X = torch.randn(V, cin + pad, generator=g).to(torch.bfloat16)
    n = C.c_size_t()
    _lib.call("pc_unet_act_bwd_workspace", cout, V, C.byref(n))
    nact = -(-V // 2048) * cout * 4 if small else n.value      # the smallest accepted: chunks of 2048 voxels
    _lib.call("pc_unet_wgrad_workspace", cout, cin, C.byref(n))
    nwg = 64 * cout * 27 * cin * 4 if small else n.value       # the smallest accepted: 64 splits
    dz = torch.full((V, cout + pad), 7.0, dtype=torch.bfloat16, device="cuda")
    db = torch.empty(cout, device="cuda")
    work = torch.empty(nact, dtype=torch.uint8, device="cuda")
    dAd, ad, Xd = dA.cuda(), a.cuda(), X.cuda()
    _lib.call("pc_unet_act_bwd", ptr(dAd), cout + pad, ptr(ad), cout + pad, cout, d, h, w, SLOPE, ptr(dz), cout + pad,
              ptr(db), ptr(work), nact, stream())
    gref = dA[:, :cout].double() * torch.where(a[:, :cout].double() > 0, 1.0, float(np.float32(SLOPE)))
    assert torch.all((dz[:, :cout].double().cpu() - gref).abs() <= 2.0 ** -8 * gref.abs() + 1e-30)
    assert bool((dz[:, cout:] == 7.0).all())
    assert torch.all((db.double().cpu() - gref.sum(0)).abs() <= (V + 2) * U * gref.abs().sum(0))
    work = torch.empty(nwg, dtype=torch.uint8, device="cuda")
    dw = torch.empty(cout, 27, cin, device="cuda")
    _lib.call("pc_unet_conv3d_wgrad", ptr(dz), cout + pad, cout, ptr(Xd), cin + pad, cin, d, h, w, ptr(dw),
              ptr(work), nwg, stream())
    z, x = dz[:, :cout].double().cpu().numpy(), X[:, :cin].double().numpy()
    for k in range(27):
        s = _shift(x, k, dims)
        err = np.abs(dw[:, k].double().cpu().numpy() - z.T @ s)
        assert np.all(err <= (V + 2) * U * (np.abs(z).T @ np.abs(s)))
