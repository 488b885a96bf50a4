"""Volumes that the layer kernels' boxes cover badly (lines and thin slabs): the
forms over voxels in flat order, against FP64, and their times.

Tolerances: K products and sums in FP32 err by at most (K + 2) 2^-24 of the sum of
their absolute values; a BF16 result by 2^-8 of itself besides."""
import ctypes as C

import numpy as np
import pytest

from tests.test_gpu_unet_edges import SLOPE, U, _shift

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cin,cout,dims", [(1, 16, (1, 1, 20001)), (1, 33, (20001, 1, 1)), (16, 16, (1, 20001, 1)),
                                           (16, 5, (2, 1, 40001)), (48, 16, (20001, 1, 1)), (64, 64, (1, 1, 20001)),
                                           (112, 48, (2, 2, 12001))])
@pytest.mark.parametrize("mode", [0, 1, 2])
def test_thin_conv(gpu, cin, cout, dims, mode):
    import torch
    from parsec_python_amd import _lib
    from parsec_python_amd.device import ptr, stream
    print(f"thin conv cin={cin} cout={cout} dims={dims} mode={mode}", flush=True)
    d, h, w = dims
    V = d * h * w
    g = torch.Generator().manual_seed(cin + cout)
    X = torch.randn(V, cin, generator=g).to(torch.bfloat16)
    W = (torch.randn(cout, 27, cin, generator=g) / 9).to(torch.bfloat16)
    b = torch.randn(cout, generator=g)
    Y = torch.full((V + 1, cout), 7.0, dtype=torch.bfloat16 if mode == 1 else torch.float32, device="cuda")
    Xd, Wd, bd = X.cuda(), W.cuda(), b.cuda()
    _lib.call("pc_unet_conv3d_fwd", ptr(Xd), cin, cin, ptr(Wd), ptr(bd) if mode < 2 else None, cout, d, h, w, mode,
              SLOPE, ptr(Y), cout, stream())
    x, wt = X.double().numpy(), W.double().numpy()
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
    assert np.all(np.abs(got[:V] - ref) <= tol)
    assert np.all(got[V:] == 7.0)


@pytest.mark.parametrize("cin,cout,dims", [(1, 16, (1, 1, 513)), (16, 1, (5000, 1, 1)), (17, 18, (1, 701, 1)),
                                           (48, 16, (1, 1, 20001)), (16, 16, (1500, 2, 1)), (3, 2, (1, 1, 512))])
@pytest.mark.parametrize("small", [True, False])
def test_thin_weight_gradient(gpu, cin, cout, dims, small):
    import torch
    from parsec_python_amd import _lib
    from parsec_python_amd.device import ptr, stream
    print(f"thin weight gradient cin={cin} cout={cout} dims={dims} small={small}", flush=True)
    d, h, w = dims
    V = d * h * w
    g = torch.Generator().manual_seed(cin + 3 * cout)
    X = torch.randn(V, cin, generator=g).to(torch.bfloat16)
    Z = torch.randn(V, cout, generator=g).to(torch.bfloat16)
    n = C.c_size_t()
    _lib.call("pc_unet_wgrad_workspace", cout, cin, C.byref(n))
    nbytes = 64 * cout * 27 * cin * 4 if small else n.value       # the smallest accepted: 64 splits
    work = torch.full((nbytes // 4 + 8,), 7.0, device="cuda")
    dw = torch.empty(cout, 27, cin, device="cuda")
    Xd, Zd = X.cuda(), Z.cuda()
    _lib.call("pc_unet_conv3d_wgrad", ptr(Zd), cout, cout, ptr(Xd), cin, cin, d, h, w, ptr(dw), ptr(work), nbytes,
              stream())
    x, z = X.double().numpy(), Z.double().numpy()
    for k in range(27):
        s = _shift(x, k, dims)
        err = np.abs(dw[:, k].double().cpu().numpy() - z.T @ s)
        assert np.all(err <= (V + 2) * U * (np.abs(z).T @ np.abs(s)))
    assert bool((work[nbytes // 4:] == 7.0).all())


@pytest.mark.parametrize("what", ["conv", "wgrad"])
def test_a_line_costs_about_as_much_as_a_cube(gpu, what):
    """110,592 voxels, 48 -> 16 channels (in boxes a line cost 30 and 12 times a
    cube; gathered it took 1.5 and 5 times as long)."""
    import torch
    from parsec_python_amd import _lib
    from parsec_python_amd.device import ptr, stream
    cin, cout, V = 48, 16, 48 ** 3
    X, Z = (torch.zeros(V, c, dtype=torch.bfloat16, device="cuda") for c in (cin, cout))
    W, dw = torch.zeros(cout, 27, cin, dtype=torch.bfloat16, device="cuda"), torch.empty(cout, 27, cin, device="cuda")
    n = C.c_size_t()
    _lib.call("pc_unet_wgrad_workspace", cout, cin, C.byref(n))
    work, Y = torch.empty(n.value, dtype=torch.uint8, device="cuda"), torch.empty(V, cout, device="cuda")
    times = []
    for dims in ((48, 48, 48), (V, 1, 1)):
        print(f"{what} {dims}", flush=True)

        def call():
            if what == "conv":
                _lib.call("pc_unet_conv3d_fwd", ptr(X), cin, cin, ptr(W), None, cout, *dims, 2, SLOPE, ptr(Y), cout,
                          stream())
            else:
                _lib.call("pc_unet_conv3d_wgrad", ptr(Z), cout, cout, ptr(X), cin, cin, *dims, ptr(dw), ptr(work),
                          n.value, stream())
        t = []
        for _ in range(9):
            e0, e1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            call()
            e0.record()
            for _ in range(4):
                call()
            e1.record()
            torch.cuda.synchronize()
            t.append(250 * e0.elapsed_time(e1))
        times.append(sorted(t)[4])
    print(f"{times[0]:.1f} and {times[1]:.1f} us", flush=True)
    assert times[1] <= (4 if what == "conv" else 9) * times[0]
