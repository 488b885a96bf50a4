"""Infinities stay where the sums put them: lanes that a kernel fills up beyond
its sum (the last round of a projector's support, taps past the 27th, voxels of a
box beyond the volume) must not turn an infinity next to them into a NaN."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

INF = float("inf")


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("size", [1, 63, 65, 300])
def test_projector_gather_infinite_value(gpu, size, dtype):
    """The support's last point holds an infinity: C is that infinity, by the signs of u."""
    import torch
    from parsec_python_amd import _lib
    from parsec_python_amd.device import ptr, stream
    print(f"projector infinity size={size} {dtype}", flush=True)
    npts, nvec = 512, 5
    aptr = np.array([0, size, 2 * size], np.int32)
    pts = np.concatenate([np.arange(size), 100 + np.arange(size)]).astype(np.int32)
    uv = np.tile([1.0, -2.0, 0.5], (2 * size, 1))
    sc = np.ones(2)
    handle = C.c_void_p()
    pi, pd = C.POINTER(C.c_int), C.POINTER(C.c_double)
    _lib.call("pc_proj_create", 2, aptr.ctypes.data_as(pi), pts.ctypes.data_as(pi), uv.ctypes.data_as(pd),
              sc.ctypes.data_as(pd), npts, C.byref(handle))
    Y = torch.ones((nvec, npts), dtype=torch.float64 if dtype == "f64" else torch.float32, device="cuda")
    Y[2, 99 + size] = INF          # the second atom's last point, vector 2
    cb = torch.empty((2, nvec, 3), dtype=torch.float64, device="cuda")
    _lib.call(f"pc_proj_gather_{dtype}", handle, ptr(Y), npts, nvec, ptr(cb), stream())
    ref = np.tile(size * np.array([1.0, -2.0, 0.5]), (2, nvec, 1))
    ref[1, 2] = [INF, -INF, INF]
    assert np.array_equal(cb.cpu().numpy(), ref)
    _lib.call("pc_proj_destroy", handle)


@pytest.mark.parametrize("dims", [(5, 6, 7), (64, 32, 64)])
def test_one_channel_conv_infinite_voxel(gpu, dims):
    """One input channel: the infinity reaches its 27 neighbours as an infinity."""
    import torch
    from parsec_python_amd import _lib
    from parsec_python_amd.device import ptr, stream
    print(f"conv infinity dims={dims}", flush=True)
    d, h, w = dims
    X = torch.ones((d, h, w), dtype=torch.bfloat16, device="cuda")
    z, y, x = 2, 3, 4
    X[z, y, x] = INF
    W = torch.ones((16, 27), dtype=torch.bfloat16, device="cuda")
    Y = torch.zeros((d, h, w, 16), device="cuda")
    _lib.call("pc_unet_conv3d_fwd", ptr(X), 1, 1, ptr(W), None, 16, d, h, w, 2, 0.1, ptr(Y), 16, stream())
    ones = torch.nn.functional.conv3d(torch.ones(1, 1, d, h, w), torch.ones(1, 1, 3, 3, 3), padding=1)[0, 0].cuda()
    ones[z - 1:z + 2, y - 1:y + 2, x - 1:x + 2] = INF
    assert torch.equal(Y, ones[..., None].expand(d, h, w, 16))


@pytest.mark.parametrize("cin,cout", [(16, 16), (16, 1), (1, 16)])
@pytest.mark.parametrize("dims", [(5, 6, 7), (4, 8, 17), (9, 8, 16), (4, 9, 24)])
def test_conv_weight_gradient_infinite_corner(gpu, cin, cout, dims):
    """An infinity in the volume's last voxel reaches only the taps that pair it
    with a voxel of the volume (also where the boxes go beyond the volume)."""
    import torch
    from parsec_python_amd import _lib
    from parsec_python_amd.device import ptr, stream
    print(f"wgrad infinity cin={cin} cout={cout} dims={dims}", flush=True)
    d, h, w = dims
    X = torch.ones((d, h, w, cin), dtype=torch.bfloat16, device="cuda")
    X[-1, -1, -1, 0] = INF
    Z = torch.ones((d, h, w, cout), dtype=torch.bfloat16, device="cuda")
    n = C.c_size_t()
    _lib.call("pc_unet_wgrad_workspace", cout, cin, C.byref(n))
    work = torch.empty(n.value, dtype=torch.uint8, device="cuda")
    dw = torch.empty((cout, 3, 3, 3, cin), device="cuda")
    _lib.call("pc_unet_conv3d_wgrad", ptr(Z), cout, cout, ptr(X), cin, cin, d, h, w, ptr(dw), ptr(work), n.value,
              stream())
    # tap (a, b, c) pairs voxel v with v + (a - 1, b - 1, c - 1): the last voxel is in it unless a component is -1
    count = [np.array([s - 1.0, s, s - 1.0]) for s in dims]
    ref = np.einsum("a,b,c->abc", *count)[..., None].repeat(cin, -1)
    ref[1:, 1:, 1:, 0] = INF
    assert np.array_equal(dw.cpu().numpy(), np.broadcast_to(ref, dw.shape))
