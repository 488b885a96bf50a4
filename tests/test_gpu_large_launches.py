"""Calls whose workgroups are more than one launch dimension of 2^32 work-items
holds, or whose volume has 2^31 voxels and more: small results of large operands,
exact by construction (whole numbers and single products)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture
def room(gpu):
    """room(bytes): skips where the card has less than that free, and frees the cache afterwards."""
    import torch

    def need(nbytes):
        torch.cuda.empty_cache()
        if torch.cuda.mem_get_info()[0] < nbytes * 1.1:
            pytest.skip("not enough free device memory")
    yield need
    torch.cuda.empty_cache()


def test_gather_of_many_atoms_and_vectors(gpu, room):
    """4,099 atoms of one point each, 16,385 vectors: 2^24 workgroups and more."""
    import torch
    from parsec_python_amd import _lib
    from parsec_python_amd.device import ptr, stream
    na, nvec, npts = 4099, 16385, 64
    print(f"gather of {na} atoms and {nvec} vectors", flush=True)
    room(na * nvec * 3 * 8 * 2)
    aptr, pts = np.arange(na + 1, dtype=np.int32), (np.arange(na) % npts).astype(np.int32)
    uv = np.stack([np.arange(na) % 7 + 1.0, np.arange(na) % 5 - 2.0, np.arange(na) % 3 + 0.5], 1)
    sc = np.ones(na)
    handle = C.c_void_p()
    pi, pd = C.POINTER(C.c_int), C.POINTER(C.c_double)
    _lib.call("pc_proj_create", na, aptr.ctypes.data_as(pi), pts.ctypes.data_as(pi), uv.ctypes.data_as(pd),
              sc.ctypes.data_as(pd), npts, C.byref(handle))
    Y = torch.arange(nvec * npts, device="cuda").remainder(1009).float().view(nvec, npts)
    cb = torch.full((na, nvec, 3), float("nan"), dtype=torch.float64, device="cuda")
    _lib.call("pc_proj_gather_f32", handle, ptr(Y), npts, nvec, ptr(cb), stream())
    u = torch.tensor(uv, device="cuda")
    y = Y.double().T[torch.tensor(pts, device="cuda").long()]          # (na, nvec)
    for m in range(3):
        assert torch.equal(cb[:, :, m], u[:, m, None] * y)
    _lib.call("pc_proj_destroy", handle)


def test_rotation_of_one_very_long_column(gpu, room):
    """FP64, 2^30 + 70 points: 2^24 workgroups of 64 points and more."""
    import torch
    from parsec_python_amd import _lib
    from parsec_python_amd.device import ptr, stream
    n = 2 ** 30 + 70
    print(f"rotation of {n} points", flush=True)
    ld = (n + 15) // 16 * 16
    room(3 * ld * 8)
    X = torch.arange(ld, dtype=torch.float64, device="cuda")
    Z = torch.full((ld,), -1.0, dtype=torch.float64, device="cuda")
    Q = torch.full((1,), 3.0, dtype=torch.float64, device="cuda")
    work = torch.empty(1, dtype=torch.float64, device="cuda")
    _lib.call("pc_rotate_f64", ptr(X), ld, ptr(Q), 1, ptr(Z), ld, n, 1, 1, ptr(work), 8, stream())
    assert bool((Z[n:] == -1.0).all())
    assert torch.equal(Z[:n], X[:n].mul_(3.0))


def test_stencil_of_many_vectors(gpu, room):
    """2^3 points, radius 6, 6,000,001 vectors: more than 2^32 work-items in workgroups of 768."""
    import torch
    from parsec_python_amd import _lib
    from parsec_python_amd.device import ptr, stream
    from parsec_python_amd.grid import DeviceGrid, make_grid
    nvec, ld = 6_000_001, 8
    print(f"stencil of {nvec} vectors", flush=True)
    room(4 * nvec * ld * 4)
    dg = DeviceGrid(make_grid(2, 0.5, 1.0, "cube"), 6)
    Y = torch.arange(nvec * ld, device="cuda").remainder(1013).float().view(nvec, ld)
    X = torch.arange(nvec * ld, device="cuda").remainder(17).float().view(nvec, ld)
    V = torch.ones(8, device="cuda")
    out = torch.full((nvec, ld), float("nan"), device="cuda")

    def step(v0, n, o):
        _lib.call("pc_stencil_f32", dg.handle, ptr(Y[v0:]), ptr(X[v0:]), ptr(o), ptr(V), n, ld, 0.5, 1.0, -0.25, 2.0,
                  None, stream())
    step(0, nvec, out)
    part = torch.empty_like(out)
    for v0 in range(0, nvec, 1_000_000):
        step(v0, min(1_000_000, nvec - v0), part[v0:])
    assert torch.equal(out, part)
    dg.close()


def test_conv_of_many_output_channels(gpu, room):
    """128 x 128 x 64 voxels, 64 -> 2^15 + 16 channels: 2^24 workgroups and more;
    equal to the same weights' channels in calls of their own."""
    import torch
    from parsec_python_amd import _lib
    from parsec_python_amd.device import ptr, stream
    d, h, w, cin, cout = 128, 128, 64, 64, 2 ** 15 + 16
    print(f"conv of {cout} output channels", flush=True)
    V = d * h * w
    room(V * cout * 2)
    g = torch.Generator(device="cuda").manual_seed(3)
    X = torch.randn((V, cin), generator=g, device="cuda").to(torch.bfloat16)
    W = torch.randn((cout, 27, cin), generator=g, device="cuda").to(torch.bfloat16)
    b = torch.randn(cout, generator=g, device="cuda")
    Y = torch.empty((V, cout), dtype=torch.bfloat16, device="cuda")

    def conv(c0, n, out):
        _lib.call("pc_unet_conv3d_fwd", ptr(X), cin, cin, ptr(W[c0:]), ptr(b[c0:]), n, d, h, w, 1, 0.1, ptr(out), n,
                  stream())
    conv(0, cout, Y)
    part = torch.empty((V, 64), dtype=torch.bfloat16, device="cuda")
    for c0 in (0, 8160, 16352, 24544, cout - 64):
        conv(c0, 64, part)
        assert torch.equal(Y[:, c0:c0 + 64], part), c0


def test_weight_gradient_of_a_large_volume(gpu, room):
    """2048 x 1024 x 1024 voxels, one channel on either side."""
    import torch
    from parsec_python_amd import _lib
    from parsec_python_amd.device import ptr, stream
    dims = (2048, 1024, 1024)
    print(f"weight gradient of {dims} voxels", flush=True)
    room(2 * 2 * 2 ** 31)
    X, Z = (torch.zeros(dims, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    ref = np.zeros((3, 3, 3))
    for q, (z, y, x) in enumerate([(0, 0, 0), (1023, 512, 3), (1024, 0, 0), (2047, 1023, 1023)]):
        Z[z, y, x] = q + 2.0
        for a in range(3):
            for b in range(3):
                for c in range(3):
                    p = (z + a - 1, y + b - 1, x + c - 1)
                    if all(0 <= p[i] < dims[i] for i in range(3)):
                        X[p] = 9.0 * a + 3.0 * b + c + 1.0
                        ref[a, b, c] += (q + 2.0) * (9.0 * a + 3.0 * b + c + 1.0)
    n = C.c_size_t()
    _lib.call("pc_unet_wgrad_workspace", 1, 1, C.byref(n))
    work = torch.empty(n.value, dtype=torch.uint8, device="cuda")
    dw = torch.empty((3, 3, 3), device="cuda")
    _lib.call("pc_unet_conv3d_wgrad", ptr(Z), 1, 1, ptr(X), 1, 1, *dims, ptr(dw), ptr(work), n.value, stream())
    assert np.array_equal(dw.cpu().numpy(), ref)


def test_activation_backward_of_a_large_volume(gpu, room):
    """2048^3 voxels of one channel: 2^24 chunks of 512."""
    import torch
    from parsec_python_amd import _lib
    from parsec_python_amd.device import ptr, stream
    n = 2048
    print("activation backward of 2048^3 voxels", flush=True)
    room(6 * n ** 3)
    dA = torch.zeros(n ** 3, device="cuda")
    dZ = torch.full((n ** 3,), 7.0, dtype=torch.bfloat16, device="cuda")
    at = torch.tensor([0, 511, 2 ** 32 - 1, 2 ** 32, n ** 3 - 1], device="cuda")
    dA[at] = torch.tensor([1.0, -2.0, 4.0, 8.0, 16.0], device="cuda")
    nb = C.c_size_t()
    _lib.call("pc_unet_act_bwd_workspace", 1, n ** 3, C.byref(nb))
    work = torch.empty(nb.value, dtype=torch.uint8, device="cuda")
    db = torch.empty(1, device="cuda")
    _lib.call("pc_unet_act_bwd", ptr(dA), 1, None, 1, 1, n, n, n, 0.1, ptr(dZ), 1, ptr(db), ptr(work), nb.value,
              stream())
    assert db.item() == 27.0
    assert dZ[at].tolist() == [1.0, -2.0, 4.0, 8.0, 16.0]
    assert int(torch.count_nonzero(dZ)) == 5
