"""The projector gather with 1, 2 and 4 wavefronts per atom (mean supports of up to
64 points, up to 256, more): supports of no, one and up to many rounds of 64
entries, short and whole last rounds, atom counts that leave wavefronts without one.

Tolerance: n products in FP64 err by at most (n + 2) 2^-53 of the sum of their
absolute values."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = {"small": [0, 1, 63, 64, 65, 30, 128, 129, 2, 33], "middle": [0, 1, 63, 64, 65, 127, 128, 129, 191, 192, 193, 320, 400, 385],
         "large": [0, 64, 256, 257, 300, 511, 512, 513, 767, 768, 769, 1100]}


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("kind", ["small", "middle", "large"])
@pytest.mark.parametrize("natoms,nvec", [(1, 5), (2, 4), (3, 1), (43, 7), (257, 13)])
def test_projector_gather_forms(gpu, natoms, nvec, kind, dtype):
    import torch
    from parsec_python_amd import _lib
    from parsec_python_amd.device import ptr, stream
    print(f"gather of {natoms} {kind} atoms, {nvec} vectors, {dtype}", flush=True)
    npts, ld = 3000, 3008
    rng = np.random.default_rng(natoms + nvec)
    sizes = [SIZES[kind][(natoms + a) % len(SIZES[kind])] for a in range(natoms)]
    aptr = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    pts = np.concatenate([np.sort(rng.choice(npts, n, replace=False)) for n in sizes]).astype(np.int32)
    uv, sc = rng.standard_normal((int(aptr[-1]), 3)), np.ones(natoms)
    handle = C.c_void_p()
    pi, pd = C.POINTER(C.c_int), C.POINTER(C.c_double)
    _lib.call("pc_proj_create", natoms, aptr.ctypes.data_as(pi), pts.ctypes.data_as(pi), uv.ctypes.data_as(pd),
              sc.ctypes.data_as(pd), npts, C.byref(handle))
    Y = torch.full((nvec, ld), float("nan"), dtype=torch.float64 if dtype == "f64" else torch.float32, device="cuda")
    Y[:, :npts] = torch.tensor(rng.standard_normal((nvec, npts)))
    cb = torch.full((natoms * nvec * 3 + 8,), 7.0, dtype=torch.float64, device="cuda")
    _lib.call(f"pc_proj_gather_{dtype}", handle, ptr(Y), ld, nvec, ptr(cb), stream())
    got = cb.cpu().numpy()
    assert np.all(got[natoms * nvec * 3:] == 7.0)
    got = got[:natoms * nvec * 3].reshape(natoms, nvec, 3)
    y = Y[:, :npts].double().cpu().numpy()
    for a in range(natoms):
        e = slice(aptr[a], aptr[a + 1])
        ref, top = y[:, pts[e]] @ uv[e], np.abs(y[:, pts[e]]) @ np.abs(uv[e])
        assert np.all(np.abs(got[a] - ref) <= 2 * (sizes[a] + 2) * 2.0 ** -53 * top), a
    _lib.call("pc_proj_destroy", handle)
