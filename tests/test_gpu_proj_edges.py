"""Edges of the projector gather and scatter: supports of one point, of just under
and over a round of 64 entries, of the 768 that the wavefronts take at once and
more, an empty support, vector counts around the 4 of a workgroup.

Against a float64 sum.  The gather adds n products in FP64: n u times the sum of
their absolute values; the scatter adds at most 3 natoms products and rounds once
to the storage type."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SUPPORTS = [[1], [63, 64, 65], [255, 256, 257, 0, 3], [767, 768, 769, 770], [1537, 2, 640]]


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("sizes", SUPPORTS)
def test_projector_edges(gpu, sizes, dtype):
    import torch
    from parsec_python_amd import _lib
    from parsec_python_amd.device import ptr, stream
    npts, ld = 2000, 2048
    tdt, u = (torch.float64, 2.0 ** -53) if dtype == "f64" else (torch.float32, 2.0 ** -24)
    rng = np.random.default_rng(sum(sizes))
    na, aptr = len(sizes), np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    pts = np.concatenate([np.sort(rng.choice(npts, n, replace=False)) for n in sizes]).astype(np.int32)
    uv = rng.standard_normal((int(aptr[-1]), 3))
    sc = rng.uniform(0.5, 2.0, na)
    handle = C.c_void_p()
    pi, pd = C.POINTER(C.c_int), C.POINTER(C.c_double)
    _lib.call("pc_proj_create", na, aptr.ctypes.data_as(pi), pts.ctypes.data_as(pi), uv.ctypes.data_as(pd),
              sc.ctypes.data_as(pd), npts, C.byref(handle))
    for nvec in (1, 3, 4, 5, 17):
        print(f"projector edge case {sizes} {dtype} nvec={nvec}", flush=True)
        Y = torch.full((nvec, ld), float("nan"), dtype=tdt, device="cuda")
        Y[:, :npts] = torch.tensor(rng.standard_normal((nvec, npts)), dtype=tdt)
        O = Y.clone()
        cb = torch.full((na * nvec * 3 + 8,), float("nan"), dtype=torch.float64, device="cuda")
        _lib.call(f"pc_proj_gather_{dtype}", handle, ptr(Y), ld, nvec, ptr(cb), stream())
        y = Y[:, :npts].double().cpu().numpy()
        got = cb.cpu().numpy()
        assert np.isnan(got[na * nvec * 3:]).all()
        got = got[:na * nvec * 3].reshape(na, nvec, 3)
        out, mag = y.copy(), np.abs(y)
        for a in range(na):
            e = slice(aptr[a], aptr[a + 1])
            ref, top = y[:, pts[e]] @ uv[e], np.abs(y[:, pts[e]]) @ np.abs(uv[e])
            assert np.all(np.abs(got[a] - ref) <= 2 * (sizes[a] + 2) * 2.0 ** -53 * top)
            np.add.at(out.T, pts[e], 0.3 * sc[a] * (uv[e] @ got[a].T))
            np.add.at(mag.T, pts[e], 0.3 * sc[a] * (np.abs(uv[e]) @ np.abs(got[a].T)))
        _lib.call(f"pc_proj_scatter_{dtype}", handle, ptr(cb), ptr(O), ld, nvec, 0.3, stream())
        res = O.double().cpu().numpy()
        assert np.all(np.abs(res[:, :npts] - out) <= (2 * u + 12 * (na + 1) * 2.0 ** -53) * mag)
        assert np.isnan(res[:, npts:]).all()
    _lib.call("pc_proj_destroy", handle)
