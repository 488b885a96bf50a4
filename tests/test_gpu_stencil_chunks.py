"""The stencil's z-chunks: the number of vectors decides how many chunks a grid's
planes are cut into, at multiples of the planes that the march runs as one block
(6, 8, 12, 12 and 16 for radius 1, 2, 3, 4 and 6).

Every point's sum has one order whatever the cut, so a vector's result has the same
bits alone (many short chunks) and among many (few long ones)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BLOCK = {1: 6, 2: 8, 3: 12, 4: 12, 6: 16}


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("kind", ["cube", "sphere"])
@pytest.mark.parametrize("planes", [lambda b: b - 1, lambda b: b, lambda b: b + 1, lambda b: 5 * b + 3, lambda b: 9 * b - 1],
                         ids=["block-1", "block", "block+1", "5block+3", "9block-1"])
@pytest.mark.parametrize("radius", [1, 2, 3, 4, 6])
def test_stencil_bits_do_not_depend_on_the_number_of_vectors(gpu, radius, planes, kind, dtype):
    import torch
    from parsec_python_amd import _lib
    from parsec_python_amd.device import ptr, stream
    from parsec_python_amd.grid import DeviceGrid, Grid
    from parsec_python_amd.hamiltonian import leading_dim
    nx, ny, nz = 21, 13, planes(BLOCK[radius])
    print(f"stencil chunks r={radius} nz={nz} {kind} {dtype}", flush=True)
    mask = np.ones((nz, ny, nx), bool)
    if kind == "sphere":   # windows of different lengths
        k, j, i = np.meshgrid(*((np.arange(m) - (m - 1) / 2) / (m / 2) for m in (nz, ny, nx)), indexing="ij")
        mask = i * i + j * j + k * k <= 1
    dg = DeviceGrid(Grid(nx=nx, ny=ny, nz=nz, h=0.4, rad=4.0, mask=mask.reshape(-1), kind="cube"), radius)
    n, ld, nvec = int(mask.sum()), leading_dim(int(mask.sum())), 1500
    tdt = torch.float64 if dtype == "f64" else torch.float32
    Y = torch.full((nvec, ld), float("nan"), dtype=tdt, device="cuda")
    Y[:, :n] = torch.randn((nvec, n), dtype=tdt, device="cuda")
    X0 = torch.randn((nvec, ld), dtype=tdt, device="cuda")
    V = torch.randn(n, dtype=tdt, device="cuda")

    def step(first, count):
        X = X0[first:first + count].clone()
        _lib.call(f"pc_stencil_{dtype}", dg.handle, ptr(Y[first:]), ptr(X), ptr(X), ptr(V), count, ld, 0.5, 0.7, -0.3, -1.1,
                  None, stream())
        return X
    alone = {v: step(v, 1)[0] for v in (0, 7, 1499)}
    for count in (40, 200, nvec):
        got = step(0, count)
        assert not bool(torch.isnan(got[:, :n]).any())
        assert torch.equal(got[:, n:], X0[:count, n:])
        for v, one in alone.items():
            if v < count:
                assert torch.equal(got[v], one)
    dg.close()


@pytest.mark.parametrize("radius", [3, 4])
def test_stencil_time_per_plane_of_planes_beyond_whole_blocks(gpu, radius):
    """23 vectors, FP32: 64 planes of 64 x 64 points run 72, an eighth more per plane
    than 60, which are five whole blocks; with the spread of two timings at most a
    fifth more (cut into five chunks of 13 planes they ran 24 each: 1.4 times)."""
    import torch
    from parsec_python_amd import _lib
    from parsec_python_amd.device import ptr, stream
    from parsec_python_amd.grid import DeviceGrid, Grid
    from parsec_python_amd.hamiltonian import leading_dim
    steps, times = [], [[], []]
    for nz in (60, 64):
        print(f"stencil time 64 x 64 x {nz} r={radius}", flush=True)
        g = Grid(nx=64, ny=64, nz=nz, h=0.4, rad=12.0, mask=np.ones(64 * 64 * nz, bool), kind="cube")
        dg, ld = DeviceGrid(g, radius), leading_dim(g.npts)
        Y, X = (torch.zeros((23, ld), device="cuda") for _ in range(2))
        V = torch.zeros(g.npts, device="cuda")

        def step(dg=dg, ld=ld, Y=Y, X=X, V=V):
            _lib.call("pc_stencil_f32", dg.handle, ptr(Y), ptr(X), ptr(X), ptr(V), 23, ld, 0.5, 1.0, 0.0, 0.5, None, stream())
        steps.append((step, nz, dg))
    for _ in range(9):
        for i, (step, nz, _dg) in enumerate(steps):
            e0, e1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            step()
            e0.record()
            for _ in range(20):
                step()
            e1.record()
            torch.cuda.synchronize()
            times[i].append(e0.elapsed_time(e1) / 20 / nz)
    whole, beyond = (sorted(t)[4] for t in times)
    print(f"{1e3 * whole:.3f} and {1e3 * beyond:.3f} us per plane", flush=True)
    assert beyond <= 1.2 * whole
    for _step, _nz, dg in steps:
        dg.close()
