"""Timing cases of the SCF hot path and of the learned start's network.

Every case is one call (or the few calls that belong together) that a program
makes through the package's public classes or its C interface, on the systems
and settings of the tests, the sample inputs and the kernel benchmark:

* ``filter``   one Chebyshev filter of a block of vectors (``Eigensolver.ch_filter``:
               the fused stencil steps with the projector gather and scatter);
* ``chefsi``   one SCF iteration's eigensolve with its density: ``chefsi1`` (Lanczos
               bound, filter, Rayleigh-Ritz), the occupations and ``pc_density``;
* ``gemm``     the block products of one Rayleigh-Ritz step (``BlockLinalg.gram``
               twice and ``rotate``);
* ``dense``    the k x k Rayleigh-Ritz problem (``BlockLinalg.dense_rr``);
* ``hartree``  one Hartree solve (``HartreeSolver.solve``), plain or multigrid CG;
* ``layer``    one convolution layer of the density network: forward, or forward and
               backward as one training step runs it (``pc_unet_*``);
* ``scf``      a whole FP64 self-consistent solve (``run_scf``).
"""
import ctypes as C
import math

import numpy as np
import torch

from parsec_python_amd import _lib, ionic
from parsec_python_amd import kernel_bench as KB
from parsec_python_amd import molecules as M
from parsec_python_amd.device import ptr, stream
from parsec_python_amd.eigensolvers import Eigensolver
from parsec_python_amd.grid import DeviceGrid, make_grid, make_index_sphere_grid
from parsec_python_amd.hamiltonian import BlockLinalg, Hamiltonian, leading_dim
from parsec_python_amd.hartree import HartreeSolver
from parsec_python_amd.occupations import occupations
from parsec_python_amd.scf import SCFConfig, SCFProblem, run_scf

DT = {"f32": torch.float32, "f64": torch.float64}
SLOPE = 0.1


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # the sample input's filter step: 5 A cube, 0.2 A, default precision (the smallest SCF in use)
        dict(name="filter-h2o-f64", kind="filter", system="h2o", h_ang=0.2, radius_ang=5.0, nev=8, domain="cube",
             fd=4, deg=10, dtype="f64"),
        # a middle-sized molecule in mixed precision on the sphere
        dict(name="filter-c10h8-f32", kind="filter", system="c10h8", h_ang=0.2, radius_ang=9.0, nev=34,
             domain="sphere", fd=4, deg=10, dtype="f32"),
        # the benchmark's filter: the widest block of the mixed-precision solve
        dict(name="filter-si87h76-f32", kind="filter", system="si87h76", h_ang=0.25, radius_ang=13.0, nev=260,
             domain="sphere", fd=4, deg=10, dtype="f32"),
        # 12th order without projectors: the synthetic kernel workload
        dict(name="filter-fd12-f32", kind="filter", system="gauss", h_ang=0.2, radius_ang=0.0, nev=241, domain="index",
             n=128, rpts=60.0, fd=6, deg=16, dtype="f32"),
        # one FP64 SCF iteration of a middle-sized molecule (precision "fp64" is the default)
        dict(name="chefsi-c10h8-f64", kind="chefsi", system="c10h8", h_ang=0.2, radius_ang=9.0, nev=34,
             domain="sphere", fd=4, deg=10, dtype="f64"),
        # Rayleigh-Ritz products of the benchmark's block in FP32 and of its last, FP64 iteration
        dict(name="gemm-605808x275-f32", kind="gemm", n=605808, k=275, dtype="f32"),
        dict(name="gemm-605808x275-f64", kind="gemm", n=605808, k=275, dtype="f64"),
        # the dense problem of the benchmark's block
        dict(name="dense-275", kind="dense", k=275),
        # Hartree solves: plain CG on the sample's cube (default), multigrid on the benchmark's sphere
        dict(name="hartree-h2o", kind="hartree", n=52, h_ang=0.2, domain="cube", fd=4, prec="none", alias=True,
             maxit=200),
        dict(name="hartree-mg-si87h76", kind="hartree", n=106, h_ang=0.25, domain="sphere", fd=4, prec="mg",
             alias=False, maxit=1000),
        # a decoder layer of the network in training (64^3 volumes), forward and backward
        dict(name="layer-d1a-64-train", kind="layer", cin=48, cout=16, d=64, h=64, w=64, act=True, train=True),
        # the whole solve of the sample input at the default settings
        dict(name="scf-h2o", kind="scf", system="h2o", h_ang=0.2, radius_ang=5.0, nev=8, domain="cube"),
    ]


def _logint(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    """One more case of the same ranges."""
    kind = rng.choice(["filter", "filter", "filter", "chefsi", "gemm", "gemm", "dense", "hartree", "hartree", "layer",
                       "scf"])
    if kind == "filter":
        dtype = rng.choice(["f32", "f64"])
        if rng.random() < 0.2:
            n = rng.randrange(40, 129)
            return dict(kind=kind, system="gauss", h_ang=0.2, radius_ang=0.0, nev=_logint(rng, 1, 220), domain="index",
                        n=n, rpts=round(rng.uniform(0.3, 0.48) * n, 2), fd=rng.choice([1, 2, 3, 4, 6]),
                        deg=rng.randrange(4, 13), dtype=dtype)
        system, lo, hi, nev = rng.choice([("h2o", 3.5, 6.0, 8), ("alkane", 5.5, 8.0, 16), ("c10h8", 6.5, 9.2, 34),
                                          ("si17", 7.0, 9.0, 60)])
        return dict(kind=kind, system=system, h_ang=round(rng.uniform(0.2, 0.3), 4),
                    radius_ang=round(rng.uniform(lo, hi), 3), nev=nev + rng.randrange(0, 40),
                    domain=rng.choice(["cube", "sphere"]), fd=rng.choice([2, 3, 4, 4, 4, 6]), deg=rng.randrange(4, 13),
                    dtype=dtype)
    if kind == "chefsi":
        return dict(kind=kind, system=rng.choice(["h2o", "alkane"]), h_ang=round(rng.uniform(0.22, 0.3), 4),
                    radius_ang=round(rng.uniform(4.5, 7.0), 3), nev=rng.randrange(12, 60),
                    domain=rng.choice(["cube", "sphere"]), fd=rng.choice([3, 4, 4]), deg=rng.randrange(8, 12),
                    dtype="f64")
    if kind == "gemm":
        return dict(kind=kind, n=_logint(rng, 9000, 600000), k=_logint(rng, 17, 270), dtype=rng.choice(["f32", "f64"]))
    if kind == "dense":
        return dict(kind=kind, k=_logint(rng, 17, 320))
    if kind == "hartree":
        prec = rng.choice(["none", "mg"])
        return dict(kind=kind, n=_logint(rng, 24, 106), h_ang=round(rng.uniform(0.2, 0.3), 4),
                    domain=rng.choice(["cube", "sphere"]), fd=rng.choice([3, 4, 4, 6]), prec=prec,
                    alias=prec == "none" and rng.random() < 0.5, maxit=rng.choice([200, 1000]))
    if kind == "layer":
        cin, cout, level = rng.choice([(1, 16, 0), (16, 16, 0), (16, 32, 1), (32, 32, 1), (32, 48, 2), (48, 48, 2),
                                       (48, 64, 3), (64, 64, 3), (112, 48, 2), (80, 32, 1), (48, 16, 0), (16, 1, 0)])
        d, h, w = [8 * rng.randrange(4, 13) >> level for _ in range(3)]
        return dict(kind=kind, cin=cin, cout=cout, d=d, h=h, w=w, act=cout > 1, train=rng.random() < 0.6)
    return dict(kind="scf", system="h2o", h_ang=round(rng.uniform(0.22, 0.3), 4),
                radius_ang=round(rng.uniform(4.0, 5.0), 3), nev=rng.randrange(6, 14),
                domain=rng.choice(["cube", "sphere"]))


# ---------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(1000003 * int(seed) + 17)
    return g


def _geometry(case, seed):
    rng = np.random.default_rng(int(seed))
    s = case["system"]
    if s == "h2o":
        geo = M.h2o_sample()
    elif s == "c10h8":
        geo = M.naphthalene_sample()
    elif s == "alkane":
        geo = M.alkane(4, rng)
    else:
        geo = M.silicon_cluster(n_si=int(s[2:].split("h")[0]))
    # every seed has its own geometry, as every step of a relaxation has
    return [(e, np.asarray(x, dtype=float) + rng.uniform(-0.02, 0.02, np.shape(x))) for e, x in geo]


def _grid(case):
    if case["kind"] == "hartree":
        h = case["h_ang"] / M.A0_ANG
        return make_grid(case["n"], h, 0.5 * h * (case["n"] - 1), case["domain"])
    return make_index_sphere_grid(case["n"], 0.5 * (case["n"] - 1), case["rpts"], KB.SYNTH_H)


def _operator(case, seed):
    """(Hamiltonian with the superposed atoms' potential, projectors, atoms)."""
    dt = DT[case["dtype"]]
    if case["system"] == "gauss":
        g = _grid(case)
        pot = torch.from_numpy(KB.synthetic_potential(g, ball_pts=0.6 * case["rpts"], seed=int(seed))).to("cuda")
        return Hamiltonian(g, case["fd"], None, pot, dt), None, None
    atoms, dom, _ = M.prepare(_geometry(case, seed), h_ang=case["h_ang"], radius_ang=case["radius_ang"],
                              nev=case["nev"])
    atoms = ionic.normalize_atoms(atoms)
    g = make_grid(int(dom["nx"]), float(dom["h"]), float(dom["radius"]), case["domain"])
    proj = ionic.DeviceProjectors(g, atoms)
    H = Hamiltonian(g, case["fd"], proj, torch.zeros(g.npts, dtype=torch.float64, device="cuda"), dt)
    rho0, hpot0, ppot, _ = ionic.pseudo_diag(g, H.dgrid, atoms)
    vx = -torch.pow(3.0 / math.pi * rho0.clamp_min(0.0) / g.h ** 3, 1.0 / 3.0)
    H.set_potential(ppot + hpot0 + vx)
    return H, proj, atoms


def _weights(radius):
    f = math.factorial
    w = [0.0] + [2.0 * (-1) ** k * f(radius) ** 2 / (k * k * f(radius - k) * f(radius + k))
                 for k in range(1, radius + 1)]
    w[0] = -2.0 * sum(w)
    return w


def _bounds(h, fd):
    """(lam1, low, high) of a filter: the wanted levels of a molecule, and the grid's kinetic bound."""
    w = _weights(fd)
    kin = 1.5 / h ** 2 * (w[0] + 2.0 * sum(abs(c) for c in w[1:]))
    return -1.0, 0.45, 1.03 * kin + 1.0


def _charges(g, seed):
    """A neutral, smooth difference density: the Hartree right-hand side 4 pi (rho - rho0)."""
    rng = np.random.default_rng(int(seed))
    idx = torch.from_numpy(g.flat_index).to("cuda")
    ijk = torch.stack([idx % g.nx, (idx // g.nx) % g.ny, idx // (g.nx * g.ny)], 1).to(torch.float64)
    rhs = torch.zeros(g.npts, dtype=torch.float64, device="cuda")
    for _ in range(24):
        c = torch.tensor((rng.uniform(-0.3, 0.3, 3) + 0.5) * (g.nx - 1), device="cuda")
        s = rng.uniform(1.5, 5.0)
        rhs += rng.normal() / s ** 3 * torch.exp(-((ijk - c) ** 2).sum(1) / (2 * s * s))
    return 4.0 * math.pi * (rhs - rhs.mean())


def _layer_inputs(case, seed):
    g = _gen(seed)
    V, ci, co = case["d"] * case["h"] * case["w"], case["cin"], case["cout"]
    r = dict(device="cuda", generator=g)
    x = torch.randn(V, ci, **r)
    x = torch.where(x > 0, x, SLOPE * x) if ci > 1 else x.abs()
    x = x.to(torch.bfloat16)
    w = ((torch.rand(co, 27, ci, **r) * 2 - 1) * math.sqrt(6.0 / (27 * ci))).to(torch.bfloat16)
    b = 0.05 * torch.randn(co, **r)
    da = torch.randn(V, co, **r) / V
    return x, w, b, da


def _dense_inputs(case, seed):
    """S = A^T A and G = A^T L A of a filtered block: columns damped towards the band edge, close levels."""
    k, rng = case["k"], np.random.default_rng(int(seed))
    lam = np.sort(rng.uniform(-1.0, 0.3, k))
    for i in range(1, k):
        lam[i] = max(lam[i], lam[i - 1] + 2e-4)
    a = (np.eye(k) + 0.3 / math.sqrt(k) * rng.standard_normal((k, k))) * np.logspace(0, -2, k)[None, :]
    return a.T @ a, a.T @ (lam[:, None] * a), lam


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind in ("filter", "chefsi"):
        H, proj, atoms = _operator(case, seed)
        k = case["nev"] + 15
        s.update(H=H, proj=proj, k=k, es=Eigensolver(H, k, seed=int(seed)))
        if kind == "filter":
            s["x0"] = torch.randn((k, H.ld), dtype=H.dtype, device="cuda", generator=_gen(seed))
            s["bounds"] = _bounds(H.h, case["fd"])
        else:
            s["nelec"] = ionic.nelectrons(atoms)
            s["W"], s["lam"] = s["es"].first_filt(k, 10)
            s["occ2"] = torch.zeros(k, dtype=torch.float64, device="cuda")
            s["rho"] = torch.empty(H.n, dtype=torch.float64, device="cuda")
    elif kind == "gemm":
        n, k, dt = case["n"], case["k"], DT[case["dtype"]]
        g = _gen(seed)
        s["la"] = BlockLinalg(n, k)
        s["Y"] = torch.randn((k, leading_dim(n)), dtype=dt, device="cuda", generator=g)
        s["HY"] = torch.randn((k, leading_dim(n)), dtype=dt, device="cuda", generator=g)
        s["T"] = torch.randn(k * k, dtype=torch.float64, device="cuda", generator=g) / math.sqrt(k)
        s["Z"] = torch.empty_like(s["Y"])
        s["S"], s["G"] = (torch.empty(k * k, dtype=torch.float64, device="cuda") for _ in range(2))
    elif kind == "dense":
        S, G, _ = _dense_inputs(case, seed)
        k = case["k"]
        s["la"] = BlockLinalg(4096, k)
        s["S0"], s["G0"] = (torch.from_numpy(m).to("cuda").reshape(-1) for m in (S, G))
        s["S"], s["G"] = torch.empty_like(s["S0"]), torch.empty_like(s["G0"])
    elif kind == "hartree":
        g = _grid(case)
        s["dg"] = DeviceGrid(g, case["fd"])
        s["hs"] = HartreeSolver(s["dg"], g.h, reference_aliasing=case["alias"], prec=case["prec"])
        s["rhs"] = _charges(g, seed)
        s["x"] = torch.empty_like(s["rhs"])
    elif kind == "layer":
        V, ci, co = case["d"] * case["h"] * case["w"], case["cin"], case["cout"]
        s["x"], s["w"], s["b"], s["da"] = _layer_inputs(case, seed)
        e = dict(device="cuda")
        s["y"] = torch.empty(V, co, dtype=torch.bfloat16 if case["act"] else torch.float32, **e)
        if case["train"]:
            s["dz"] = torch.empty(V, co, dtype=torch.bfloat16, **e)
            s["dx"] = torch.empty(V, ci, dtype=torch.float32, **e)
            s["dw"] = torch.empty(co, 27, ci, dtype=torch.float32, **e)
            s["db"] = torch.empty(co, dtype=torch.float32, **e)
            s["wt"] = torch.empty_like(s["w"])
            a, b = C.c_size_t(), C.c_size_t()
            _lib.call("pc_unet_wgrad_workspace", co, ci, C.byref(a))
            _lib.call("pc_unet_act_bwd_workspace", co, V, C.byref(b))
            s["work"] = torch.empty(max(a.value, b.value), dtype=torch.uint8, **e)
    else:
        atoms, dom, nev = M.prepare(_geometry(case, seed), h_ang=case["h_ang"], radius_ang=case["radius_ang"],
                                    nev=case["nev"])
        s["prob"] = SCFProblem(atoms, dom, nev, SCFConfig(domain=case["domain"], seed=int(seed)))
    return s


# ---------------------------------------------------------------- one pass
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "filter":
        es, k = s["es"], s["k"]
        es.bufs[0].copy_(s["x0"])
        y = es.ch_filter(es.bufs[0], k, case["deg"], *s["bounds"])
        return y[:k, :s["H"].n]
    if kind == "chefsi":
        es, k, nev, H = s["es"], s["k"], case["nev"], s["H"]
        W, lam = es.chefsi1(s["W"], s["lam"], case["deg"], nev)
        s["W"], s["lam"] = W, lam
        _, occ = occupations(lam[:nev], 500.0, s["nelec"], 1e-6)
        s["occ2"][:nev].copy_(torch.from_numpy(2.0 * occ))
        _lib.call("pc_density_f64", ptr(W), W.shape[1], H.n, nev, ptr(s["occ2"]), ptr(s["rho"]), stream())
        return {"ritz": lam[:nev], "rho": s["rho"]}
    if kind == "gemm":
        la, k, n = s["la"], case["k"], case["n"]
        la.gram(s["Y"], s["Y"], k, k, s["S"], sym=True)
        la.gram(s["Y"], s["HY"], k, k, s["G"], sym=False)
        la.rotate(s["Y"], s["T"], k, k, s["Z"])
        return {"S": s["S"].view(k, k), "G": s["G"].view(k, k), "Z": s["Z"][:, :n]}
    if kind == "dense":
        s["S"].copy_(s["S0"])
        s["G"].copy_(s["G0"])
        T, lam = s["la"].dense_rr(s["S"], s["G"], case["k"])
        return {"T": T, "ritz": lam}
    if kind == "hartree":
        s["x"].zero_()
        s["hs"].solve(s["rhs"], s["x"], case["maxit"], 1e-5)
        return s["x"]
    if kind == "layer":
        return _layer(s)
    r = run_scf(s["prob"])
    return {"energy_ry": r.energies["total_ry"], "ritz": r.eigenvalues[:case["nev"]], "rho": r.rho, "hpot": r.hpot}


def _layer(s):
    case = s["case"]
    d, h, w, ci, co, st = case["d"], case["h"], case["w"], case["cin"], case["cout"], stream()
    _lib.call("pc_unet_conv3d_fwd", ptr(s["x"]), ci, ci, ptr(s["w"]), ptr(s["b"]), co, d, h, w, 1 if case["act"] else 0,
              SLOPE, ptr(s["y"]), co, st)
    if not case["train"]:
        return {"y": s["y"]}
    work = s["work"]
    _lib.call("pc_unet_act_bwd", ptr(s["da"]), co, ptr(s["y"]) if case["act"] else None, co if case["act"] else 0, co,
              d, h, w, SLOPE, ptr(s["dz"]), co, ptr(s["db"]), ptr(work), work.numel(), st)
    _lib.call("pc_unet_conv3d_wgrad", ptr(s["dz"]), co, co, ptr(s["x"]), ci, ci, d, h, w, ptr(s["dw"]), ptr(work),
              work.numel(), st)
    out = {"y": s["y"], "dw": s["dw"], "db": s["db"]}
    if ci > 1 and co % 16 == 0 or co == 1 and ci > 1:      # the first layer's input needs no gradient
        _lib.call("pc_unet_conv3d_wflip", ptr(s["w"]), co, ci, ptr(s["wt"]), st)
        _lib.call("pc_unet_conv3d_fwd", ptr(s["dz"]), co, co, ptr(s["wt"]), None, ci, d, h, w, 2, SLOPE, ptr(s["dx"]),
                  ci, st)
        out["dx"] = s["dx"]
    return out


# ---------------------------------------------------------------- what a pass cannot do without
def _size(case):
    """(domain points, atoms' projector entries) of a case, from its geometry."""
    if case["system"] == "gauss":
        return 4.18879 * case["rpts"] ** 3, 0.0
    n = 2 * ((int(2 * case["radius_ang"] / case["h_ang"]) + 2) // 2)
    pts = n ** 3 * (1.0 if case["domain"] == "cube" else 0.5236)
    atoms = {"h2o": 3, "c10h8": 18, "alkane": 14, "si17": 53, "si87h76": 163}[case["system"]]
    return pts, atoms * 4.18879 * (1.2 / case["h_ang"]) ** 3


def _filter_work(pts, ents, k, fd, deg, size):
    return {"bytes": size * (pts * (k * (3 * deg - 1) + 1) + 3.0 * deg * k * ents),
            "flops": deg * k * (pts * (7.0 * fd + 6) + 12.0 * ents)}


def work(case):
    kind = case["kind"]
    if kind in ("filter", "chefsi", "scf"):
        pts, ents = _size(case)
        k, size = case["nev"] + 15, 4 if case.get("dtype") == "f32" else 8
        w = _filter_work(pts, ents, k, case.get("fd", 4), case.get("deg", 10), size)
        if kind == "filter":
            return w
        # one H Y, two symmetric products, the rotation and the density
        rr = {"bytes": size * pts * k * 8.0, "flops": 4.0 * pts * k * k + pts * k * 36.0}
        passes = 1 if kind == "chefsi" else 17      # an SCF of the sample takes about 17
        cg = 0.0 if kind == "chefsi" else 11 * 90 * pts
        return {"bytes": passes * (w["bytes"] + rr["bytes"]) + 56.0 * cg,
                "flops": passes * (w["flops"] + rr["flops"]) + 40.0 * cg}
    if kind == "gemm":
        n, k, size = case["n"], case["k"], 4 if case["dtype"] == "f32" else 8
        return {"bytes": 3.0 * n * k * size + 24.0 * k * k, "flops": 5.0 * n * k * k}
    if kind == "dense":
        k = case["k"]
        return {"bytes": 32.0 * k * k, "flops": (1.0 / 3 + 2 + 4.0 / 3 + 3 + 2) * k ** 3}
    if kind == "hartree":
        pts = case["n"] ** 3 * (1.0 if case["domain"] == "cube" else 0.5236)
        its = 26 if case["prec"] == "mg" else min(case["maxit"], 2.4 * case["n"])
        per = (88.0, 7.0 * case["fd"] + 12) if case["prec"] == "none" else (150.0, 3 * 7.0 * case["fd"] + 40)
        return {"bytes": its * pts * per[0], "flops": its * pts * per[1]}
    V, ci, co = case["d"] * case["h"] * case["w"], case["cin"], case["cout"]
    f = 2.0 * 27 * V * ci * co
    if not case["train"]:
        return {"bytes": 2.0 * V * (ci + co) + 54.0 * ci * co, "flops": f}
    return {"bytes": V * (8.0 * ci + 8.0 * co) + 270.0 * ci * co, "flops": 3 * f}


# ---------------------------------------------------------------- the same in 64 bits
def _stencil64(v, w, R):
    """-lap of zero-bounded volumes (..., z, y, x) with 1D weights w, in units of h^-2."""
    p = torch.nn.functional.pad(v, (R,) * 6)
    nz, ny, nx = v.shape[-3:]
    out = 3.0 * w[0] * v
    for d in range(1, R + 1):
        for s in (-d, d):
            out += w[d] * p[..., R:R + nz, R:R + ny, R + s:R + s + nx]
            out += w[d] * p[..., R:R + nz, R + s:R + s + ny, R:R + nx]
            out += w[d] * p[..., R + s:R + s + nz, R:R + ny, R:R + nx]
    return out


def _exact_filter(case, seed):
    H, proj, _ = _operator(case, seed)
    k, R, n, g = case["nev"] + 15, case["fd"], H.n, H.grid
    x0 = torch.randn((k, H.ld), dtype=H.dtype, device="cuda", generator=_gen(seed))[:, :n]
    w, idx = _weights(R), torch.from_numpy(g.flat_index).to("cuda")
    shape = (g.nz, g.ny, g.nx)
    U = None
    if proj is not None and proj.natoms:
        aptr, pt, u, sc = proj.tables
        atom = torch.from_numpy(np.repeat(np.arange(proj.natoms), np.diff(aptr)).astype(np.int64)).to("cuda")
        U = (atom, torch.from_numpy(pt.astype(np.int64)).to("cuda"), torch.from_numpy(u).to("cuda"),
             torch.from_numpy(sc).to("cuda"))
    lam1, low, high = _bounds(H.h, R)
    e, c = (high - low) / 2, (high + low) / 2
    out = torch.empty((k, n), dtype=torch.float64, device="cuda")

    def apply(y):
        vol = torch.zeros((y.shape[0], g.nx * g.ny * g.nz), dtype=torch.float64, device="cuda")
        vol[:, idx] = y
        r = 0.5 / H.h ** 2 * _stencil64(vol.view(-1, *shape), w, R).reshape(y.shape[0], -1)[:, idx] + H.pot * y
        if U is not None:
            atom, pt, u, sc = U
            yp = y[:, pt]
            for m in range(3):
                co = torch.zeros((y.shape[0], len(sc)), dtype=torch.float64, device="cuda")
                co.index_add_(1, atom, yp * u[:, m])
                r.index_add_(1, pt, (co * sc)[:, atom] * u[:, m])
        return r

    for b in range(0, k, 16):
        x = x0[b:b + 16].to(torch.float64)
        sigma1 = sigma = e / (lam1 - c)
        y = (apply(x) - c * x) * (sigma1 / e)
        for _ in range(2, case["deg"] + 1):
            new = 1.0 / (2.0 / sigma1 - sigma)
            x, y = y, (apply(y) - c * y) * (2.0 * new / e) - sigma * new * x
            sigma = new
        out[b:b + 16] = y
    return out


def _exact_hartree(case, seed):
    g = _grid(case)
    b, w, R = _charges(g, seed), _weights(case["fd"]), case["fd"]
    idx = torch.from_numpy(g.flat_index).to("cuda")
    vol = torch.zeros(g.nx * g.ny * g.nz, dtype=torch.float64, device="cuda")

    def apply(v):
        vol[idx] = v
        return _stencil64(vol.view(g.nz, g.ny, g.nx), w, R).reshape(-1)[idx] / g.h ** 2

    x, r = torch.zeros_like(b), b.clone()
    p, rr = r.clone(), torch.dot(r, r)
    stop = float(rr) * 1e-26
    for it in range(4000):
        ap = apply(p)
        alpha = rr / torch.dot(p, ap)
        x += alpha * p
        r -= alpha * ap
        new = torch.dot(r, r)
        if it % 20 == 0 and float(new) < stop:
            break
        p = r + (new / rr) * p
        rr = new
    return x


def _exact_layer(case, seed):
    x, w, b, da = _layer_inputs(case, seed)
    d, h, ww, ci, co = case["d"], case["h"], case["w"], case["cin"], case["cout"]
    V = d * h * ww
    x, w, b, da = (t.to(torch.float64) for t in (x, w, b, da))

    def shifted(t, k, c):
        p = torch.nn.functional.pad(t.view(d, h, ww, c), (0, 0, 1, 1, 1, 1, 1, 1))
        return p[k // 9:k // 9 + d, k // 3 % 3:k // 3 % 3 + h, k % 3:k % 3 + ww].reshape(V, c)

    y = b.expand(V, co).clone()
    for k in range(27):
        y += shifted(x, k, ci) @ w[:, k].t().contiguous()
    if case["act"]:
        y = torch.where(y > 0, y, SLOPE * y)
    if not case["train"]:
        return {"y": y}
    dz = torch.where(y > 0, da, SLOPE * da) if case["act"] else da
    dw = torch.stack([dz.t().contiguous() @ shifted(x, k, ci) for k in range(27)], 1)
    out = {"y": y, "dw": dw, "db": dz.sum(0)}
    if ci > 1:
        dx = torch.zeros(V, ci, dtype=torch.float64, device="cuda")
        for k in range(27):
            dx += shifted(dz, 26 - k, co) @ w[:, k]
        out["dx"] = dx
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "filter":
        return _exact_filter(case, seed)
    if kind == "gemm":
        n, k, g = case["n"], case["k"], _gen(seed)
        dt = DT[case["dtype"]]
        Y = torch.randn((k, leading_dim(n)), dtype=dt, device="cuda", generator=g)[:, :n].to(torch.float64)
        HY = torch.randn((k, leading_dim(n)), dtype=dt, device="cuda", generator=g)[:, :n].to(torch.float64)
        T = torch.randn(k * k, dtype=torch.float64, device="cuda", generator=g).view(k, k) / math.sqrt(k)
        # column-major results: row j of the returned arrays is column j
        return {"S": Y @ Y.t(), "G": HY @ Y.t(), "Z": T @ Y}
    if kind == "dense":
        return {"T": None, "ritz": _dense_inputs(case, seed)[2]}
    if kind == "hartree":
        return _exact_hartree(case, seed)
    if kind == "layer":
        return _exact_layer(case, seed)
    return None
