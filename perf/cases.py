"""Performance cases of the demag convolution and the LLG integrators, through the package's public
entry points (boris2_amd.api): what a program of this library has it do, from the smallest film to
the largest mesh.

A case is a dict with a "kind" and its sizes:

  conv    Demag.convolute of one mesh: open or periodic, field set or added, with or without the energy
  avg     Demag.convolute_averaged with both outputs (the two-sublattice convolution)
  layers  MultiLayerDemag.convolute of a stack of 2D layers
  llg     `steps` integration steps of one mesh (FMSolver): TEuler, RK4, RKDP54, optionally with the
          demag evaluation speedup
  stack   `steps` RK4 steps of a layer stack (LayerStackSolver), its layers grouped into 3D meshes or not
  batch   `steps` RK4 steps of many films of uneven sizes in one batch (BatchSolver)
  adj     loss and gradients of an RK4 rollout (RK4Adjoint forward and backward)

A pass of an integrating case goes on from the state that the pass before it left, as a simulation
does.  exact() gives the first pass on new inputs in FP64 from the formulas alone: Newell's prism
tensor near, the dipole averaged over both cells far, torch FFTs, and the LLG equation.
"""
import math
import random

import numpy as np
import torch

from boris2_amd import api

MU0 = 1.256637061435916e-6
GAMMA = 2.212761569e5
DEM, EXC, ANI, ZEE = api.BM_MOD_DEMAG, api.BM_MOD_EXCHANGE, api.BM_MOD_ANIS_UNI, api.BM_MOD_ZEEMAN
METHODS = {"TEULER": api.BM_EVAL_TEULER, "RK4": api.BM_EVAL_RK4, "RKDP54": api.BM_EVAL_RKDP54}
STAGES = {"TEULER": 2, "RK4": 4, "RKDP54": 6}
# fixed steps, and the largest step that the adaptive method may take: small enough for the short
# exchange waves of the inputs, so that it takes that step throughout
DT = {"TEULER": 5e-14, "RK4": 2.5e-13, "RKDP54": 1.5e-13}
FILM = (64, 96, 128, 192, 256)          # film sides of a batch


def _conv(name, nx, ny, nz, pbc=0, add=False, energy=False):
    return {"name": name, "kind": "conv", "nx": nx, "ny": ny, "nz": nz, "pbc": pbc, "add": add, "energy": energy}


def _llg(name, method, nx, ny, nz, steps, anis=False, speedup=0):
    return {"name": name, "kind": "llg", "method": method, "nx": nx, "ny": ny, "nz": nz, "steps": steps, "anis": anis, "speedup": speedup}


def listed():
    return [
        # the smallest call: the field of a small film, where launches and latency count
        _conv("conv 64x64x1", 64, 64, 1),
        # a mesh whose sides have no transform length of their own, added to other fields, with its energy
        _conv("conv 100x75x5 add energy", 100, 75, 5, add=True, energy=True),
        # a periodic strip: images along x and y
        _conv("conv pbc 256x192x4", 256, 192, 4, pbc=5),
        # one evaluation of a large film
        _conv("conv 1024x1024x1", 1024, 1024, 1),
        # a small film integrated at fixed step: the common desktop run (vortex, standard problems)
        _llg("llg RK4 128x64x1", "RK4", 128, 64, 1, 10),
        # an ordinary 3D film with the default adaptive method
        _llg("llg RKDP54 256x256x8", "RKDP54", 256, 256, 8, 3, anis=True),
        # the largest workload: the headline mesh of bench.py
        _llg("llg RKDP54 512x512x32", "RKDP54", 512, 512, 32, 2, anis=True),
        # an ordinary mesh with the demag evaluation speedup (quadratic extrapolation)
        _llg("llg speedup 256x256x16", "RKDP54", 256, 256, 16, 4, anis=True, speedup=3),
        # the multilayered demag of three 2D layers, one stack of bench.py's
        {"name": "stack RK4 3x256x256", "kind": "stack", "nx": 256, "ny": 256, "planes": "1,1,1", "steps": 3},
        # three 3D meshes as ten planes: the multilayered demag of the trilayer example
        {"name": "stack RK4 10x128x64", "kind": "stack", "nx": 128, "ny": 64, "planes": "4,2,4", "steps": 3},
        # films of uneven sizes in one batch: a parameter sweep
        {"name": "batch RK4 32 films", "kind": "batch", "films": 32, "sizes": 64, "steps": 3},
        # gradients of a film's rollout in its Ms map and its field pulse
        {"name": "adjoint 128x128x4", "kind": "adj", "nx": 128, "ny": 128, "nz": 4, "steps": 8, "every": 4},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    """One more case: sizes over the whole range, odd ones among them, at most 4 M cells."""
    kind = rng.choice(["conv", "conv", "conv", "avg", "layers", "llg", "llg", "llg", "stack", "batch", "adj"])

    def mesh(cap):
        while True:
            nx, ny = _log(rng, 20, 1100), _log(rng, 20, 1100)
            nz = rng.choice([1, 1, 2, 3, 4, 6, 8, 12, 16, 24])
            if rng.random() < 0.5:
                p2 = [32, 48, 64, 96, 128, 192, 256, 384, 512, 768, 1024]
                nx, ny = rng.choice(p2), rng.choice(p2)
            if nx * ny * nz <= cap:
                return nx, ny, nz

    def plain():
        p2 = [32, 48, 64, 96, 128, 192, 256, 384, 512]
        return rng.choice(p2), rng.choice(p2)

    if kind == "conv":
        if rng.random() < 0.25:
            nx, ny = plain()
            c = _conv("", nx, ny, rng.choice([1, 2, 4, 8]), pbc=rng.choice([2, 3, 5]), add=rng.random() < 0.5)
        else:
            c = _conv("", *mesh(4_000_000), add=rng.random() < 0.5, energy=rng.random() < 0.5)
    elif kind == "avg":
        nx, ny, nz = mesh(1_000_000)
        c = {"kind": "avg", "nx": nx, "ny": ny, "nz": nz}
    elif kind == "layers":
        nx, ny = plain()
        c = {"kind": "layers", "nx": nx, "ny": ny, "layers": rng.choice([2, 3, 4, 5, 8, 12])}
    elif kind == "llg":
        method = rng.choice(["TEULER", "RK4", "RKDP54", "RKDP54"])
        nx, ny, nz = mesh(2_000_000)
        c = _llg("", method, nx, ny, nz, rng.choice([2, 3, 5]), anis=rng.random() < 0.5, speedup=rng.choice([0, 0, 0, 2, 3]) if method != "TEULER" else 0)
    elif kind == "stack":
        nx, ny = plain()
        c = {"kind": "stack", "nx": nx, "ny": ny, "planes": rng.choice(["1,1", "1,1,1", "1,1,1,1,1", "2,2", "3,2,3", "4,2,4"]), "steps": rng.choice([2, 3, 4])}
    elif kind == "batch":
        c = {"kind": "batch", "films": _log(rng, 4, 40), "sizes": rng.randrange(1 << 20), "steps": rng.choice([2, 3])}
    else:
        nx, ny = rng.choice([32, 48, 64, 96, 100, 128, 192]), rng.choice([32, 48, 64, 75, 96, 128, 192])
        c = {"kind": "adj", "nx": nx, "ny": ny, "nz": rng.choice([1, 2, 4, 6]), "steps": rng.choice([4, 6, 8]), "every": rng.choice([2, 3, 4])}
    c.pop("name", None)
    return c


# ------------------------------------------------------------------------------------------
# Inputs

def _rand(seed, salt):
    return np.random.default_rng([int(seed), int(salt)])


def _texture(n, seed, salt=0):
    """A smooth unit vector field on n = (nx, ny, nz): waves of up to three periods per in-plane
    axis, varying a little through the thickness, with 1 % of uncorrelated noise; (cells, 3) FP32
    on the GPU."""
    nx, ny, nz = n
    r = _rand(seed, 1000 + salt)
    g = torch.Generator(device="cuda").manual_seed(int(r.integers(1 << 40)))
    basis = []
    for m in (nx, ny):
        x = (torch.arange(m, dtype=torch.float64, device="cuda") + 0.5) / m
        basis.append(torch.stack([f(2 * math.pi * k * x) for k in range(4) for f in (torch.cos, torch.sin)]))
    w = np.array([1.0 / (1 + a // 2 + b // 2) for a in range(8) for b in range(8)]).reshape(8, 8)
    z = (torch.arange(nz, dtype=torch.float64, device="cuda") + 0.5) / nz
    f = torch.empty((nz, ny, nx, 3), dtype=torch.float32, device="cuda")
    for c in range(3):
        a, b = (torch.tensor(r.normal(size=(8, 8)) * w, device="cuda") for _ in range(2))
        p, q = basis[1].T @ a @ basis[0], basis[1].T @ b @ basis[0]
        f[..., c] = (p[None] + 0.2 * (z - 0.5)[:, None, None] * q[None]).float()
    f += 0.01 * torch.randn(f.shape, generator=g, device="cuda")
    f /= f.norm(dim=-1, keepdim=True)
    return f.reshape(-1, 3)


def _cell(c):
    return (4e-9, 4e-9, 4e-9)


def _material(c, seed):
    r = _rand(seed, 7)
    base = dict(Ms=float(r.uniform(7e5, 1e6)), A=1.3e-11, alpha=float(r.uniform(0.02, 0.2)), ea=(0.0, 0.0, 1.0),
                Ha=tuple(float(v) for v in r.normal(0.0, 2e4, 3)), modules=DEM | EXC | ZEE)
    if c.get("anis"):
        base.update(K1=1e5, modules=DEM | EXC | ANI | ZEE)
    return base


def _n(c):
    return c["nx"], c["ny"], c["nz"]


def _pbc(c):
    return (c["pbc"], c["pbc"], 0) if c.get("pbc") else (0, 0, 0)


def _stack(c):
    """Thickness, bottom height and mesh of every plane: meshes of touching 4 nm planes, 4 nm apart."""
    meshes, z = [], 0.0
    for p in (int(v) for v in c["planes"].split(",")):
        meshes.append((p, 4e-9, z))
        z += (p + 1) * 4e-9
    hz, z0, grp = [], [], []
    for m, (p, h, zb) in enumerate(meshes):
        for k in range(p):
            hz.append(h); z0.append(zb + k * h); grp.append(m)
    return np.array(hz), np.array(z0), np.array(grp, dtype=np.int32)


def _films(c):
    r = np.random.default_rng(c["sizes"])
    return [(int(r.choice(FILM)), int(r.choice(FILM)), int(r.choice([1, 2, 4, 8]))) for _ in range(c["films"])]


def _film_materials(c, seed):
    r = _rand(seed, 9)
    return [dict(Ms=float(r.uniform(4e5, 1.2e6)), A=1.3e-11, alpha=float(r.uniform(0.01, 0.5)), modules=DEM | EXC) for _ in range(c["films"])]


def _adj_inputs(c, seed):
    n = _n(c)
    ms = (5e5 + 6e5 * (0.5 + 0.5 * _texture(n, seed, 21)[:, 0])).contiguous()
    r = _rand(seed, 8)
    d = r.normal(size=3)
    d /= np.linalg.norm(d)
    p = dict(Ms=8e5, A=1.3e-11, alpha=0.05, modules=DEM | EXC | ZEE, wave=1, amp=20e-3 / MU0, w=2 * math.pi / 1e-9, t0=0.5e-9, dir=tuple(float(v) for v in d))
    return ms, p, _texture(n, seed, 22), _texture(n, seed, 23)


def prepare(case, seed):
    c, k, h = case, case["kind"], _cell(case)
    if k in ("conv", "avg"):
        n = _n(c)
        M = 8e5 * _texture(n, seed)
        s = {"case": c, "demag": api.Demag(n, h, _pbc(c)), "M": M, "H": torch.zeros_like(M)}
        if k == "avg":
            s["M2"], s["H2"] = -7e5 * _texture(n, seed, 1), torch.zeros_like(M)
        elif c["add"]:
            s["H0"] = 1e4 * _texture(n, seed, 2)
        if c.get("energy"):
            s["e"] = torch.zeros(1, dtype=torch.float32, device="cuda")
        return s
    if k == "layers":
        L = c["layers"]
        d = api.MultiLayerDemag(c["nx"], c["ny"], h[0], h[1], [h[2]] * L, [8e-9 * l for l in range(L)])
        M = 8e5 * _texture((c["nx"], c["ny"], L), seed)
        return {"case": c, "demag": d, "M": M, "H": torch.empty_like(M)}
    if k == "llg":
        p = api.FMParams(**_material(c, seed))
        s = api.FMSolver(METHODS[c["method"]], _n(c), h, p)
        s.M.copy_(p.Ms * _texture(_n(c), seed))
        s.set_dt(DT[c["method"]])
        if c["method"] == "RKDP54":
            s.set_astep(dT_max=DT["RKDP54"])
        if c["speedup"]:
            s.set_eval_speedup(c["speedup"])
        return {"case": c, "solver": s, "it": 0}
    if k == "stack":
        hz, z0, grp = _stack(c)
        p = api.FMParams(**_material(c, seed))
        s = api.LayerStackSolver(api.BM_EVAL_RK4, c["nx"], c["ny"], h[0], h[1], hz, z0, p)
        if len(set(grp)) < len(grp):
            s.set_layer_meshes(grp)
        s.M.copy_(p.Ms * _texture((c["nx"], c["ny"], len(hz)), seed))
        s.set_dt(DT["RK4"])
        return {"case": c, "solver": s, "it": 0}
    if k == "batch":
        films, mats = _films(c), _film_materials(c, seed)
        b = api.BatchSolver(api.BM_EVAL_RK4, [(n, h, api.FMParams(**m)) for n, m in zip(films, mats)])
        for q, (n, m) in enumerate(zip(films, mats)):
            b.mesh(q).copy_(m["Ms"] * _texture(n, seed, 100 + q))
        b.set_dt(DT["RK4"])
        return {"case": c, "batch": b}
    ms, p, m0, mt = _adj_inputs(c, seed)
    return {"case": c, "adj": api.RK4Adjoint(_n(c), h, api.FMParams(**p), ms, DT["RK4"], c["steps"], c["every"]), "m0": m0, "mt": mt}


def run(state):
    c, k = state["case"], state["case"]["kind"]
    if k == "conv":
        if c["add"]:
            state["H"].copy_(state["H0"])       # another module's field, which the demag field is added to
        H = state["demag"].convolute(state["M"], state["H"], clear_out=not c["add"], energy=state.get("e"))
        return [H, state["e"]] if "e" in state else [H]
    if k == "avg":
        state["demag"].convolute_averaged(state["M"], state["M2"], state["H"], state["H2"])
        return [state["H"], state["H2"]]
    if k == "layers":
        return [state["demag"].convolute(state["M"], state["H"])]
    if k in ("llg", "stack"):
        state["it"] += c["steps"]
        state["solver"].run_to_iteration(state["it"])
        return [state["solver"].M]
    if k == "batch":
        state["batch"].run(c["steps"])
        return [state["batch"].M]
    loss, M = state["adj"].forward(state["m0"], state["mt"])
    g, ga = state["adj"].backward()
    return [np.float32(loss), M, g, np.float32(ga)]


# ------------------------------------------------------------------------------------------
# What a pass cannot do without

def _sizes(n, pbc=(0, 0, 0)):
    N = [m if p else 2 * m for m, p in zip(n, pbc)]
    if n[2] == 1:
        N[2] = 1
    return N


def _conv_work(n, pbc=(0, 0, 0)):
    """Bytes of M, H and the demag kernel (six real components on a reduced octant, four in 2D), and
    the operations of six real transforms and the kernel product."""
    N, cells = _sizes(n, pbc), n[0] * n[1] * n[2]
    pts, full = (N[0] // 2 + 1) * (N[1] // 2 + 1) * (N[2] // 2 + 1), N[0] * N[1] * N[2]
    return 24.0 * cells + 4.0 * (4 if n[2] == 1 else 6) * pts, 6 * 2.5 * full * math.log2(max(2, full)) + 18.0 * full


def _layers_work(nx, ny, L):
    """The same with one kernel per distance between planes."""
    pts, full = (nx + 1) * (ny + 1), 4 * nx * ny
    return 24.0 * nx * ny * L + 4.0 * 6 * pts * L, L * 6 * 2.5 * full * math.log2(full) + 18.0 * full * L * L


def work(case):
    c, k = case, case["kind"]
    if k == "conv":
        b, f = _conv_work(_n(c), _pbc(c))
        return {"bytes": b + (24.0 * math.prod(_n(c)) if c["add"] else 0.0), "flops": f}
    if k == "avg":
        b, f = _conv_work(_n(c))
        return {"bytes": b + 24.0 * math.prod(_n(c)), "flops": f}
    if k == "layers":
        b, f = _layers_work(c["nx"], c["ny"], c["layers"])
        return {"bytes": b, "flops": f}
    if k == "llg":
        b, f = _conv_work(_n(c))
        cells, s = math.prod(_n(c)), STAGES[c["method"]] * c["steps"]
        conv = c["steps"] if c["speedup"] else s
        return {"bytes": conv * (b - 24.0 * cells) + s * 24.0 * cells, "flops": conv * f + 100.0 * s * cells}
    if k == "stack":
        L = len(_stack(c)[0])
        b, f = _layers_work(c["nx"], c["ny"], L)
        return {"bytes": 4 * c["steps"] * b, "flops": 4 * c["steps"] * (f + 100.0 * c["nx"] * c["ny"] * L)}
    if k == "batch":
        w = [_conv_work(n) for n in _films(c)]
        return {"bytes": 4 * c["steps"] * sum(b for b, _ in w), "flops": 4 * c["steps"] * sum(f for _, f in w)}
    b, f = _conv_work(_n(c))                # forward, the backward pass's own convolution, and its stored stages
    return {"bytes": 4 * c["steps"] * 3.0 * b, "flops": 4 * c["steps"] * 3.0 * f}


# ------------------------------------------------------------------------------------------
# FP64 from the formulas alone

def _newell(x, y, z):
    """Newell's f and g (A. Newell, W. Williams, D. Dunlop, J. Geophys. Res. 98, 9551 (1993))."""
    R = torch.sqrt(x * x + y * y + z * z)

    def ash(a, p, q):       # asinh(a / sqrt(p^2 + q^2)), 0 where its factor is 0 too
        s = torch.sqrt(p * p + q * q)
        return torch.where(s > 0, torch.asinh(a / torch.where(s > 0, s, torch.ones_like(s))), torch.zeros_like(s))

    def atn(a, b):          # atan(a / b), 0 where b is 0 (its factor is 0 too)
        return torch.where(b != 0, torch.atan(a / torch.where(b != 0, b, torch.ones_like(b))), torch.zeros_like(b))

    f = (y / 2 * (z * z - x * x) * ash(y, x, z) + z / 2 * (y * y - x * x) * ash(z, x, y) - x * y * z * atn(y * z, x * R)
         + (2 * x * x - y * y - z * z) * R / 6)
    g = (x * y * z * ash(z, x, y) + y / 6 * (3 * z * z - y * y) * ash(x, y, z) + x / 6 * (3 * z * z - x * x) * ash(y, x, z)
         - z ** 3 / 6 * atn(x * y, z * R) - z * y * y / 2 * atn(x * z, y * R) - z * x * x / 2 * atn(y * z, x * R) - x * y * R / 3)
    return f, g


def _tensor_at(i, j, k, h):
    """Demag tensor N (xx, yy, zz, xy, xz, yz) between equal cells at offsets (i, j, k), given as
    three 1D grids; exact within 12 cells, else the dipole averaged over both cells by a three-point
    rule per axis (right to the sixth order in cell size over distance)."""
    s = max(h)
    h = [v / s for v in h]
    V = h[0] * h[1] * h[2]
    X, Y, Z = torch.meshgrid(i, j, k, indexing="ij")
    out = [torch.zeros_like(X) for _ in range(6)]
    w, wgt = math.sqrt(0.4), ((-1, 5 / 24), (0, 7 / 12), (1, 5 / 24))
    for a, wa in wgt:
        for b, wb in wgt:
            for c, wc in wgt:
                x, y, z = (X + a * w) * h[0], (Y + b * w) * h[1], (Z + c * w) * h[2]
                r2 = x * x + y * y + z * z
                r2 = torch.where(r2 > 0, r2, torch.ones_like(r2))
                q = wa * wb * wc * V / (4 * math.pi) * r2 ** -2.5
                for o, t in zip(out, (r2 - 3 * x * x, r2 - 3 * y * y, r2 - 3 * z * z, -3 * x * y, -3 * x * z, -3 * y * z)):
                    o += q * t
    near = ((X * h[0]) ** 2 + (Y * h[1]) ** 2 + (Z * h[2]) ** 2) < 144
    x0, y0, z0 = X[near], Y[near], Z[near]
    if x0.numel():
        acc = [torch.zeros_like(x0) for _ in range(6)]
        for a, wa in ((-1, -1.0), (0, 2.0), (1, -1.0)):
            for b, wb in ((-1, -1.0), (0, 2.0), (1, -1.0)):
                for c, wc in ((-1, -1.0), (0, 2.0), (1, -1.0)):
                    x, y, z = (x0 + a) * h[0], (y0 + b) * h[1], (z0 + c) * h[2]
                    q = wa * wb * wc / (4 * math.pi * V)
                    for m, (u, v, t) in enumerate(((x, y, z), (y, x, z), (z, y, x))):
                        acc[m] += q * _newell(u, v, t)[0]
                    for m, (u, v, t) in enumerate(((x, y, z), (x, z, y), (y, z, x))):
                        acc[3 + m] += q * _newell(u, v, t)[1]
        for o, v in zip(out, acc):
            o[near] = v
    return out


class _Field:
    """H = -N M of one mesh by zero-padded (or, along periodic axes, cyclic) FFTs."""

    def __init__(self, n, h, pbc=(0, 0, 0)):
        self.n, self.N = n, _sizes(n, pbc)
        grid = []
        for m, p in zip(n, pbc):
            grid.append(torch.arange(m if p else 2 * m - 1, dtype=torch.float64, device="cuda") - (0 if p else m - 1))
        D = [0.0] * 6
        for a in range(-pbc[0], pbc[0] + 1):
            for b in range(-pbc[1], pbc[1] + 1):
                D = [u + v for u, v in zip(D, _tensor_at(grid[0] + a * n[0], grid[1] + b * n[1], grid[2], h))]
        self.K = []
        odd = ((), (), (), (0, 1), (0, 2), (1, 2))
        for q, d in enumerate(D):
            full = torch.zeros(self.N, dtype=torch.float64, device="cuda")
            at = [g.long() % m for g, m in zip(grid, self.N)]
            full[at[0][:, None, None], at[1][None, :, None], at[2][None, None, :]] = d
            for ax in range(3):     # a window of images has no centre for offsets other than 0: its even (odd) part acts
                if pbc[ax]:
                    back = torch.roll(torch.flip(full, [ax]), 1, ax)
                    full = (full - back) / 2 if ax in odd[q] else (full + back) / 2
            self.K.append(torch.fft.rfftn(full))

    def __call__(self, M):
        n, N, (xx, yy, zz, xy, xz, yz) = self.n, self.N, self.K
        v = M.reshape(n[2], n[1], n[0], 3).permute(3, 2, 1, 0)
        f = [torch.fft.rfftn(v[c], s=N) for c in range(3)]
        g = (xx * f[0] + xy * f[1] + xz * f[2], xy * f[0] + yy * f[1] + yz * f[2], xz * f[0] + yz * f[1] + zz * f[2])
        H = [-torch.fft.irfftn(t, s=N)[:n[0], :n[1], :n[2]] for t in g]
        return torch.stack(H).permute(3, 2, 1, 0).reshape(-1, 3)


class _Layers:
    """H = -N M of planes at heights z0, all of one thickness."""

    def __init__(self, nx, ny, h, z0):
        self.nx, self.ny, self.L = nx, ny, len(z0)
        gx = torch.arange(2 * nx - 1, dtype=torch.float64, device="cuda") - (nx - 1)
        gy = torch.arange(2 * ny - 1, dtype=torch.float64, device="cuda") - (ny - 1)
        self.K = {}
        self.at = [[round((z0[d] - z0[s]) / h[2]) for s in range(self.L)] for d in range(self.L)]
        for k in sorted({v for r in self.at for v in r}):
            D = _tensor_at(gx, gy, torch.tensor([float(k)], dtype=torch.float64, device="cuda"), h)
            ks = []
            for d in D:
                full = torch.zeros((2 * nx, 2 * ny), dtype=torch.float64, device="cuda")
                full[(gx.long() % (2 * nx))[:, None], (gy.long() % (2 * ny))[None, :]] = d[:, :, 0]
                ks.append(torch.fft.rfftn(full))
            self.K[k] = ks

    def __call__(self, M):
        N = (2 * self.nx, 2 * self.ny)
        v = M.reshape(self.L, self.ny, self.nx, 3).permute(0, 3, 2, 1)
        f = torch.fft.rfftn(v, s=N, dim=(2, 3))
        H = []
        for d in range(self.L):
            g = [0.0, 0.0, 0.0]
            for s in range(self.L):
                xx, yy, zz, xy, xz, yz = self.K[self.at[d][s]]
                a, b, c = f[s]
                g = [g[0] + xx * a + xy * b + xz * c, g[1] + xy * a + yy * b + yz * c, g[2] + xz * a + yz * b + zz * c]
            H.append(-torch.fft.irfftn(torch.stack(g), s=N, dim=(1, 2))[:, :self.nx, :self.ny])
        return torch.stack(H).permute(0, 3, 2, 1).reshape(-1, 3)


def _laplacian(M, n, h, grp=None):
    """Sum of second differences over h^2 with free ends; planes of different meshes are not coupled."""
    v = M.reshape(n[2], n[1], n[0], 3)
    out = torch.zeros_like(v)
    for ax, m, d in ((2, n[0], h[0]), (1, n[1], h[1]), (0, n[2], h[2])):
        if m > 1:
            e = torch.diff(v, dim=ax) / (d * d)
            if ax == 0 and grp is not None:
                same = torch.tensor(np.diff(grp) == 0, dtype=v.dtype, device=v.device)
                e = e * same[:, None, None, None]
            pad = torch.zeros_like(v.narrow(ax, 0, 1))
            out = out + torch.cat([e, pad], ax) - torch.cat([pad, e], ax)
    return out.reshape(-1, 3)


def _rhs(p, n, h, demag, Ms, Ha, grp=None):
    """M -> dM/dt (Landau-Lifshitz form of the Gilbert equation); demag: M -> its field."""
    ea = torch.tensor(p.get("ea", (1.0, 0.0, 0.0)), dtype=torch.float64, device="cuda")
    al, K1 = p["alpha"], p.get("K1", 0.0)

    def f(M):
        H = demag(M) + 2 * p["A"] / (MU0 * Ms * Ms) * _laplacian(M, n, h, grp) + Ha
        if p["modules"] & ANI:
            H = H + 2 * K1 / (MU0 * Ms * Ms) * (M @ ea)[:, None] * ea
        mxh = torch.linalg.cross(M, H)
        return -GAMMA / (1 + al * al) * (mxh + al * torch.linalg.cross(M / Ms, mxh))
    return f


def _unit(M, Ms):
    return M / M.norm(dim=1, keepdim=True) * Ms


def _rk4(f, M, dt, Ms):
    k1 = f(M)
    k2 = f(M + dt / 2 * k1)
    k3 = f(M + dt / 2 * k2)
    k4 = f(M + dt * k3)
    return _unit(M + dt / 6 * (k1 + 2 * k2 + 2 * k3 + k4), Ms)


def _heun(f, M, dt, Ms):
    P = M + dt * f(M)
    return _unit((M + P + dt * f(P)) / 2, Ms)


_A = ((), (1 / 5,), (3 / 40, 9 / 40), (44 / 45, -56 / 15, 32 / 9), (19372 / 6561, -25360 / 2187, 64448 / 6561, -212 / 729),
      (9017 / 3168, -355 / 33, 46732 / 5247, 49 / 176, -5103 / 18656), (35 / 384, 0.0, 500 / 1113, 125 / 192, -2187 / 6784, 11 / 84))


def _dp5(f, M, dt, Ms):
    k = []
    for s in range(6):
        k.append(f(M + dt * sum(a * q for a, q in zip(_A[s], k)) if s else M))
    return _unit(M + dt * sum(a * q for a, q in zip(_A[6], k)), Ms)


class _Speedup:
    """The demag field convolved at the start of each step only, else extrapolated in time from the
    last p of these less the cell's own part; convolved as well until p are saved."""

    def __init__(self, field, p, times):
        self.field, self.p, self.times, self.saved, self.call = field, p, times, [], 0
        self.stages = len(times)

    def __call__(self, M):
        step, s = divmod(self.call, self.stages)
        t = step + self.times[s]
        self.call += 1
        if s == 0 or len(self.saved) < self.p:
            H = self.field(M)
            if s == 0:
                self.saved = (self.saved + [(t, H + M / 3)])[-self.p:]     # cubic cells: N = 1/3 of a cell on itself
            return H
        H = -M / 3
        for q, (tq, Hq) in enumerate(self.saved):
            a = 1.0
            for r, (tr, _) in enumerate(self.saved):
                if r != q:
                    a *= (t - tr) / (tq - tr)
            H = H + a * Hq
        return H


_TIMES = {"TEULER": (0.0, 1.0), "RK4": (0.0, 0.5, 0.5, 1.0), "RKDP54": (0.0, 0.2, 0.3, 0.8, 8 / 9, 1.0)}
_STEP = {"TEULER": _heun, "RK4": _rk4, "RKDP54": _dp5}


def _ha(p):
    return torch.tensor(p.get("Ha", (0.0, 0.0, 0.0)), dtype=torch.float64, device="cuda")


def exact(case, seed):
    c, k, h = case, case["kind"], _cell(case)
    if k == "conv":
        n = _n(c)
        M = (8e5 * _texture(n, seed)).double()
        H = _Field(n, h, _pbc(c))(M)
        e = -MU0 / 2 * (M * H).sum().reshape(1) / M.shape[0]
        if c["add"]:
            H = H + (1e4 * _texture(n, seed, 2)).double()
        return [H, e] if c.get("energy") else [H]
    if k == "avg":
        n = _n(c)
        H = _Field(n, h)(((8e5 * _texture(n, seed)).double() + (-7e5 * _texture(n, seed, 1)).double()) / 2)
        return [H, H]
    if k == "layers":
        L = c["layers"]
        return [_Layers(c["nx"], c["ny"], h, [8e-9 * l for l in range(L)])((8e5 * _texture((c["nx"], c["ny"], L), seed)).double())]
    if k == "llg":
        n, p = _n(c), _material(c, seed)
        M = (p["Ms"] * _texture(n, seed)).double()
        field = _Field(n, h)
        if c["speedup"]:
            field = _Speedup(field, c["speedup"], _TIMES[c["method"]])
        f = _rhs(p, n, h, field, p["Ms"], _ha(p))
        for _ in range(c["steps"]):
            M = _STEP[c["method"]](f, M, DT[c["method"]], p["Ms"])
        return [M]
    if k == "stack":
        hz, z0, grp = _stack(c)
        n, p = (c["nx"], c["ny"], len(hz)), _material(c, seed)
        f = _rhs(p, n, h, _Layers(c["nx"], c["ny"], h, z0), p["Ms"], _ha(p), grp)
        M = (p["Ms"] * _texture(n, seed)).double()
        for _ in range(c["steps"]):
            M = _rk4(f, M, DT["RK4"], p["Ms"])
        return [M]
    if k == "batch":
        out = []
        for q, (n, p) in enumerate(zip(_films(c), _film_materials(c, seed))):
            f = _rhs(p, n, h, _Field(n, h), p["Ms"], _ha(p))
            M = (p["Ms"] * _texture(n, seed, 100 + q)).double()
            for _ in range(c["steps"]):
                M = _rk4(f, M, DT["RK4"], p["Ms"])
            out.append(M)
        return [torch.cat(out)]
    n = _n(c)
    ms, p, m0, mt = _adj_inputs(c, seed)
    Ms = ms.double()[:, None].requires_grad_(True)
    amp = torch.tensor(p["amp"], dtype=torch.float64, device="cuda", requires_grad=True)
    d, field = torch.tensor(p["dir"], dtype=torch.float64, device="cuda"), _Field(n, h)
    M = Ms * m0.double()
    for s in range(c["steps"]):
        x = p["w"] * (s * DT["RK4"] - p["t0"])
        M = _rk4(_rhs(p, n, h, field, Ms, amp * d * (math.sin(x) / x if x else 1.0)), M, DT["RK4"], Ms)
    loss = 1 - ((M / Ms) * mt.double()).sum() / M.shape[0]
    loss.backward()
    return [np.float64(loss.item()), M.detach(), Ms.grad.reshape(-1), np.float64(amp.grad.item())]
