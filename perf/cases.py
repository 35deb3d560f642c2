"""Workloads that measure the lattice update through the package's public entry points.

Each case is one thing a user of the package has it do over and over:
  * step    a solver run between two write steps: Case.step(n), then the fields a write
            step hands out (Case.get).  D2Q9 and D3Q15, periodic boxes and walled columns,
            with and without the energy field, every storage precision.  The sizes are those
            of the example dictionaries (3 x 301 column, 101^3 bubble), of the benchmark
            (256^3 bubble, 128 x 128 x 384 column, 128^2 droplet) and ragged ones between.
  * batch   an ensemble of small D2Q9 cases advanced together (Batch.run_to_steady).
  * train   one Adam run of the warm-start network (Mlp.train).

FP64 runs use the per-routine solver defaults (fused off, heat transfer on where the case
has an energy field); the other precisions use the fused kernels, as the benchmark does.
Fields come back from the library as doubles that hold the precision's own values, so
reduced-precision outputs are handed on as float32.
"""
import ctypes
import math
import tempfile

import numpy as np
import torch

import multiphaselb_amd as M
from multiphaselb_amd.casefiles import BC, CaseSpec
from multiphaselb_amd.initfields import maxwell, vdw_critical

TC = vdw_critical(0.5, 4.0)[1]
PRECISION = {"fp64": M.FP64, "fp32": M.FP32, "fp16s": M.FP16S, "fp16n": M.FP16N}
LAM9 = (1.0, 1.1, 1.1, 1.0, 1.1, 1.0, 1.1, 0.8, 0.8)
GLAM9 = (0.0, 1.0, 1.0, 0.8, 1.0, 0.8, 1.0, 1.0, 1.0)
LAM15 = (1.0, 1.1, 1.1, 1.0, 1.1, 1.0, 1.1, 1.0, 1.1, 1.0, 1.0, 1.0, 1.0, 1.0, 1.2)
GLAM15 = (0.0, 1.0, 1.0, 1.2, 1.0, 1.2, 1.0, 1.0, 1.0, 1.0, 1.0, 1.0, 1.0, 1.0, 1.0)
WIDTHS = (9, 256, 256, 256, 128)
BOX = {"XY": 3, "XYZ": 5, "column2d": 1, "column3d": 3}


def _step(name, box, nx, ny, nz, precision, thermal, steps, tr=0.8, surf=False):
    return {"name": name, "kind": "step", "box": box, "nx": nx, "ny": ny, "nz": nz, "precision": precision,
            "thermal": thermal, "steps": steps, "tr": tr, "surf": surf}


def listed():
    return [
        # the reference's evaporation column (examples: 3 x 301, walls at two temperatures, 200 000 steps,
        # a write step every 25 000): the smallest lattice, where launches and latency are everything
        _step("column2d_3x301_fp64", "column2d", 3, 301, 1, "fp64", True, 500, 0.9),
        # a 128^2 droplet, the parity workload of the 2D solver
        _step("droplet2d_128_fp64", "XY", 128, 128, 1, "fp64", False, 500, 0.85),
        # a mid-size ragged 2D case with the energy field, FP32 fused kernels
        _step("droplet2d_401x333_thermal_fp32", "XY", 401, 333, 1, "fp32", True, 500, 0.85),
        # the reference's 3D bubble example (101^3) at its defaults: FP64, energy field on
        _step("bubble3d_101_thermal_fp64", "XYZ", 101, 101, 101, "fp64", True, 40),
        # the isothermal FP64 solver at a production size
        _step("bubble3d_160_fp64", "XYZ", 160, 160, 160, "fp64", False, 40),
        # the headline benchmark: 256^3 bubble, FP32
        _step("bubble3d_256_fp32", "XYZ", 256, 256, 256, "fp32", False, 500),
        # FP16 storage, a ragged box (one reference density)
        _step("bubble3d_201x150x180_fp16s", "XYZ", 201, 150, 180, "fp16s", False, 500),
        # FP16 storage with per-node references, with the energy field
        _step("bubble3d_160_thermal_fp16n", "XYZ", 160, 160, 160, "fp16n", True, 200),
        # the benchmark's thermal workload, FP32, at 192^3
        _step("bubble3d_192_thermal_fp32", "XYZ", 192, 192, 192, "fp32", True, 300),
        # the walled evaporation column of the accuracy workload, FP32
        _step("column3d_128x128x384_fp32", "column3d", 128, 128, 384, "fp32", True, 200),
        # 256 small cases advanced together, as the benchmark's ensemble
        {"name": "ensemble_256_fp32", "kind": "batch", "count": 256, "lmin": 64, "lmax": 256, "precision": "fp32",
         "steps": 1000},
        # one stage of the warm-start network's training
        {"name": "train_256x400", "kind": "train", "batch": 256, "iters": 400, "samples": 4096},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["box2d", "box2d", "column2d", "box3d", "box3d", "box3d", "box3d", "column3d", "batch", "train"])
    if kind == "train":
        return {"kind": "train", "batch": 32 * rng.randint(1, 8), "iters": 20 * rng.randint(3, 20),
                "samples": rng.randint(500, 6000)}
    if kind == "batch":
        lo = rng.randint(32, 128)
        return {"kind": "batch", "count": _logint(rng, 12, 200), "lmin": lo, "lmax": rng.randint(lo + 8, 256),
                "precision": rng.choice(["fp64", "fp32", "fp16n"]), "steps": 100 * rng.randint(2, 6)}
    if kind == "column2d":
        nx, ny = _logint(rng, 3, 120), _logint(rng, 65, 500)
        prec = rng.choice(["fp64", "fp64", "fp32"])
        return _unnamed(_step("", "column2d", nx, ny, 1, prec, True, 20 * rng.randint(8, 25), rng.uniform(0.85, 0.92)))
    if kind == "box2d":
        nx, ny = _logint(rng, 65, 700), _logint(rng, 65, 700)
        prec = rng.choice(["fp64", "fp32", "fp16n"])
        return _unnamed(_step("", "XY", nx, ny, 1, prec, rng.random() < 0.4, 20 * rng.randint(8, 25),
                              rng.uniform(0.75, 0.9), rng.random() < 0.25))
    prec = rng.choice(["fp64", "fp32", "fp32", "fp16s", "fp16n"])
    hi = 150 if prec == "fp64" else 200
    if kind == "column3d":
        nx, ny, nz = _logint(rng, 20, 110), _logint(rng, 20, 110), _logint(rng, 80, 320)
        prec = rng.choice(["fp64", "fp32", "fp16n"])
        return _unnamed(_step("", "column3d", nx, ny, nz, prec, True, rng.randint(30, 80)))
    nx, ny, nz = (_logint(rng, 48, hi) for _ in range(3))
    return _unnamed(_step("", "XYZ", nx, ny, nz, prec, rng.random() < 0.45, rng.randint(40, 120),
                          rng.uniform(0.75, 0.88), rng.random() < 0.25))


def _unnamed(case):
    del case["name"]
    return case


# --------------------------------------------------------------------------------------
# inputs


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _spec(c):
    three = c["box"] in ("XYZ", "column3d")
    column = c["box"].startswith("column")
    kw = dict(lbmodel=1 if three else 0, nx=c["nx"], ny=c["ny"], nz=c["nz"], btype=BOX[c["box"]],
              f_model=2 if three else 0, f_Lambda=LAM15 if three else LAM9, f_sigma=0.125, f_st=int(c["surf"]),
              f_kappa=0.3 if c["surf"] else 0.0, g_model=1, g_Lambda=GLAM15 if three else GLAM9, g_alpha1=0.25,
              g_alpha2=0.25, Cv=4.0, end=2 * 10 ** 9, write_interval=c["steps"])
    if column:
        wall = "Z" if three else "Y"
        kw["g"] = (0.0, 0.0, -1e-5) if three else (0.0, -1.234567e-07, 0.0)
        kw["f_bc"] = {wall + "0": BC("bounceBack"), wall + "1": BC("bounceBack")}
        hot = BC("fixedRandomT", (0.95 * TC,), pert=0.5, duration=10 ** 8) if three else BC("fixedT", (0.92 * TC,))
        kw["g_bc"] = {wall + "0": hot, wall + "1": BC("fixedT", (c["tr"] * TC,))}
    return CaseSpec(**kw)


def _copy_ends(a, axes):
    """The last plane of a periodic axis stores the first one's sites again."""
    for ax in axes:
        a.select(ax, a.shape[ax] - 1).copy_(a.select(ax, 0))
    return a


def _fields(c, seed):
    """rho (N), U (N, 3) and T (N) of the start, node-major, as doubles on the device: a
    bubble, droplet or pool between the coexistence densities in a smooth flow."""
    dev = _device()
    gen = torch.Generator(device=dev).manual_seed(seed)
    r = np.random.default_rng(seed)
    nx, ny, nz = c["nx"], c["ny"], c["nz"]
    three = c["box"] in ("XYZ", "column3d")
    column = c["box"].startswith("column")
    rv, rl = maxwell(c["tr"] * TC)
    x, y, z = (torch.arange(n, dtype=torch.float64, device=dev) for n in (nx, ny, nz))
    X, Y, Z = x[None, None, :], y[None, :, None], z[:, None, None]
    if column:
        h, n = (Z, nz) if three else (Y, ny)
        level = n * r.uniform(0.3, 0.4)
        rho = 0.5 * (rl + rv) + 0.5 * (rv - rl) * torch.tanh(2.0 * (h - level) / 5.0)
        rho = rho.expand(nz, ny, nx).contiguous()
    else:
        low = min(nx, ny, nz) if three else min(nx, ny)
        R = low * r.uniform(0.17, 0.22)
        cen = [(n - 1) / 2.0 + r.uniform(-2.0, 2.0) for n in (nx, ny, nz)]
        d2 = (X - cen[0]) ** 2 + (Y - cen[1]) ** 2 + ((Z - cen[2]) ** 2 if three else 0.0)
        inside, outside = (rl, rv) if c["box"] == "XY" else (rv, rl)
        rho = 0.5 * (inside + outside) + 0.5 * (outside - inside) * torch.tanh(2.0 * (d2.sqrt() - R) / 5.0)
    rho = rho + 1e-4 * (2.0 * torch.rand(rho.shape, generator=gen, dtype=torch.float64, device=dev) - 1.0)
    U = torch.zeros((nz, ny, nx, 3), dtype=torch.float64, device=dev)
    kx, ky = 2.0 * math.pi / (nx - 1), 2.0 * math.pi / (ny - 1)
    kz = 2.0 * math.pi / max(1, nz - 1)
    px, py, pz = r.uniform(0.0, 2.0 * math.pi, 3)
    amp = 0.02
    if column and three:
        damp = torch.sin(0.5 * kz * Z) ** 2
        U[..., 0] = amp * damp * torch.sin(ky * Y + py)
        U[..., 1] = amp * damp * torch.sin(kx * X + px)
    elif column:
        pass
    else:
        U[..., 0] = amp * torch.sin(ky * Y + py) * (torch.cos(kz * Z + pz) if three else 1.0)
        U[..., 1] = amp * torch.sin(kx * X + px) * (torch.cos(kz * Z) if three else 1.0)
        if three:
            U[..., 2] = amp * torch.sin(kx * X + py) * torch.cos(ky * Y + px)
    periodic = {"XY": (2, 1), "XYZ": (2, 1, 0), "column2d": (2,), "column3d": (2, 1)}[c["box"]]
    _copy_ends(rho, periodic)
    _copy_ends(U, periodic)
    T = torch.full((nz * ny * nx,), c["tr"] * TC, dtype=torch.float64, device=dev)
    if c["precision"] != "fp64":
        # what the library's FP32 arrays hold of them
        rho, U, T = (v.float().double() for v in (rho, U, T))
    return rho.reshape(-1), U.reshape(-1, 3), T


def _batch_cases(c, seed):
    """Sizes, densities and temperatures of an ensemble: droplets and bubbles on L x L boxes."""
    r = np.random.default_rng(seed + 77)
    layout = np.random.default_rng(c["count"])      # the sizes belong to the case, not to the seed
    sizes = np.unique(np.linspace(c["lmin"], c["lmax"], 5).round().astype(int))
    out = []
    for _ in range(c["count"]):
        L = int(layout.choice(sizes))
        tr = float(r.uniform(0.7, 0.95))
        rv, rl = maxwell(tr * TC)
        R = r.uniform(6.0, max(7.0, L / 4.0))
        inside, outside = (rl, rv) if r.random() < 0.5 else (rv, rl)
        i = np.arange(L) - (L - 1) / 2.0
        rad = np.sqrt(i[None, :] ** 2 + i[:, None] ** 2)
        rho = 0.5 * (inside + outside) + 0.5 * (outside - inside) * np.tanh(2.0 * (rad - R) / 5.0)
        rho += 1e-4 * (2.0 * r.random((L, L)) - 1.0)
        rho[:, -1] = rho[:, 0]
        rho[-1, :] = rho[0, :]
        if c["precision"] != "fp64":
            rho = rho.astype(np.float32).astype(np.float64)
        out.append((L, rho.ravel(), tr * TC))
    return out


def _train_data(c, seed):
    r = np.random.default_rng(seed)
    X = r.uniform(-1.0, 1.0, (c["samples"], WIDTHS[0])).astype(np.float32)
    d = np.linspace(-4.0, 4.0, WIDTHS[-1])
    Y = np.tanh(d[None, :] * (1.0 + 0.5 * X[:, :1]) + X[:, 1:2]) * (1.0 + 0.3 * X[:, 2:3]) + 0.2 * X[:, 5:6]
    idx = r.integers(0, c["samples"], c["iters"] * c["batch"]).astype(np.int32)
    parts = []
    for a, b in zip(WIDTHS[:-1], WIDTHS[1:]):
        lim = math.sqrt(6.0 / (a + b))
        parts += [r.uniform(-lim, lim, a * b), np.zeros(b)]
    return X, Y.astype(np.float32), idx, np.concatenate(parts).astype(np.float32)


def prepare(case, seed):
    c = case
    if c["kind"] == "train":
        X, Y, idx, p = _train_data(c, seed)
        net = M.Mlp(list(WIDTHS), c["batch"])
        net.set_params(p)
        return {"kind": "train", "net": net, "X": X, "Y": Y, "idx": idx, "p": p}
    if c["kind"] == "batch":
        cases = _batch_cases(c, seed)
        hosts = {}
        for L, _, _ in cases:
            if L not in hosts:
                with tempfile.TemporaryDirectory(prefix="mplb_perf_") as d:
                    M.write_case(d, CaseSpec(lbmodel=0, nx=L, ny=L, btype=3, f_model=0, end=2 * 10 ** 9,
                                             write_interval=10 ** 9))
                    hosts[L] = M.Case(d, heat_transfer=False, device=-1)
        b = M.Batch([hosts[L] for L, _, _ in cases], [rho for _, rho, _ in cases], [T for _, _, T in cases],
                    precision=PRECISION[c["precision"]])
        b.init()
        return {"kind": "batch", "batch": b, "steps": c["steps"], "fp64": c["precision"] == "fp64"}
    rho, U, T = (v.cpu().numpy() for v in _fields(c, seed))
    with tempfile.TemporaryDirectory(prefix="mplb_perf_") as d:
        M.write_case(d, _spec(c))
        k = M.Case(d, precision=PRECISION[c["precision"]], heat_transfer=c["thermal"], fused=c["precision"] != "fp64")
    k.set("rho", rho)
    k.set("U", U)
    k.set("T", T)
    k.init()
    return {"kind": "step", "case": k, "steps": c["steps"], "fp64": c["precision"] == "fp64",
            "names": ("rho", "U", "T") if c["thermal"] else ("rho", "U")}


def run(state):
    s = state
    if s["kind"] == "train":
        s["net"].set_params(s["p"])
        hist = s["net"].train(s["X"], s["Y"], s["idx"], lr=1e-3)
        return {"loss": hist, "params": s["net"].get_params()}
    if s["kind"] == "batch":
        b = s["batch"]
        b.run_to_steady(0.0, check_every=100, max_steps=s["steps"])
        out = np.concatenate([b.get(k) for k in range(b.n)])
        return {"rho": out if s["fp64"] else out.astype(np.float32)}
    k = s["case"]
    k.step(s["steps"])
    out = {n: k.get(n) for n in s["names"]}
    return out if s["fp64"] else {n: v.astype(np.float32) for n, v in out.items()}


def work(case):
    """Every population read once and written once per step, the macroscopic fields that
    the next step's stencils need (density, and with the energy field temperature and
    velocity) written and read once; the arithmetic of the moment transforms and sources."""
    c = case
    if c["kind"] == "train":
        macs = sum(max(32, a) * b for a, b in zip(WIDTHS[:-1], WIDTHS[1:]))
        P = sum(a * b + b for a, b in zip(WIDTHS[:-1], WIDTHS[1:]))
        return {"bytes": c["iters"] * (P * 4 * 7 + c["batch"] * (WIDTHS[0] + WIDTHS[-1]) * 4),
                "flops": 6.0 * macs * c["batch"] * c["iters"]}
    s_pdf = {"fp64": 8, "fp32": 4, "fp16s": 2, "fp16n": 2}[c["precision"]]
    s_mac = 8 if c["precision"] == "fp64" else 4
    ref = 4 if c["precision"] == "fp16n" else 0
    if c["kind"] == "batch":
        nodes = sum(L * L for L, _, _ in _batch_sizes(c))
        return {"bytes": float(nodes) * c["steps"] * (18 * s_pdf + ref), "flops": 250.0 * nodes * c["steps"]}
    three = c["box"] in ("XYZ", "column3d")
    q = 15 if three else 9
    n = float(c["nx"] * c["ny"] * c["nz"]) * c["steps"]
    per = 2 * q * s_pdf * (2 if c["thermal"] else 1) + 2 * s_mac * ((2 + (3 if three else 2)) if c["thermal"] else 1) + ref
    fl = (500.0 if three else 250.0) * (2.2 if c["thermal"] else 1.0)
    return {"bytes": n * per, "flops": n * fl}


def _batch_sizes(c):
    layout = np.random.default_rng(c["count"])
    sizes = np.unique(np.linspace(c["lmin"], c["lmax"], 5).round().astype(int))
    return [(int(layout.choice(sizes)), None, None) for _ in range(c["count"])]


# --------------------------------------------------------------------------------------
# the same in 64 bits, from the equations


class _Lattice:
    """Velocities, weights, moment matrix and its inverse of D2Q9 or D3Q15."""

    def __init__(self, three, dev):
        if three:
            self.c = np.array([(0, 0, 0), (1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1),
                               (1, 1, 1), (-1, 1, 1), (1, -1, 1), (-1, -1, 1), (1, 1, -1), (-1, 1, -1), (1, -1, -1),
                               (-1, -1, -1)])
            w = {0: (2 / 9, 0.0), 1: (1 / 9, 1 / 3), 3: (1 / 72, 1 / 24)}
        else:
            self.c = np.array([(0, 0, 0), (1, 0, 0), (0, 1, 0), (-1, 0, 0), (0, -1, 0), (1, 1, 0), (-1, 1, 0),
                               (-1, -1, 0), (1, -1, 0)])
            w = {0: (4 / 9, 0.0), 1: (1 / 9, 1 / 3), 2: (1 / 36, 1 / 12)}
        self.three, self.Q = three, len(self.c)
        c2 = (self.c ** 2).sum(1)
        self.omega, self.w = ([w[s][i] for s in c2] for i in (0, 1))
        self.rev = [int(np.where((self.c == -v).all(1))[0][0]) for v in self.c]
        x, y, z = self.c.T.astype(float)
        if three:
            rows = [1 + 0 * x, c2 - 2, (15 * c2 ** 2 - 55 * c2 + 32) / 2, x, x * (5 * c2 - 13) / 2, y,
                    y * (5 * c2 - 13) / 2, z, z * (5 * c2 - 13) / 2, 3 * x * x - c2, y * y - z * z, x * y, y * z, x * z,
                    x * y * z]
        else:
            rows = [1 + 0 * x, 3 * c2 - 4, (9 * c2 ** 2 - 21 * c2 + 8) / 2, x, (3 * c2 - 5) * x, y, (3 * c2 - 5) * y,
                    x * x - y * y, x * y]
        m = np.array(rows)
        self.M = torch.tensor(m, device=dev)
        self.Minv = torch.tensor(m.T / (m ** 2).sum(1), device=dev)


def _table(c, lat, dev):
    """Upstream node x - c_k of every node and link (-1: no such node).  Periodic axes
    store the first plane's sites again in the last one: a node at one end takes its
    missing links from its copy at the other.  The walls of a 3D column are closed at
    their four corners only, as the solver's lattice generator does it."""
    nx, ny, nz = c["nx"], c["ny"], c["nz"]
    idx = torch.arange(nx * ny * nz, dtype=torch.int32, device=dev).reshape(nz, ny, nx)
    nb = torch.full((lat.Q, nz, ny, nx), -1, dtype=torch.int32, device=dev)
    for k, (cx, cy, cz) in enumerate(lat.c):
        def cut(n, s):
            return (slice(max(0, s), n + min(0, s)), slice(max(0, -s), n + min(0, -s)))
        (xd, xs), (yd, ys), (zd, zs) = cut(nx, cx), cut(ny, cy), cut(nz, cz)
        nb[k, zd, yd, xd] = idx[zs, ys, xs]

    def pair(a, b):
        a.copy_(torch.where(a == -1, b, a))
        b.copy_(torch.where(b == -1, a, b))

    def corners(z):
        cor = [nb[:, z, 0, 0], nb[:, z, 0, nx - 1], nb[:, z, ny - 1, 0], nb[:, z, ny - 1, nx - 1]]
        for i in range(4):
            for j in range(4):
                if i != j:
                    cor[i].copy_(torch.where(cor[i] == -1, cor[j], cor[i]))

    if c["box"] == "XYZ":
        pair(nb[:, :, :, 0], nb[:, :, :, nx - 1])
        pair(nb[:, :, 0, :], nb[:, :, ny - 1, :])
        pair(nb[:, 0], nb[:, nz - 1])
    elif c["box"] == "column3d":
        pair(nb[:, 1:nz - 1, :, 0], nb[:, 1:nz - 1, :, nx - 1])
        pair(nb[:, 1:nz - 1, 0, :], nb[:, 1:nz - 1, ny - 1, :])
        corners(0)
        corners(nz - 1)
    elif c["box"] == "XY":
        pair(nb[:, 0, 1:ny - 1, 0], nb[:, 0, 1:ny - 1, nx - 1])
        pair(nb[:, 0, 0, 1:nx - 1], nb[:, 0, ny - 1, 1:nx - 1])
        corners(0)
    else:
        pair(nb[:, 0, :, 0], nb[:, 0, :, nx - 1])
    return nb.reshape(lat.Q, -1)


class _Exact:
    """The time step written down from its equations, whole arrays at a time."""

    def __init__(self, lat, nb, rho, U, T, spec, thermal, wall=()):
        self.lat, self.nb, self.rho, self.U, self.T = lat, nb, rho, list(U), T
        self.s, self.thermal, self.wall = spec, thermal, wall
        self.periodic = not wall
        self.interior = None if self.periodic else (nb != -1).all(0)
        dev = rho.device
        self.lam = torch.tensor(spec.f_Lambda, dtype=torch.float64, device=dev)[:, None]
        self.glam = list(spec.g_Lambda)
        self.f = torch.stack([self._feq(k) for k in range(lat.Q)])
        if thermal:
            self.g = self._geq(self.T, self.U)
        self._force()
        self.S = self._heat() if thermal else None

    def at(self, q, k):
        """q at x - c_k (own value where there is no such node)."""
        if self.periodic:
            return q.index_select(0, self.nb[k])
        return torch.where(self.nb[k] == -1, q, q.index_select(0, self.nb[k].clamp(min=0)))

    def _p(self, rho, T):
        s = self.s
        return rho * s.R * T / (s.M - rho * s.b) - s.a * rho * rho / s.M ** 2

    def _feq(self, k):
        cu = sum(int(v) * u for v, u in zip(self.lat.c[k], self.U))
        if isinstance(cu, int):
            cu = 0.0 * self.rho
        u2 = sum(u * u for u in self.U)
        return self.rho * self.lat.omega[k] * (1 + 3 * cu + 4.5 * cu * cu - 1.5 * u2)

    def _neq(self, T, U):
        n = torch.zeros((self.lat.Q,) + T.shape, dtype=torch.float64, device=T.device)
        n[0], n[1], n[2] = T, self.s.g_alpha1 * T, self.s.g_alpha2 * T
        for d in range(3 if self.lat.three else 2):
            n[3 + 2 * d] = T * U[d]
            n[4 + 2 * d] = -n[3 + 2 * d]
        return n

    def _geq(self, T, U):
        return self.lat.Minv @ self._neq(T, U)

    def _force(self):
        lat, s = self.lat, self.s
        self.psi = torch.sqrt(2 * (self._p(self.rho, self.T) - self.rho / 3) / s.G)
        F = [torch.zeros_like(self.rho) for _ in range(3)]
        self.dpsi = {}
        for k in range(1, lat.Q):
            p = self.at(self.psi, lat.rev[k])
            if s.f_st:
                self.dpsi[k] = p - self.psi
            for d in range(3):
                if lat.c[k][d]:
                    F[d] += float(lat.c[k][d]) * lat.w[k] * p
        self.Fi = []
        for d in range(3):
            v = -s.G * self.psi * F[d]
            self.Fi.append(v if self.periodic else torch.where(self.interior, v, torch.zeros_like(v)))

    def _total(self, rho):
        # the benchmark cases have rho_0 <= 0 (reference density 0) and no external force
        return [F + rho * g for F, g in zip(self.Fi, self.s.g)]

    def _collide_f(self):
        lat, s, rho, U = self.lat, self.s, self.rho, self.U
        m = lat.M @ self.f
        F = self._total(rho)
        u2 = U[0] ** 2 + U[1] ** 2 + U[2] ** 2
        eq, S = torch.zeros_like(m), torch.zeros_like(m)
        L = s.f_Lambda
        if lat.three:
            uF = sum(u * f for u, f in zip(U, F))
            F2 = sum(f * f for f in F)
            eq[0], eq[1], eq[2] = rho, rho * (u2 - 1), rho * (1 - 5 * u2)
            S[1] = 2 * uF + 6 * s.f_sigma * F2 / (self.psi ** 2 * (1 / L[1] - 0.5))
            S[2] = -10 * uF
            for d in range(3):
                eq[3 + 2 * d], eq[4 + 2 * d] = rho * U[d], -7 / 3 * rho * U[d]
                S[3 + 2 * d], S[4 + 2 * d] = F[d], -7 / 3 * F[d]
            eq[9], eq[10] = rho * (2 * U[0] ** 2 - U[1] ** 2 - U[2] ** 2), rho * (U[1] ** 2 - U[2] ** 2)
            S[9], S[10] = 4 * U[0] * F[0] - 2 * U[1] * F[1] - 2 * U[2] * F[2], 2 * U[1] * F[1] - 2 * U[2] * F[2]
            for i, (a, b) in zip((11, 12, 13), ((0, 1), (1, 2), (0, 2))):
                eq[i], S[i] = rho * U[a] * U[b], U[a] * F[b] + U[b] * F[a]
        else:
            uF = U[0] * F[0] + U[1] * F[1]
            F2 = self.Fi[0] ** 2 + self.Fi[1] ** 2
            eq[0], eq[1], eq[2] = rho, rho * (3 * u2 - 2), rho * (1 - 3 * u2)
            S[1] = 6 * uF + 12 * s.f_sigma * F2 / (self.psi ** 2 * (1 / L[1] - 0.5))
            S[2] = -6 * uF - 12 * s.f_sigma * F2 / (self.psi ** 2 * (1 / L[2] - 0.5))
            for d in range(2):
                eq[3 + 2 * d], eq[4 + 2 * d], S[3 + 2 * d], S[4 + 2 * d] = rho * U[d], -rho * U[d], F[d], -F[d]
            eq[7], eq[8] = rho * (U[0] ** 2 - U[1] ** 2), rho * U[0] * U[1]
            S[7], S[8] = 2 * (U[0] * F[0] - U[1] * F[1]), U[0] * F[1] + U[1] * F[0]
        m = m - self.lam * (m - eq) + (1 - 0.5 * self.lam) * S
        if s.f_st:
            D = 3 if lat.three else 2
            Qt = [[torch.zeros_like(rho) for _ in range(D)] for _ in range(D)]
            for k in range(1, lat.Q):
                for a in range(D):
                    for b in range(a, D):
                        cc = int(lat.c[k][a] * lat.c[k][b])
                        if cc:
                            Qt[a][b] += cc * lat.w[k] * self.dpsi[k]
            sc = 0.5 * self.psi * s.G * s.f_kappa
            q = lambda a, b: Qt[a][b] * sc  # noqa: E731
            if lat.three:
                m[1] += 4 * L[1] * (q(0, 0) + q(1, 1) + q(2, 2)) / 5
                m[9] -= L[10] * (2 * q(0, 0) - q(1, 1) - q(2, 2))
                m[10] -= L[10] * (q(1, 1) - q(2, 2))
                for i, (a, b) in zip((11, 12, 13), ((0, 1), (1, 2), (0, 2))):
                    m[i] -= L[10] * q(a, b)
            else:
                m[1] += 1.5 * L[1] * (q(0, 0) + q(1, 1))
                m[2] -= 1.5 * L[2] * (q(0, 0) + q(1, 1))
                m[7] -= L[8] * (q(0, 0) - q(1, 1))
                m[8] -= L[8] * q(0, 1)
        return lat.Minv @ m

    def _collide_g(self):
        n = self.lat.M @ self.g
        d = n - self._neq(self.T, self.U)
        lam = self.glam
        for k in range(self.lat.Q):
            n[k] -= lam[k] * d[k]
        for i in range(3 if self.lat.three else 2):
            n[3 + 2 * i] -= lam[4 + 2 * i] * (lam[3 + 2 * i] / 2 - 1) * d[4 + 2 * i]
        n[0] += (1 - 0.5 * lam[0]) * self.S
        return self.lat.Minv @ n

    def _stream(self, f):
        return torch.stack([self.at(f[k], k) for k in range(self.lat.Q)])

    def _bounce(self, f):
        lat = self.lat
        for nodes, _ in self.wall:
            v = f[:, nodes]
            miss = self.nb[:, nodes] == -1
            for k in range(lat.Q):
                r = lat.rev[k]
                axis = int((lat.c[k] ** 2).sum()) == 1
                avg = 0.5 * (v[k] + v[r])
                both = ~miss[k] & ~miss[r] if axis else torch.zeros_like(miss[k])
                v[k] = torch.where(miss[k], v[r], torch.where(both, avg, v[k]))
                v[r] = torch.where(both, v[k], v[r])
            f[:, nodes] = v

    def _wall_temperature(self, g):
        lat = self.lat
        for nodes, bc in self.wall:
            old = g.clone()
            hit, inner = [], []
            for k in range(lat.Q):
                i = self.nb[lat.rev[k], nodes]
                hit.append((self.nb[k, nodes] == -1) & (i != -1))
                inner.append(i.clamp(min=0).long())
            rnd = None
            if bc.type == "fixedRandomT":
                # one draw per such link, node by node and link by link, of the host's rand()
                flags = torch.stack(hit).T.contiguous()
                draws = torch.zeros(flags.shape, dtype=torch.float64, device=g.device)
                draws[flags] = self._rand(int(flags.sum()))
                rnd = draws.T
            for k in range(lat.Q):
                if not bool(hit[k].any()):
                    continue
                sel = hit[k]
                i = inner[k][sel]
                U = [u[i] for u in self.U]
                Tw = torch.full_like(U[0], bc.value[0])
                if rnd is not None:
                    lo, hi = (bc.value[0] * (100 + s * bc.pert) / 100 for s in (-1, 1))
                    Tw = lo + (hi - lo) * rnd[k][sel]
                g[k, nodes[sel]] = self._geq(Tw, U)[k] + old[k, i] - self._geq(self.T[i], U)[k]

    def _rand(self, n):
        if not hasattr(self, "_draws") or self._draws.numel() != n:
            libc = ctypes.CDLL(None)
            libc.srand(0)
            self._draws = torch.tensor([libc.rand() / 2147483647.0 for _ in range(n)], dtype=torch.float64,
                                       device=self.rho.device)
        return self._draws

    def _heat(self):
        """With the new density and the old temperature and velocity."""
        lat, s = self.lat, self.s
        L3 = s.g_Lambda[3]
        if lat.three:
            lam = self.rho * s.Cv * (1 / L3 - 0.5) * (6 + 11 * s.g_alpha1 + s.g_alpha2) / 9
        else:
            lam = self.rho * s.Cv * (1 / L3 - 0.5) * (4 + 3 * s.g_alpha1 + 2 * s.g_alpha2) / 6
        dot, div = torch.zeros_like(self.rho), torch.zeros_like(self.rho)
        for d in range(3 if lat.three else 2):
            unit = np.eye(3, dtype=int)[d]
            up = int(np.where((lat.c == -unit).all(1))[0][0])     # upstream of -e is x + e
            dn = int(np.where((lat.c == unit).all(1))[0][0])
            scale = 0.5
            if not self.periodic:
                one = (self.nb[up] == -1) | (self.nb[dn] == -1)
                scale = torch.where(one, 1.0, 0.5)
            diff = lambda q: scale * (self.at(q, up) - self.at(q, dn))  # noqa: E731
            dot += diff(self.T) * diff(1 / self.rho)
            div += diff(self.U[d])
        dpdT = self.rho * s.R / (s.M - self.rho * s.b)
        return -lam * dot / s.Cv + div * self.T * (1 - dpdT / (self.rho * s.Cv))

    def step(self):
        lat = self.lat
        self.f = self._stream(self._collide_f())
        self._bounce(self.f)
        if self.thermal:
            self.g = self._stream(self._collide_g())
            self._wall_temperature(self.g)
        self.rho = self.f.sum(0)
        if self.thermal:
            self.S = self._heat()
            self.T = self.g.sum(0) + 0.5 * self.S
        self._force()
        F = self._total(self.rho)
        for d in range(3):
            j = sum(float(lat.c[k][d]) * self.f[k] for k in range(lat.Q) if lat.c[k][d])
            self.U[d] = (j + 0.5 * F[d]) / self.rho


def _exact_train(c, seed):
    dev = _device()
    X, Y, idx, p = _train_data(c, seed)
    X, Y, p = (torch.tensor(v, dtype=torch.float64, device=dev) for v in (X, Y, p))
    idx = torch.tensor(idx, dtype=torch.long, device=dev).reshape(c["iters"], c["batch"])
    m, v, hist = torch.zeros_like(p), torch.zeros_like(p), []
    layers = list(zip(WIDTHS[:-1], WIDTHS[1:]))
    for it in range(c["iters"]):
        x, t = X[idx[it]], Y[idx[it]]
        W, o = [], 0
        for a, b in layers:
            W.append((p[o:o + a * b].reshape(a, b), p[o + a * b:o + a * b + b]))
            o += a * b + b
        acts = [x]
        for n, (w, b) in enumerate(W):
            z = acts[-1] @ w + b
            acts.append(torch.tanh(z) if n < len(W) - 1 else z)
        d = acts[-1] - t
        hist.append((d * d).mean())
        dz = 2 * d / d.numel()
        grads = []
        for n in range(len(W) - 1, -1, -1):
            grads = [(acts[n].T @ dz).reshape(-1), dz.sum(0)] + grads
            if n:
                dz = (dz @ W[n][0].T) * (1 - acts[n] ** 2)
        g = torch.cat(grads)
        m = 0.9 * m + 0.1 * g
        v = 0.999 * v + 0.001 * g * g
        p = p - 1e-3 * (m / (1 - 0.9 ** (it + 1))) / ((v / (1 - 0.999 ** (it + 1))).sqrt() + 1e-8)
    return {"loss": torch.stack(hist), "params": p}


def _exact_batch(c, seed):
    dev = _device()
    lat = _Lattice(False, dev)
    cases = _batch_cases(c, seed)
    spec = CaseSpec(lbmodel=0, btype=3)
    out = [None] * len(cases)
    for L in sorted({L for L, _, _ in cases}):
        who = [k for k, v in enumerate(cases) if v[0] == L]
        one = _table({"box": "XY", "nx": L, "ny": L, "nz": 1}, lat, dev)
        nb = torch.cat([one + j * L * L for j in range(len(who))], dim=1)
        rho = torch.tensor(np.concatenate([cases[k][1] for k in who]), device=dev)
        T = torch.tensor(np.repeat([cases[k][2] for k in who], L * L), device=dev)
        e = _Exact(lat, nb, rho, [torch.zeros_like(rho) for _ in range(3)], T, spec, False)
        # initialisation leaves an ensemble at its first collision: one level behind the steps it counts
        for _ in range(c["steps"] + 1):
            e.step()
        for j, k in enumerate(who):
            out[k] = e.rho[j * L * L:(j + 1) * L * L]
    return {"rho": torch.cat(out)}


def exact(case, seed):
    c = case
    if c["kind"] == "train":
        return _exact_train(c, seed)
    if c["kind"] == "batch":
        return _exact_batch(c, seed)
    dev = _device()
    three = c["box"] in ("XYZ", "column3d")
    lat = _Lattice(three, dev)
    rho, U, T = _fields(c, seed)
    spec = _spec(c)
    wall = ()
    if c["box"].startswith("column"):
        plane = c["nx"] * c["ny"] if three else c["nx"]
        n = plane * (c["nz"] if three else c["ny"])
        name = "Z" if three else "Y"
        lo = torch.arange(plane, device=dev)
        wall = ((lo, spec.g_bc[name + "0"]), (lo + n - plane, spec.g_bc[name + "1"]))
    e = _Exact(lat, _table(c, lat, dev), rho, U.T.contiguous(), T, spec, c["thermal"], wall)
    for _ in range(c["steps"]):
        e.step()
    out = {"rho": e.rho, "U": torch.stack(e.U, 1)}
    if c["thermal"]:
        out["T"] = e.T
    return out
