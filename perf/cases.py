"""Performance cases: what programs built on this framework have it do.

Each case is one pass of a program's main loop through the public entry
points, on inputs made from a seed:

  frame     a simulation frame: `substeps` substeps of one scene, then the
            download of its particles (FluidSystem::advance + exportToData)
  restart   as a frame, from a state the program hands over first
            (setupFromData)
  rollout   substeps on the program's own device arrays (lf_step_noalloc):
            tight loops that hold the state as tensors, from a given state
  batch     many scenes stepped together, then all their particles
  serve     a burst of jobs through the continuous-batching server

Fluids: `plain` is pressure and XSPH only (stiff Tait fluid, dt 1e-4), `full`
has every force term at the command-line driver's coefficients (adhesion 0.1,
viscosity 0.2, surface tension 1.0, damping 0.5).  Layouts: a jittered block
in the corner of its box, the double dam break of the driver, a block under a
spray layer, spray alone, and a finely spaced block whose stencil rows hold
more than 64 particles.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from libfluid_amd import Batch, Scene
from libfluid_amd import _lib as L
from libfluid_amd.scene import make_params
from libfluid_amd.serve import Server

DX, H = 0.01, 0.02


# -- the cases ---------------------------------------------------------------

def listed() -> list:
    return [
        # The command-line driver as it starts by default: 10,000 particles on
        # a 16^3 grid, every force term, one substep of 0.002 per frame, each
        # frame exported in cell order.
        dict(name="driver_default", kind="frame", layout="double_dam", fluid="full", n=10000, substeps=1, order="cell"),
        # A small device-resident roll-out: 2,000 particles, 20 substeps.
        dict(name="rollout_2k", kind="rollout", layout="block", fluid="plain", n=2000, substeps=20),
        # The largest double dam that the allocation-free entry point takes in
        # earnest, every force term; an odd count.
        dict(name="rollout_50k_full", kind="rollout", layout="double_dam", fluid="full", n=50001, substeps=20),
        # The 32,768-particle dam break, a frame of 100 substeps.
        dict(name="dam_32k", kind="frame", layout="block", fluid="plain", n=32768, substeps=100, order="id"),
        # A production double dam: 200,000 particles, every force term.
        dict(name="dam_200k_full", kind="frame", layout="double_dam", fluid="full", n=200000, substeps=40, order="id"),
        # The 1,048,576-particle collapsing column, a frame of 100 substeps.
        dict(name="column_1m", kind="frame", layout="block", fluid="plain", n=1048576, substeps=100, order="id"),
        # 8,388,608 particles: a block under a spray layer (dense and nearly
        # empty cells).
        dict(name="spray_8m", kind="frame", layout="block_spray", fluid="plain", n=8388608, substeps=40, order="id"),
        # Spray alone: a few neighbours each, near-isolated particles.
        dict(name="spray_262k", kind="frame", layout="spray", fluid="plain", n=262144, substeps=50, order="id"),
        # A finely spaced block (h/4, about 64 particles a cell), an edited
        # state handed over before each frame.
        dict(name="dense_100k", kind="restart", layout="dense", fluid="plain", n=100003, substeps=10, order="id"),
        # The batched workload: 256 uneven scenes of 2,048 to 65,536 particles.
        dict(name="batch_256", kind="batch", layout="block", fluid="plain", scenes=256, lo=2048, hi=65536, substeps=100),
        # A few small scenes, half of them with every force term.
        dict(name="batch_12_mixed", kind="batch", layout="block", fluid="mixed", scenes=12, lo=1500, hi=9000,
             substeps=50),
        # A burst of 40 jobs of 4,096 to 65,536 particles through the server.
        dict(name="serve_40", kind="serve", layout="block", fluid="plain", jobs=40, lo=4096, hi=65536, steps_lo=50,
             steps_hi=200),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["frame", "frame", "frame", "frame_full", "rollout", "rollout", "restart", "spray", "dense",
                       "batch", "serve"])
    if kind == "frame":
        return dict(kind="frame", layout="block", fluid="plain", n=_log_int(rng, 2000, 1500000),
                    substeps=rng.randint(10, 100), order=rng.choice(["id", "cell"]))
    if kind == "frame_full":
        return dict(kind="frame", layout="double_dam", fluid="full", n=_log_int(rng, 2000, 400000),
                    substeps=rng.randint(1, 40), order=rng.choice(["id", "cell"]))
    if kind == "rollout":
        full = rng.random() < 0.5
        return dict(kind="rollout", layout="double_dam" if full else "block", fluid="full" if full else "plain",
                    n=_log_int(rng, 500, 60000), substeps=rng.randint(4, 40))
    if kind == "restart":
        return dict(kind="restart", layout="block", fluid="plain", n=_log_int(rng, 2000, 500000),
                    substeps=rng.randint(5, 40), order="id")
    if kind == "spray":
        return dict(kind="frame", layout="spray", fluid="plain", n=_log_int(rng, 20000, 600000),
                    substeps=rng.randint(10, 60), order="id")
    if kind == "dense":
        return dict(kind="frame", layout="dense", fluid="plain", n=_log_int(rng, 5000, 200000),
                    substeps=rng.randint(5, 20), order="id")
    if kind == "batch":
        return dict(kind="batch", layout="block", fluid=rng.choice(["plain", "mixed"]),
                    scenes=_log_int(rng, 2, 64), lo=1000, hi=_log_int(rng, 4000, 65536), substeps=rng.randint(20, 100))
    return dict(kind="serve", layout="block", fluid="plain", jobs=_log_int(rng, 4, 40), lo=2048,
                hi=_log_int(rng, 8192, 65536), steps_lo=rng.randint(20, 60), steps_hi=rng.randint(61, 200))


# -- inputs ------------------------------------------------------------------

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _lattice(nx, ny, nz, spacing, origin, jitter, n, gen):
    """The first n points (x outermost) of a jittered lattice."""
    k = torch.arange(n, device="cuda", dtype=torch.int64)
    idx = torch.stack([k // (ny * nz), (k // nz) % ny, k % nz], 1).double()
    u = 2.0 * torch.rand(n, 3, generator=gen, device="cuda", dtype=torch.float64) - 1.0
    org = torch.tensor(origin, device="cuda", dtype=torch.float64)
    return (org + (idx + 0.5) * spacing + u * jitter).float()


def _plain(box, grid, h, spacing, gravity):
    return dict(rest_density=1000.0, gas_constant=2500.0, gamma=7.0, mass=1000.0 * spacing ** 3,
                particle_size=spacing / 2, xsph_scale=0.5, surface_tension=0.0, viscosity=0.0, adhesion=0.0,
                vel_limit=5.0, acc_limit=150.0, vdamp=0.5, gravity=tuple(gravity), h=h, inv_cell=(1.0 / h,) * 3,
                grid=tuple(grid), box=tuple(box))


def _full(p):
    """Every force term at the driver's coefficients, the driver's stiffness."""
    return dict(p, gas_constant=100.0, surface_tension=1.0, viscosity=0.2, adhesion=0.1)


def _scene(layout, fluid, n, gen, factor=(1.6, 1.6, 1.6), gravity=(0.0, -9.8, 0.0)):
    """(parameters, positions [n,3] on the GPU, substep length)."""
    if layout == "double_dam":
        # createFluidBlock's two blocks on the unit cube, the grid scaled with
        # the count so that cells hold as many particles as by default
        res = max(8, round(16 * (n / 1e4) ** (1 / 3)))
        ext, half = (0.33, 0.9, 0.33), (n // 2, n - n // 2)
        vol = ext[0] * ext[1] * ext[2] / half[1]
        s = 0.985 * vol ** (1 / 3)
        nx = max(1, int(ext[0] / s))
        nz = max(1, int(ext[2] / s))
        ny = -(-half[1] // (nx * nz))
        s = min(s, 0.98 / ny)
        pos = torch.cat([_lattice(nx, ny, nz, s, (0.0, 0.0, 0.0), 0.05 * s, half[0], gen),
                         _lattice(nx, ny, nz, s, (0.66, 0.0, 0.66), 0.05 * s, half[1], gen)])
        p = _full(_plain((1.0, 1.0, 1.0), (res,) * 3, 1.0 / res, s, gravity))
        return p, pos, 0.002 * 16.0 / max(res, 16)
    if layout == "spray":
        box = max(0.2, 1.28 * (n / 262144) ** (1 / 3))
        g = math.ceil(box / H)
        lo, hi = 0.08 * box, 0.92 * box
        pos = (lo + (hi - lo) * torch.rand(n, 3, generator=gen, device="cuda", dtype=torch.float64)).float()
        return _plain((box,) * 3, (g,) * 3, H, DX, gravity), pos, 1e-4
    if layout == "block_spray":
        side = round((n * 0.8984 / 0.449) ** (1 / 3))
        ny = round(0.449 * side)
        nb = side * ny * side
        ext = side * DX
        block = _lattice(side, ny, side, DX, (0.0, 0.0, 0.0), 0.05 * DX, nb, gen)
        u = torch.rand(n - nb, 3, generator=gen, device="cuda", dtype=torch.float64)
        lo = torch.tensor([0.0, 0.586, 0.0], device="cuda", dtype=torch.float64) * ext
        hi = torch.tensor([1.0, 0.976, 1.0], device="cuda", dtype=torch.float64) * ext
        g = math.ceil(ext / H - 1e-9)
        return _plain((ext,) * 3, (g,) * 3, H, DX, gravity), torch.cat([block, (lo + (hi - lo) * u).float()]), 1e-4
    if layout == "dense":
        s = 0.25 * H
        side = math.ceil(n ** (1 / 3))
        box = (0.6 + side * s,) * 3
        pos = _lattice(side, side, side, s, (0.203, 0.107, 0.111), 0.05 * s, n, gen)
        return _plain(box, [math.ceil(b / H) for b in box], H, s, gravity), pos, 1e-4
    if n == 1048576:  # the column's own block: 128 x 64 x 128
        nx, ny, nz, factor = 128, 64, 128, (2.0, 2.0, 2.0)
    else:
        nx = nz = math.ceil(n ** (1 / 3))
        ny = math.ceil(n / (nx * nz))
    box = [k * DX * f for k, f in zip((nx, ny, nz), factor)]
    p = _plain(box, [math.ceil(b / H - 1e-9) for b in box], H, DX, gravity)
    pos = _lattice(nx, ny, nz, DX, (0.0, 0.0, 0.0), 0.05 * DX, n, gen)
    return (_full(p) if fluid == "full" else p), pos, 1e-4


def _many(case, seed):
    """The scenes of a batch or a burst of jobs, and the jobs' step counts:
    counts log-uniform, each its own box and gravity direction."""
    rng = np.random.Generator(np.random.PCG64(seed))
    gen = _generator(seed)
    out = []
    for k in range(case.get("scenes") or case["jobs"]):
        # the counts are part of the case, the particles of the seed
        shape = np.random.Generator(np.random.PCG64([case["lo"], case["hi"], k]))
        n = int(round(math.exp(shape.uniform(math.log(case["lo"]), math.log(case["hi"])))))
        factor = shape.uniform(1.5, 2.5, 3)
        steps = int(shape.integers(case["steps_lo"], case["steps_hi"] + 1)) if "jobs" in case else 0
        g = rng.normal(size=3)
        g *= 9.8 / np.linalg.norm(g)
        fluid = "full" if case["fluid"] == "mixed" and k % 2 else "plain"
        p, pos, dt = _scene("block", fluid, n, gen, tuple(factor), tuple(g))
        out.append((p, pos, dt, steps))
    return out


def _cells(p):
    return p["grid"][0] * p["grid"][1] * p["grid"][2]


# -- the pass ----------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    if kind in ("batch", "serve"):
        scenes = _many(case, seed)
        host = [(make_params(**p), pos.cpu().numpy(), dt, steps) for p, pos, dt, steps in scenes]
        slots = sum((len(pos) + 511) // 512 * 512 for _, pos, _, _ in host)
        cells = sum(_cells(p) + 1 for p, _, _, _ in scenes)
        if kind == "serve":
            # room for about half of the burst at a time
            need = max((len(pos) + 511) // 512 * 512 for _, pos, _, _ in host)
            most = max(_cells(p) + 1 for p, _, _, _ in scenes)
            return dict(case=case, jobs=host, server=Server(max(need, slots // 2), max(most, cells // 2), len(host)))
        b = Batch(slots, cells, len(host))
        ids = []
        for p, pos, dt, _ in host:
            ids.append(b.add(p, len(pos), dt))
            b.upload(ids[-1], pos)
        return dict(case=case, batch=b, ids=ids)
    p, pos, dt = _scene(case["layout"], case["fluid"], case["n"], _generator(seed))
    params = make_params(**p)
    st = dict(case=case, params=params, dt=dt, order=L.LF_ORDER_CELL if case.get("order") == "cell" else L.LF_ORDER_ID)
    if kind == "rollout":
        zero = torch.zeros_like(pos)
        st["init"] = (pos, zero, zero.clone())
        st["state"] = tuple(torch.empty_like(pos) for _ in range(3))
        return st
    st["scene"] = Scene(params, len(pos))
    if kind == "restart":
        st["pos"], st["vel"] = pos.cpu().numpy(), np.zeros((len(pos), 3), np.float32)
    else:
        st["scene"].upload(pos.cpu().numpy())
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "rollout":
        for a, b in zip(st["state"], st["init"]):
            a.copy_(b)
        x, v, a = st["state"]
        k = case["substeps"]
        L.check(L.lib.lf_step_noalloc(ctypes.byref(st["params"]), x.shape[0], st["dt"] * k, k, x.data_ptr(),
                                      v.data_ptr(), a.data_ptr(), torch.cuda.current_stream().cuda_stream),
                "lf_step_noalloc")
        return dict(pos=x, vel=v, acc=a)
    if kind == "batch":
        b = st["batch"]
        b.step(case["substeps"])
        got = [b.download(i) for i in st["ids"]]
        return {k: np.concatenate([g[k] for g in got]) for k in ("pos", "vel")}
    if kind == "serve":
        s = st["server"]
        ids = [s.submit(p, pos, None, dt, steps) for p, pos, dt, steps in st["jobs"]]
        left = set(ids)
        got = {}
        while left:
            if s.tick():
                for j in s.take_finished():
                    got[j] = s.result(j)
                    left.discard(j)
        return {k: np.concatenate([got[j][k] for j in ids]) for k in ("pos", "vel")}
    sc = st["scene"]
    if kind == "restart":
        sc.upload(st["pos"], st["vel"])
    sc.step(st["dt"] * case["substeps"], case["substeps"])
    return sc.download(st["order"])


# -- what a pass cannot do without ---------------------------------------------

def work(case):
    """Per substep each particle's state (position in two words per axis,
    velocity, acceleration) is read and written once, and each of its
    neighbours within h costs about 10 operations in the density, 30 (60 with
    every force term) in the forces and 20 in XSPH; the program's own arrays
    cross once."""
    def one(n, substeps, fluid, layout, out):
        per_h3 = {"double_dam": 12.4, "dense": 64.0, "spray": 1.5}.get(layout, 8.0)
        nb = per_h3 * 4.19
        return np.array([n * (96.0 * substeps + out), n * substeps * nb * (90.0 if fluid == "full" else 60.0)])

    if case["kind"] in ("batch", "serve"):
        total = np.zeros(2)
        for k in range(case.get("scenes") or case["jobs"]):
            shape = np.random.Generator(np.random.PCG64([case["lo"], case["hi"], k]))
            n = int(round(math.exp(shape.uniform(math.log(case["lo"]), math.log(case["hi"])))))
            shape.uniform(1.5, 2.5, 3)
            steps = int(shape.integers(case["steps_lo"], case["steps_hi"] + 1)) if "jobs" in case else case["substeps"]
            full = case["fluid"] == "mixed" and k % 2
            total += one(n, steps, "full" if full else "plain", "block", 24.0 if "scenes" in case else 36.0)
    else:
        out = {"rollout": 72.0, "restart": 76.0}.get(case["kind"], 52.0)
        total = one(case["n"], case["substeps"], case["fluid"], case["layout"], out)
    return {"bytes": float(total[0]), "flops": float(total[1])}


# -- the same in 64 bits -------------------------------------------------------

def _sdf(p, x):
    half = torch.tensor([0.5 * float(np.float32(b)) for b in p["box"]], device=x.device, dtype=torch.float64)
    q = (x - half).abs() - half
    return q.max(1).values.clamp(max=0.0) + q.clamp(min=0.0).norm(dim=1)


def _wall_normal(p, x):
    e = float(np.float32(1e-4))
    n = torch.empty_like(x)
    for a in range(3):
        d = torch.zeros(3, device=x.device, dtype=torch.float64)
        d[a] = e
        n[:, a] = _sdf(p, x + d) - _sdf(p, x - d)
    return n / n.norm(dim=1, keepdim=True)


def _neighbours(x, radius, reach):
    """[n, k] matrix of the other points within `radius` (padded with n)."""
    n = x.shape[0]
    c = torch.floor(x / reach).long()
    c -= c.min(0).values - 1
    g = c.max(0).values + 2
    key = (c[:, 2] * g[1] + c[:, 1]) * g[0] + c[:, 0]
    order = torch.argsort(key)
    cells = int(g[0] * g[1] * g[2])
    count = torch.bincount(key, minlength=cells)
    start = torch.cumsum(count, 0) - count
    most = int(count.max())
    per, chunk = [], max(1, 60_000_000 // (27 * most))
    off = torch.tensor([(dz * int(g[1]) + dy) * int(g[0]) + dx for dz in (-1, 0, 1) for dy in (-1, 0, 1)
                        for dx in (-1, 0, 1)], device=x.device)
    slot = torch.arange(most, device=x.device)
    for i0 in range(0, n, chunk):
        i = torch.arange(i0, min(n, i0 + chunk), device=x.device)
        k = key[i][:, None] + off
        s = start[k][:, :, None] + slot
        ok = (slot < count[k][:, :, None]).reshape(len(i), -1)
        j = order[s.clamp(max=n - 1).reshape(len(i), -1)]
        ok &= ((x[j] - x[i][:, None]).square().sum(2) < radius * radius) & (j != i[:, None])
        width = int(ok.sum(1).max())
        j = torch.where(ok, j, torch.full_like(j, n))
        per.append(torch.sort(j, 1).values[:, :max(width, 1)])
    width = max(t.shape[1] for t in per)
    return torch.cat([torch.nn.functional.pad(t, (0, width - t.shape[1]), value=n) for t in per])


def _simulate(p, pos, vel, dt, substeps):
    """`substeps` WCSPH substeps of length dt in 64 bits: (pos, vel, acc,
    colour)."""
    f = lambda v: float(np.float32(v))  # noqa: E731  parameters are held in 32 bits
    h, m, rho0, eps = f(p["h"]), f(p["mass"]), f(p["rest_density"]), float(np.finfo(np.float32).tiny)
    pi = 3.141592654
    c6, cg6, cgs = 315 / (64 * pi * h ** 9), -945 / (32 * pi * h ** 9), -45 / (pi * h ** 6)
    K, gamma, sigma, nu, alpha = (f(p[k]) for k in ("gas_constant", "gamma", "surface_tension", "viscosity", "adhesion"))
    psize, alim, vlim, vdamp, xs = (f(p[k]) for k in ("particle_size", "acc_limit", "vel_limit", "vdamp", "xsph_scale"))
    grav = torch.tensor([f(g) for g in p["gravity"]], device=pos.device, dtype=torch.float64)
    h2 = float(np.float32(np.float32(h) * np.float32(h)))
    x, v = pos.double(), vel.double()
    a = torch.zeros_like(x)
    n = x.shape[0]
    pad = lambda t: torch.cat([t, torch.zeros_like(t[:1])])  # noqa: E731
    reach = 1.15 * h
    list_at = J = None

    def pairs(x, sl):  # of the points sl: x_j - x_i, r^2 and whether within h
        j = J[sl]
        d = pad(x)[j] - x[sl][:, None]
        rr = d.square().sum(2)
        return j, d, rr, (j < n) & (rr <= h2)

    def chunks():
        step = max(1, 40_000_000 // J.shape[1])
        return [slice(i, min(n, i + step)) for i in range(0, n, step)]

    for _ in range(substeps):
        if J is None or float((x - list_at).norm(dim=1).max()) > 0.07 * h:
            J, list_at = _neighbours(x, reach, reach), x.clone()
        total = torch.empty(n, device=x.device, dtype=torch.float64)
        for sl in chunks():
            _, _, rr, ok = pairs(x, sl)
            total[sl] = torch.where(ok, m * c6 * (h * h - rr).clamp(min=0.0) ** 3, 0.0 * rr).sum(1)
        t = _sdf(p, x).abs() / h
        edge = 128 - 315 * t + t ** 3 * (420 - 378 * t ** 2 + t ** 4 * (180 - 35 * t ** 2))
        fixed = total + torch.where(t < 1, rho0 * f(0.0039062) * edge, 0.0 * t)
        rho = torch.where(total == 0, torch.full_like(total, rho0), fixed)
        prs = torch.where(fixed == 0, 0.0 * fixed, K * rho0 / gamma * ((fixed / rho0) ** gamma - 1))
        cs = K * (fixed / rho0) ** (gamma - 1)
        normal = torch.zeros_like(x)
        if sigma:
            for sl in chunks():
                j, d, rr, ok = pairs(x, sl)
                ok &= (rr > eps) & (pad(rho)[j] > eps)
                w = torch.where(ok, m * cg6 * (h * h - rr).clamp(min=0.0) ** 2 / pad(rho)[j].clamp(min=eps), 0.0 * rr)
                normal[sl] = -h * (w[..., None] * d).sum(1)
        force = torch.zeros_like(x)
        for sl in chunks():
            j, d, rr, ok = pairs(x, sl)
            rj, ri = pad(rho)[j], rho[sl][:, None]
            ok &= (rr > eps) & (rj > eps)
            r = torch.where(ok, rr, torch.full_like(rr, h * h)).sqrt()
            rj = torch.where(ok, rj, torch.full_like(rj, rho0))
            mid = pad(prs)[j] / ri ** 2 + prs[sl][:, None] / rj ** 2
            com = torch.where(ok, m * cgs * (h - r).clamp(min=0.0) ** 2 / r, 0.0 * r)
            total3 = ((com * mid)[..., None] * d).sum(1)
            force[sl] += total3
            if nu:
                u = -((v[sl][:, None] - pad(v)[j]) * d).sum(2)
                mu = h * u / (rr + 0.01 * h2)
                visc = torch.where(u < 0, -nu * (cs[sl][:, None] + pad(cs)[j]) * mu / (ri + rj), 0.0 * u)
                force[sl] += nu * ((com * (mid + visc))[..., None] * d).sum(1)
            if sigma:
                b = (h - r).clamp(min=0.0) ** 3 * r ** 3
                coh = torch.where(r > 0.5 * h, b, 2 * b - h ** 6 * f(0.0156))
                coh = torch.where(ok & (r < h), -m * m * coh / r, 0.0 * r)
                curv = torch.where(ok[..., None], normal[sl][:, None] - pad(normal)[j], 0.0 * d)
                force[sl] += sigma * rho0 / ri * ((coh[..., None] * d) - sigma * m * curv).sum(1)
        if alpha:
            z = -_sdf(p, x).clamp(max=0.0) * 0.25 / psize
            at = (z < 1).nonzero()[:, 0]
            s = alpha * rho[at] / rho0 / (1 - z[at]) ** 3
            force[at] += s[:, None] * _wall_normal(p, x[at])
        new = force * m + grav
        new = new * (alim / new.norm(dim=1, keepdim=True).clamp(min=alim))
        x = x + v * dt + 0.5 * a * dt * dt
        v = v + 0.5 * (a + new) * dt
        v = v * (vlim / v.norm(dim=1, keepdim=True).clamp(min=vlim))
        a = new
        dist = _sdf(p, x)
        at = (dist > -psize).nonzero()[:, 0]
        w = _wall_normal(p, x[at])
        x[at] -= (dist[at] + psize)[:, None] * w
        v[at] -= (1 + vdamp) * (w * v[at]).sum(1, keepdim=True) * w
        blend = torch.empty_like(v)
        for sl in chunks():
            j, d, rr, ok = pairs(x, sl)
            both = rho[sl][:, None] + pad(rho)[j]
            w = torch.where(ok & (both > eps), c6 * (h * h - rr).clamp(min=0.0) ** 3 * 2 * m / both, 0.0 * rr)
            blend[sl] = (w[..., None] * (pad(v)[j] - v[sl][:, None])).sum(1)
        v = v + xs * blend
    q = (rho / rho0)[:, None]
    one, zero = torch.ones_like(q), torch.zeros_like(q)
    colour = torch.where(q < 1, torch.cat([zero, q, 1 - q], 1),
                         torch.where(q < 2, torch.cat([q - 1, 2 - q, zero], 1), torch.cat([one, zero, zero], 1)))
    return x, v, a, colour


def exact(case, seed):
    kind = case["kind"]
    if kind in ("batch", "serve"):
        scenes = _many(case, seed)
        if sum(len(s[1]) * (s[3] or case["substeps"]) for s in scenes) > 6e6 or len(scenes) > 16:
            return None  # too long
        got = [_simulate(p, pos, torch.zeros_like(pos), float(np.float32(dt)), steps or case["substeps"])
               for p, pos, dt, steps in scenes]
        return dict(pos=torch.cat([g[0] for g in got]), vel=torch.cat([g[1] for g in got]))
    if case.get("order") == "cell" or case["n"] * case["substeps"] > 2e7:
        return None  # the order needs 32-bit cell keys; too long
    p, pos, dt = _scene(case["layout"], case["fluid"], case["n"], _generator(seed))
    k = case["substeps"]
    part = float(np.float32(np.float32(dt * k) / np.float32(k)))
    x, v, a, colour = _simulate(p, pos, torch.zeros_like(pos), part, k)
    if kind == "rollout":
        return dict(pos=x, vel=v, acc=a)
    return dict(pos=x, colour=colour, vel=v, acc=a, ids=None)
