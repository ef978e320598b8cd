"""The work that users of the hydro path have it do, as cases to be timed and compared.

A case names one call pattern of the public API with its sizes:

* ``step``: ``HydroStep.compute_forces`` (std-hydro force evaluation from unsorted particles),
  with ``integrate`` followed by ``HydroStep.integrate`` (a whole time step);
* ``ve``: ``VeHydroStep.compute_forces`` (the VE propagator), optionally with AV cleaning;
* ``density_op`` / ``momentum_energy_op``: the differentiable operators, forward and backward;
* ``search``: cornerstone tree from sorted keys, then ``find_neighbors`` with neighbor lists.

Workloads: ``turbulence`` (jittered periodic lattice, solenoidal-like velocities of a few
large modes, rms Mach 0.3), ``sedov`` (near-exact periodic lattice with a hot centre), ``evrard``
(open sphere, density ~ 1/r), ``uniform`` (random positions in a periodic box).  Smoothing
lengths scatter by 1 % around the value for ``ng`` neighbors, as they do in a running
simulation, whose updates depend on each particle's neighbor count.
"""
from __future__ import annotations

import math

import numpy as np
import torch

GAMMA = 5.0 / 3.0
DT = 1e-4  # the time step before the measured one (integration, AV switches)


def _case(name, kind, workload, n, precision, ng=100, ngmax=150, **kw):
    return dict(name=name, kind=kind, workload=workload, n=n, precision=precision, ng=ng, ngmax=ngmax, **kw)


def listed():
    return [
        # a small test problem stepped in time: launches and host reads count
        _case("small_step_mixed", "step", "uniform", 10_007, "mixed", integrate=True),
        # the Sedov blast at the classical 30^3, one FP64 time step
        _case("sedov30_fp64", "step", "sedov", 27_000, "fp64", integrate=True),
        # differentiable density on a 100^3 glass (one relaxation iteration: forward and backward)
        _case("density_op_fp64", "density_op", "turbulence", 1_000_000, "fp64", ngmax=256),
        # a plain neighbor search with lists, as an analysis of a snapshot makes it
        _case("search_fp64", "search", "uniform", 500_009, "fp64"),
        # uniform random particles with ~800 neighbors each, FP64
        _case("uniform800_fp64", "step", "uniform", 1_000_000, "fp64", ng=800, ngmax=1024, integrate=False),
        # one rank's share of a 256^3 run on 8 GPUs, a whole time step in the application's precision
        _case("turbulence128_mixed", "step", "turbulence", 128 ** 3, "mixed", integrate=True),
        # the default (VE) propagator at that size, mixed, and an odd size in FP64
        _case("ve128_mixed", "ve", "turbulence", 128 ** 3, "mixed", av_clean=False),
        _case("ve_uniform_fp64", "ve", "uniform", 1_000_003, "fp64", av_clean=False),
        # gradients of accelerations and energy rates with respect to positions
        _case("momentum_energy_op_mixed", "momentum_energy_op", "turbulence", 128 ** 3, "mixed", ngmax=256),
        # an Evrard-like collapse: open box, strongly varying density, counts up to ngmax
        _case("evrard4m_mixed", "step", "evrard", 4_194_304, "mixed", ngmax=512, integrate=False),
        # the headline workload, 256^3, in both precisions
        _case("turbulence256_mixed", "step", "turbulence", 256 ** 3, "mixed", integrate=False),
        _case("turbulence256_fp64", "step", "turbulence", 256 ** 3, "fp64", integrate=False),
    ]


def draw(rng):
    kind = rng.choices(["step", "ve", "density_op", "momentum_energy_op", "search"], [6, 3, 1, 1, 1])[0]
    workload = rng.choice(["turbulence", "uniform", "evrard"])
    precision = rng.choice(["mixed", "fp64"])
    top = {"step": 16_000_000, "ve": 6_000_000, "density_op": 4_000_000, "momentum_energy_op": 4_000_000,
           "search": 4_000_000}[kind]
    n = int(math.exp(rng.uniform(math.log(5_000), math.log(top))))
    if rng.random() < 0.5:
        n |= 1
    ng = 100
    if kind == "step" and workload == "uniform" and 100_000 < n < 1_500_000 and rng.random() < 0.4:
        ng = rng.choice([200, 400, 800])
    ngmax = {100: rng.choice([150, 256]), 200: 320, 400: 600, 800: 1024}[ng]
    if workload == "evrard":
        ngmax = 512
    elif kind.endswith("_op"):
        ngmax = 256
    c = dict(kind=kind, workload=workload, n=n, precision=precision, ng=ng, ngmax=ngmax)
    if kind == "step":
        c["integrate"] = rng.random() < 0.5
    if kind == "ve":
        c["av_clean"] = rng.random() < 0.3
    return c


# ------------------------------------------------------------------------------------- inputs
def _h0(n, ng, volume=1.0):
    return 0.5 * (3.0 * ng * volume / (4.0 * math.pi * n)) ** (1.0 / 3.0)


def _fields(case, seed):
    """(unsorted FP64 fields on the GPU, box limits (lo, hi) per dimension, periodic)."""
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(int(seed) % (1 << 31))
    n, w = case["n"], case["workload"]
    rand = lambda: torch.rand(n, dtype=torch.float64, device=dev, generator=g)
    randn = lambda: torch.randn(n, dtype=torch.float64, device=dev, generator=g)
    lo, hi, periodic = [0.0] * 3, [1.0] * 3, True
    u = torch.ones(n, dtype=torch.float64, device=dev)
    if w in ("turbulence", "sedov"):
        # n cells of a lattice of side^3 cells, in lattice order (all of them when n is a cube)
        side = math.ceil(round(n ** (1.0 / 3.0), 9))
        cell = torch.randperm(side ** 3, device=dev, generator=g)[:n].sort()[0] if n < side ** 3 else \
            torch.arange(n, device=dev)
        pos = [(c.double() + 0.5) / side for c in (cell // side ** 2, (cell // side) % side, cell % side)]
        # sedov: the lattice after its first steps, a thousandth of a cell from its sites
        pos = [torch.remainder(p + (0.1 if w == "turbulence" else 1e-3) / side * randn(), 1.0) for p in pos]
    elif w == "uniform":
        pos = [rand() for _ in range(3)]
    else:  # evrard
        r, ct, phi = rand().sqrt(), 2.0 * rand() - 1.0, 2.0 * math.pi * rand()
        st = (1.0 - ct * ct).sqrt()
        pos = [r * st * phi.cos(), r * st * phi.sin(), r * ct]
        lo, hi, periodic = [-1.0] * 3, [1.0] * 3, False
        u *= 0.05
    h = torch.full((n,), _h0(n, case["ng"]), dtype=torch.float64, device=dev)
    if w == "evrard":
        h = 0.5 * (1.5 * case["ng"] * r / n) ** (1.0 / 3.0)
        v = [-0.1 * p + 0.01 * randn() for p in pos]
    elif w == "sedov":
        # specific energy 1 in the centre over a cold gas; small random velocities
        r = sum((p - 0.5) ** 2 for p in pos).sqrt()
        inner = r < 0.1
        u = torch.where(inner, n / inner.sum().double(), torch.full_like(u, 1e-10))
        v = [1e-3 * randn() for _ in range(3)]
    elif w == "uniform":
        v = [0.1 * randn() for _ in range(3)]
    else:
        v = [torch.zeros_like(u) for _ in range(3)]
        gc = torch.Generator().manual_seed(int(seed) % (1 << 31))
        for _ in range(24):
            k = torch.randint(-3, 4, (3,), generator=gc).tolist()
            amp = (torch.randn(3, generator=gc) / (1.0 + sum(a * a for a in k))).tolist()
            ph = 2.0 * math.pi * (k[0] * pos[0] + k[1] * pos[1] + k[2] * pos[2] + float(torch.rand(1, generator=gc)))
            s = torch.sin(ph)
            for d in range(3):
                v[d] += amp[d] * s
        scale = 0.3 * math.sqrt(GAMMA * (GAMMA - 1.0)) / sum((a * a).mean() for a in v).sqrt()
        v = [a * scale for a in v]
    if w != "sedov":
        h = h * (1.0 + 0.01 * randn().clamp(-3.0, 3.0))
    f = dict(x=pos[0], y=pos[1], z=pos[2], h=h, m=torch.full_like(u, 1.0 / n), vx=v[0], vy=v[1], vz=v[2], u=u)
    return {k: t.contiguous() for k, t in f.items()}, (lo, hi, periodic), g


def _inputs(case, seed):
    """The fields in the case's precision (x, y, z always FP64) and everything else a call takes."""
    f, box, g = _fields(case, seed)
    dt = torch.float64 if case["precision"] == "fp64" else torch.float32
    rn = lambda: torch.randn(case["n"], dtype=torch.float64, device=f["x"].device, generator=g)
    if case["kind"] == "step" and case["integrate"]:
        # X_n - X_{n-1} and the last step's energy rate
        f["x_m1"], f["y_m1"], f["z_m1"] = (f[k] * DT for k in ("vx", "vy", "vz"))
        f["du_m1"] = 0.1 * rn()
    if case["kind"] == "ve":
        f["alpha"] = 0.05 + 0.5 * torch.rand(case["n"], dtype=torch.float64, device=f["x"].device, generator=g)
    if case["kind"] == "momentum_energy_op":
        # a state near equilibrium: rho = 1 or 1/r, ideal gas, near-isotropic IAD tensors
        rho = torch.ones_like(f["u"])
        if case["workload"] == "evrard":
            rho = 0.5 / math.pi / sum(f[k] ** 2 for k in "xyz").sqrt()
        f["rho"] = rho * (1.0 + 0.01 * rn())
        f["p"], f["c"] = f["rho"] * (GAMMA - 1.0) * f["u"], (GAMMA * (GAMMA - 1.0) * f["u"]).sqrt()
        iso = 4.9 / f["h"] ** 2
        for k in ("c11", "c22", "c33"):
            f[k] = iso * (1.0 + 0.02 * rn())
        for k in ("c12", "c13", "c23"):
            f[k] = iso * 0.02 * rn()
        for k in ("g_ax", "g_ay", "g_az", "g_du"):
            f[k] = rn()
    return {k: (t if k in ("x", "y", "z") else t.to(dt)) for k, t in f.items()}, box


_CTX = []


def _context():
    """The program's library handle: one for all states."""
    from sphexa_amd import hydro

    if not _CTX:
        _CTX.append(hydro.Context(0))
    return _CTX[0]


def prepare(case, seed):
    from sphexa_amd import autodiff, hydro
    from sphexa_amd._lib import BC_OPEN, BC_PERIODIC, FP64, MIXED

    ctx = _context()
    inp, (lo, hi, periodic) = _inputs(case, seed)
    box = hydro.make_box(lo, hi, BC_PERIODIC if periodic else BC_OPEN)
    prec = FP64 if case["precision"] == "fp64" else MIXED
    kind, n = case["kind"], case["n"]
    s = dict(case=case, ctx=ctx, inp=inp, box=box)
    if kind == "step":
        s["step"] = hydro.HydroStep(ctx, n, box, prec, ng0=case["ng"], ngmax=case["ngmax"])
        if case["integrate"]:
            s["step"].d.allocate(ctx.device, integration=True)
    elif kind == "ve":
        s["step"] = hydro.VeHydroStep(ctx, n, box, prec, av_clean=case["av_clean"], ng0=case["ng"],
                                      ngmax=case["ngmax"])
    elif kind == "density_op":
        s["op"] = autodiff.DensityOp(ctx, box, prec, ngmax=case["ngmax"])
        s["leaves"] = [inp[k].requires_grad_(True) for k in ("x", "y", "z", "h")]
    elif kind == "momentum_energy_op":
        s["op"] = autodiff.MomentumEnergyOp(ctx, box, prec, ngmax=case["ngmax"])
        s["leaves"] = [inp[k].requires_grad_(True) for k in ("x", "y", "z")]
        s["fields"] = {k: inp[k] for k in autodiff._ME_FIELDS}
    else:
        # a snapshot: particles in SFC order with their keys
        keys = hydro.compute_sfc_keys(ctx, inp["x"], inp["y"], inp["z"], box)
        order = hydro.sequence(ctx, n)
        hydro.sort_by_key(ctx, keys, order)
        s["sorted"] = [hydro.gather(ctx, order, inp[k].double().contiguous()) for k in ("x", "y", "z", "h")]
        s["keys"] = keys
    return s


STD = ("rho", "p", "c", "c11", "c12", "c13", "c22", "c23", "c33", "ax", "ay", "az", "du", "h")
MOVED = ("x", "y", "z", "x_m1", "y_m1", "z_m1", "vx", "vy", "vz", "u")
VE = ("xm", "kx", "gradh", "prho", "divv", "curlv", "alpha")


def run(state):
    from sphexa_amd import hydro

    case = state["case"]
    kind = case["kind"]
    if kind == "step":
        step = state["step"]
        d = step.compute_forces(state["inp"])
        out = {k: getattr(d, k) for k in STD}
        out["nc"], out["order"], out["keys"] = d.nc, step.order, step.keys
        if case["integrate"]:
            ts = step.integrate(hydro.TimestepState(minDt=DT, minDt_m1=DT), remove_unconverged=True)
            out.update({k: getattr(d, k) for k in MOVED})
            out["minDt"] = ts.minDt
        return out
    if kind == "ve":
        step = state["step"]
        d = step.compute_forces(state["inp"], dt=DT)
        out = {k: getattr(d, k) for k in STD}
        out.update({k: getattr(step.ve, k) for k in VE})
        out["nc"], out["order"], out["minDtRho"] = d.nc, step.order, step.minDtRho
        return out
    if kind == "density_op":
        i = state["inp"]
        rho = state["op"](i["x"], i["y"], i["z"], i["h"], i["m"])
        loss = ((rho.double() - rho.detach().double().mean()) ** 2).sum()
        g = torch.autograd.grad(loss, state["leaves"])
        return dict(rho=rho.detach(), gx=g[0], gy=g[1], gz=g[2], gh=g[3])
    if kind == "momentum_energy_op":
        i = state["inp"]
        o = state["op"](i["x"], i["y"], i["z"], **state["fields"])
        g = torch.autograd.grad(o, state["leaves"], [i[k] for k in ("g_ax", "g_ay", "g_az", "g_du")])
        o = [t.detach() for t in o]
        return dict(ax=o[0], ay=o[1], az=o[2], du=o[3], gx=g[0], gy=g[1], gz=g[2])
    ctx, (x, y, z, h) = state["ctx"], state["sorted"]
    tree = hydro.tree_from_keys(ctx, state["keys"], state["box"])
    nb, nc = hydro.find_neighbors(ctx, x, y, z, h, state["box"], tree, case["ngmax"])
    return dict(nb=nb, nc=nc, leaves=tree.leaves, layout=tree.layout)


def work(case):
    """Inputs read once, outputs written once; flops of the pair loops and of one distance test per
    neighbor (19 density, 37 IAD, 121 momentum-energy, 11 per test; the VE loops 19, 35, 37, 40,
    40 and 130; adjoints twice their loops)."""
    n, ng = case["n"], case["ng"]
    s = 8 if case["precision"] == "fp64" else 4
    pairs = float(n) * ng
    kind = case["kind"]
    if kind == "step":
        return dict(bytes=n * (24 + 6 * s + 14 * s + 16 + (24 + 11 * s if case["integrate"] else 0)),
                    flops=pairs * (11 + 19 + 37 + 121))
    if kind == "ve":
        return dict(bytes=n * (24 + 7 * s + 21 * s + 8), flops=pairs * (11 + 19 + 35 + 37 + 40 + 40 + 130))
    if kind == "density_op":
        return dict(bytes=n * (24 + 2 * s + s + 24 + s), flops=pairs * (2 * 11 + 19 + 2 * 19))
    if kind == "momentum_energy_op":
        return dict(bytes=n * (24 + 14 * s + 4 * s + 4 * s + 24), flops=pairs * (2 * 11 + 121 + 2 * 121))
    return dict(bytes=n * (32 + 8 + 4 * min(ng, case["ngmax"])), flops=pairs * 11)


# ------------------------------------------------------------------------------------- in 64 bits
CHUNK = 1 << 24


def _hilbert(ix, iy, iz):
    """64-bit Hilbert keys of integer coordinates on 21 levels (the framework's curve)."""
    digit = torch.tensor([0, 1, 3, 2, 7, 6, 4, 5], device=ix.device)
    key = torch.zeros_like(ix)
    for level in range(20, -1, -1):
        a, b, c = (ix >> level) & 1, (iy >> level) & 1, (iz >> level) & 1
        key = (key << 3) + digit[(a << 2) | (b << 1) | c]
        na, nb, nc = 1 - a, 1 - b, 1 - c
        px, py, pz = ix ^ -(a & (nb | c)), iy ^ -((a & (b | c)) | (b & nc)), iz ^ -((a & nb & nc) | (b & nc))
        turn, swap = c == 1, (c == 0) & (b == 0)
        ix = torch.where(turn, py, torch.where(swap, pz, px))
        iy = torch.where(turn, pz, py)
        iz = torch.where(turn, px, torch.where(swap, px, pz))
    return key


def _order(x, y, z, lo, hi):
    c = []
    for p, l, u in zip((x, y, z), lo, hi):
        m = 2097152.0 * (1.0 / (u - l))
        c.append((torch.floor(p * m) - l * m).long().clamp(max=(1 << 21) - 1))
    return torch.argsort(_hilbert(*c), stable=True)


class _Pairs:
    """Ordered neighbor pairs (i, j): |x_i - x_j| < 2 h_i, j != i, by a cell grid."""

    def __init__(self, x, lo, hi, periodic):
        self.x, self.lo, self.hi, self.periodic = x, lo, hi, periodic
        self.len = [u - l for l, u in zip(lo, hi)]

    def grid(self, hmax):
        self.m = [max(1, min(int(L / (2.0 * hmax * 1.0001)), 512)) for L in self.len]
        if self.periodic and min(self.m) < 3:
            self.m = [1, 1, 1]
        c = [((p - l) / L * m).long().clamp(0, m - 1) for p, l, L, m in zip(self.x, self.lo, self.len, self.m)]
        self.cell3 = c
        cell = (c[0] * self.m[1] + c[1]) * self.m[2] + c[2]
        self.perm = torch.argsort(cell)
        cnt = torch.bincount(cell, minlength=self.m[0] * self.m[1] * self.m[2])
        self.start = torch.cat([cnt.new_zeros(1), cnt.cumsum(0)])

    def offsets(self, i, j):
        r = [p[i] - p[j] for p in self.x]
        if self.periodic:
            r = [a - L * torch.round(a / L) for a, L in zip(r, self.len)]
        return r

    def of(self, targets, h):
        """Chunks of (targets, j[row, k], mask[row, k]): each row a target's neighbors, padded with
        the target itself."""
        shifts = [(a, b, c) for a in (-1, 0, 1) for b in (-1, 0, 1) for c in (-1, 0, 1)] if max(self.m) > 1 \
            else [(0, 0, 0)]
        n = self.x[0].numel()
        step = max(64, int(CHUNK / (max(1.0, n / len(self.start)) * len(shifts))))
        k = 0
        while k < targets.numel():
            t = targets[k:k + step]
            first, count = [], []
            for sh in shifts:
                c = [self.cell3[d][t] + sh[d] for d in range(3)]
                if self.periodic:
                    ok, c = torch.ones_like(t, dtype=torch.bool), [a % m for a, m in zip(c, self.m)]
                else:
                    ok = sum(((a < 0) | (a >= m)).int() for a, m in zip(c, self.m)) == 0
                    c = [a.clamp(0, m - 1) for a, m in zip(c, self.m)]
                cell = (c[0] * self.m[1] + c[1]) * self.m[2] + c[2]
                first.append(self.start[cell])
                count.append(torch.where(ok, self.start[cell + 1] - self.start[cell], 0))
            first, count = torch.stack(first, 1).reshape(-1), torch.stack(count, 1).reshape(-1)
            total = int(count.sum())
            if total > 4 * CHUNK and step > 64:
                step = max(64, step // 4)  # a dense region
                continue
            row = torch.repeat_interleave(torch.arange(t.numel(), device=t.device).repeat_interleave(len(shifts)),
                                          count, output_size=total)
            j = self.perm[torch.repeat_interleave(first - (count.cumsum(0) - count), count, output_size=total) +
                          torch.arange(total, device=t.device)]
            i = t[row]
            r = self.offsets(i, j)
            hit = ((r[0] * r[0] + r[1] * r[1] + r[2] * r[2] < 4.0 * h[i] * h[i]) & (i != j)).nonzero()[:, 0]
            row, j = row[hit], j[hit]
            cnt = torch.bincount(row, minlength=t.numel())
            kmax = int(cnt.max())
            col = torch.arange(row.numel(), device=t.device) - (cnt.cumsum(0) - cnt)[row]
            nb = t[:, None].int().repeat(1, kmax)
            nb[row, col] = j.int()
            yield t, nb, torch.arange(kmax, device=t.device)[None, :] < cnt[:, None]
            k += t.numel()


def _neighbors(f, box, h, ng0, ngmax, h32):
    """Neighbor rows with the smoothing-length iteration: (chunks of _Pairs.of, h, nc counting self)."""
    lo, hi, periodic = box
    P = _Pairs([f["x"], f["y"], f["z"]], lo, hi, periodic)
    h = h.clone()
    nc = torch.zeros(h.numel(), dtype=torch.long, device=h.device)
    todo = torch.arange(h.numel(), device=h.device)
    for k in range(11 if ng0 else 1):
        P.grid(float(h.max()))
        got = list(P.of(todo, h))
        for t, _, mask in got:
            nc[t] = mask.sum(1) + 1
        chunks = got if k == 0 else chunks + got
        out = ((ng0 // 4 > nc) | (nc - 1 > ngmax)).nonzero()[:, 0] if ng0 else todo[:0]
        if out.numel() == 0 or k == 10:
            break
        new = h[out] * 0.5 * (1.0 + 1023.0 * ng0 / nc[out].double()) ** 0.1
        h[out] = new.float().double() if h32 else new
        # the rows of the particles searched again are dropped
        stale = torch.zeros_like(nc, dtype=torch.bool)
        stale[out] = True
        chunks = [(t[~stale[t]], nb[~stale[t]], mask[~stale[t]]) if bool(stale[t].any()) else (t, nb, mask)
                  for t, nb, mask in chunks]
        todo = out
    return P, chunks, h, nc


def _kernel(n=6):
    """K and the table-linear kernel W(v) with its slope, and its derivative table's lookup."""
    v = np.arange(20000) * (2.0 / 19999)
    pv = 0.5 * np.pi * v
    s = np.where(v > 0, np.sin(pv) / np.where(v > 0, pv, 1.0), 1.0)
    ds = np.where(v > 0, (np.cos(pv) - s) / np.where(v > 0, v, 1.0), 0.0)
    q = np.linspace(0.0, 2.0, 2001)
    sq = np.where(q > 0, np.sin(0.5 * np.pi * q) / np.where(q > 0, 0.5 * np.pi * q, 1.0), 1.0)
    fq = 4.0 * np.pi * q * q * sq ** n
    K = 1.0 / (1e-3 / 3.0 * (fq[0] + fq[-1] + 4.0 * math.fsum(fq[1::2]) + 2.0 * math.fsum(fq[2:-1:2])))
    tab, der = torch.from_numpy(s ** n).cuda(), torch.from_numpy(n * s ** (n - 1) * ds).cuda()

    def look(t, v):
        k = (v.detach() * (19999 / 2.0)).long()
        inside = k < 19999
        k = k.clamp(max=19998)
        w0 = t[k]
        w = w0 + (t[k + 1] - w0) * (19999 / 2.0) * (v - k.double() * (2.0 / 19999))
        return torch.where(inside, w, torch.zeros_like(w))

    return K, lambda v: look(tab, v), lambda v: look(der, v)


class _Sum:
    """Per-particle sums over the neighbor rows."""

    def __init__(self, P, h, chunks):
        self.P, self.h, self.chunks = P, h, chunks

    def each(self):
        """(i[rows, 1], j[rows, k], mask, offsets r_ij, |r_ij|); padding has a harmless offset."""
        for t, nb, mask in self.chunks:
            rows = max(1, CHUNK // max(1, nb.shape[1]))
            for a in range(0, t.numel(), rows):
                i, j, w = t[a:a + rows, None], nb[a:a + rows].long(), mask[a:a + rows]
                r = [torch.where(w, q, self.h[i]) for q in self.P.offsets(i, j)]
                yield i, j, w, r

    def __call__(self, terms, k):
        out = [torch.zeros_like(self.h) for _ in range(k)]
        for i, j, w, r in self.each():
            for o, t in zip(out, terms(i, j, w, r)):
                o[i[:, 0]] = torch.where(w, t, torch.zeros_like(t)).sum(1)
        return out


def _max_row(into, i, w, v):
    into[i[:, 0]] = torch.maximum(into[i[:, 0]], torch.where(w, v, torch.zeros_like(v)).amax(1)) if v.shape[1] \
        else into[i[:, 0]]


def _dist(r):
    return (r[0] ** 2 + r[1] ** 2 + r[2] ** 2).sqrt()


def _iad(S, h, vol, K, W):
    def terms(i, j, mask, r):
        w = vol[j] * W(_dist(r) / h[i])
        return [r[0] * r[0] * w, r[0] * r[1] * w, r[0] * r[2] * w, r[1] * r[1] * w, r[1] * r[2] * w, r[2] * r[2] * w]

    a, b, c, d, e, g = (t / h ** 2 for t in S(terms, 6))  # in units of h^2
    det = a * d * g + 2.0 * b * e * c - a * e * e - d * c * c - g * b * b
    q = h / (det * K)
    return [(d * g - e * e) * q, (c * e - g * b) * q, (b * e - d * c) * q, (a * g - c * c) * q, (c * b - a * e) * q,
            (a * d - b * b) * q]


def _sym(c, q, r):
    return (c[0][q] * r[0] + c[1][q] * r[1] + c[2][q] * r[2], c[1][q] * r[0] + c[3][q] * r[1] + c[4][q] * r[2],
            c[2][q] * r[0] + c[4][q] * r[1] + c[5][q] * r[2])


def _me_pair(i, j, r, f, h, m, rho, p, c, cs, W):
    """The std momentum-energy terms of pairs with offsets r, and the signal velocity."""
    dist = _dist(r)
    v = [f[k][i] - f[k][j] for k in ("vx", "vy", "vz")]
    Wi, Wj = W(dist / h[i]) / h[i] ** 3, W(dist / h[j]) / h[j] ** 3
    Ai, Aj = _sym(cs, i, r), _sym(cs, j, r)
    w = (r[0] * v[0] + r[1] * v[1] + r[2] * v[2]) / dist
    cc = c[i] + c[j]
    pi = 0.5 * torch.where(w < 0, -(0.5 * cc - 2.0 * w) * w, torch.zeros_like(w))
    mp, mr, mW = m[j] * p[i] / rho[i] ** 2, m[i] / rho[i], m[j] / rho[j] * Wj
    a, b = Wi * (mp + pi * mr), mW * (p[j] / rho[j] + pi)
    a2, b2 = Wi * (2.0 * mp + pi * mr), pi * mW
    return [a * Ai[k] + b * Aj[k] for k in range(3)] + \
        [sum(v[k] * (a2 * Ai[k] + b2 * Aj[k]) for k in range(3))], cc - 3.0 * w


def _sorted_inputs(case, seed):
    inp, (lo, hi, periodic) = _inputs(case, seed)
    f = {k: t.double() for k, t in inp.items()}
    if not periodic:
        lo, hi = [float(f[k].min()) for k in "xyz"], [float(f[k].max()) for k in "xyz"]
    o = _order(f["x"], f["y"], f["z"], lo, hi)
    return {k: t[o] for k, t in f.items()}, (lo, hi, periodic), o


def exact(case, seed):
    if float(case["n"]) * case["ng"] > 1.2e9 or case["kind"] == "search":
        return None  # whole numbers, or too many pairs
    f, box, order = _sorted_inputs(case, seed)
    ng0 = (0 if case["kind"].endswith("_op") else case["ng"])
    K, W, dW = _kernel()
    P, chunks, h, nc = _neighbors(f, box, f["h"], ng0, case["ngmax"], case["precision"] != "fp64")
    S = _Sum(P, h, chunks)
    m, vel = f["m"], [f["vx"], f["vy"], f["vz"]]

    def back(t):  # to the caller's order
        out = torch.empty_like(t)
        out[order] = t
        return out

    if case["kind"] == "momentum_energy_op":
        cs = [f[k] for k in ("c11", "c12", "c13", "c22", "c23", "c33")]
        g = [f[k] for k in ("g_ax", "g_ay", "g_az", "g_du")]
        out = [torch.zeros_like(h) for _ in range(4)]
        grad = [torch.zeros_like(h) for _ in range(3)]
        sign = (K, K, K, -0.5 * K)
        for i, j, w, r in S.each():
            r = [a.requires_grad_(True) for a in r]
            t, _ = _me_pair(i, j, r, f, h, m, f["rho"], f["p"], f["c"], cs, W)
            t = [torch.where(w, a, torch.zeros_like(a)) for a in t]
            for o, a, s in zip(out, t, sign):
                o[i[:, 0]] = s * a.detach().sum(1)
            dr = torch.autograd.grad(sum((s * gg[i] * a).sum() for a, gg, s in zip(t, g, sign)), r)
            for o, d in zip(grad, dr):
                o[i[:, 0]] += d.sum(1)
                o.index_add_(0, j[w], -d[w])
        return dict(ax=back(out[0]), ay=back(out[1]), az=back(out[2]), du=back(out[3]), gx=back(grad[0]),
                    gy=back(grad[1]), gz=back(grad[2]))

    rho0 = m + S(lambda i, j, w, r: [m[j] * W(_dist(r) / h[i])], 1)[0]
    rho = rho0 * K / h ** 3
    if case["kind"] == "density_op":
        g = 2.0 * (rho - rho.mean())
        grad, gh = [torch.zeros_like(h) for _ in range(3)], -3.0 * rho / h * g
        for i, j, w, r in S.each():
            d = _dist(r)
            v = (d / h[i]).requires_grad_(True)
            slope = torch.autograd.grad(W(v).sum(), v)[0]
            q = torch.where(w, g[i] * K / h[i] ** 4 * m[j] * slope, torch.zeros_like(d))
            gh[i[:, 0]] -= (q * d / h[i]).sum(1)
            for o, a in zip(grad, r):
                o[i[:, 0]] += (q * a / d).sum(1)
                o.index_add_(0, j[w], -(q * a / d)[w])
        return dict(rho=back(rho), gx=back(grad[0]), gy=back(grad[1]), gz=back(grad[2]), gh=back(gh))

    tmp = f["u"] * (GAMMA - 1.0)
    none = dict(nc=None, order=None, keys=None)
    vmax = torch.zeros_like(h)
    if case["kind"] == "step":
        p, c = rho * tmp, (GAMMA * tmp).sqrt()
        cs = _iad(S, h, m / rho, K, W)

        def terms(i, j, w, r):
            t, signal = _me_pair(i, j, r, f, h, m, rho, p, c, cs, W)
            _max_row(vmax, i, w, signal)
            return t

        t = S(terms, 4)
        acc, du = [K * a for a in t[:3]], -0.5 * K * t[3]
        out = dict(zip(("rho", "p", "c", "c11", "c12", "c13", "c22", "c23", "c33", "ax", "ay", "az", "du"),
                       [rho, p, c] + cs + acc + [du]), h=h, **none)
        if case["integrate"]:
            courant = float(np.float32(0.2)) * h / torch.where(vmax > 0, vmax, c)
            dt = min(float(courant.min()), 1.1 * DT)
            for k, (q, a, u, l) in enumerate(zip("xyz", acc, box[1], box[0])):
                vn = f[q + "_m1"] / DT + 0.5 * DT * a
                dx = (vn + 0.5 * a * dt) * dt
                new = f[q] + dx
                if box[2]:
                    new = torch.where(new > u, new - (u - l), torch.where(new < l, new + (u - l), new))
                out[q], out[q + "_m1"], out["v" + q] = new, dx, vn + a * dt
            u = f["u"] + du * dt + 0.5 * (du - f["du_m1"]) / DT * dt * dt
            out["u"] = torch.where(u < 0, f["u"] * torch.exp(u * dt / f["u"]), u)
            out["h"] = h * 0.5 * (1.0 + 1023.0 * case["ng"] / nc.double()) ** 0.1
            out["minDt"] = dt
        return out

    # the VE propagator
    xm = m / rho
    none.pop("keys")

    def gradh_terms(i, j, mask, r):
        v = _dist(r) / h[i]
        w, d = W(v), dW(v)
        t = -(3.0 * w + v * d)
        return [w * xm[j], t * xm[j], t * m[j]]

    a, b, c0 = S(gradh_terms, 3)
    kx, wom, wr0 = (a + xm) * K / h ** 3, (b - 3.0 * xm) * K / h ** 4, (c0 - 3.0 * m) * K / h ** 4
    wom = wom * m / xm + (kx - K * xm / h ** 3) * wr0
    rho = kx * m / xm
    gradh = 1.0 + h / (3.0 * rho) * wom
    p, c = rho * tmp, (GAMMA * tmp).sqrt()
    prho = p / (kx * m * m * gradh)
    cs = _iad(S, h, xm / kx, K, W)

    def grad_terms(i, j, mask, r):
        w = W(_dist(r) / h[i])
        A = [-t * w for t in _sym(cs, i, r)]
        return [(q[j] - q[i]) * xm[j] * t for q in vel for t in A]

    d = [t * K / h ** 3 / kx for t in S(grad_terms, 9)]
    divv = d[0] + d[4] + d[8]
    curlv = ((d[7] - d[5]) ** 2 + (d[2] - d[6]) ** 2 + (d[3] - d[1]) ** 2).sqrt()
    dV = [d[0], d[1] + d[3], d[2] + d[6], d[4], d[5] + d[7], d[8]]
    vsig = 1e-40 * c

    def av_terms(i, j, mask, r):
        q = _dist(r)
        rv = sum(r[k] * (vel[k][i] - vel[k][j]) for k in range(3))
        _max_row(vsig, i, mask, torch.where(rv < 0, c[i] + c[j] - 3.0 * rv / q, torch.zeros_like(rv)))
        w = K / h[i] ** 3 * W(q / h[i]) * (xm / kx)[j] * (divv[i] - divv[j])
        return [-t * w for t in _sym(cs, i, r)]

    gd = S(av_terms, 3)
    ac = h * h * (gd[0] ** 2 + gd[1] ** 2 + gd[2] ** 2).sqrt()
    loc = torch.where(divv < 0, ac / (ac + h * divv.abs() + 0.05 * c), torch.zeros_like(ac))
    old = f["alpha"]
    rate = (torch.where(loc >= 0.05, loc, torch.full_like(loc, 0.05)) - old) * 0.2 * vsig / h
    alpha = torch.where(loc >= old, loc, old + rate * DT)
    eta = (32.0 * math.pi / 3.0 / nc.double()) ** (1.0 / 3.0)

    def me_terms(i, j, mask, r):
        q = _dist(r)
        v = [a[i] - a[j] for a in vel]
        v1, v2 = q / h[i], q / h[j]
        Wi, Wj = W(v1) / h[i] ** 3, W(v2) / h[j] ** 3
        A, B = [-t * Wi for t in _sym(cs, i, r)], [-t * Wj for t in _sym(cs, j, r)]
        rv = sum(a * b for a, b in zip(r, v))
        if case["av_clean"]:
            quad = lambda k: (r[0] * (dV[0][k] * r[0] + dV[1][k] * r[1] + dV[2][k] * r[2]) +
                              r[1] * (dV[3][k] * r[1] + dV[4][k] * r[2]) + dV[5][k] * r[2] * r[2])
            d1, d2 = quad(i), quad(j)
            e = torch.minimum(v1, v2) - eta[i]
            d3 = torch.where(e < 0, torch.exp(-(5.0 * e) ** 2), torch.ones_like(e))
            ab = torch.where(d2 != 0, d1 / d2, torch.zeros_like(d1))
            rv = rv - 0.5 * d3 * (4.0 * ab / (1.0 + ab) ** 2).clamp(0.0, 1.0) * (d1 + d2)
        w = rv / q
        cc = c[i] + c[j]
        visc = torch.where(w < 0, -((alpha[i] + alpha[j]) * 0.25 * cc - 2.0 * w) * w, torch.zeros_like(w))
        at = (rho[i] - rho[j]).abs() / (rho[i] + rho[j])
        s = (10.0 * (at - 0.1)).clamp(0.0, 1.0)
        ratio = (xm[j] / xm[i]) ** s
        am, bm = xm[i] ** 2 * ratio, xm[j] ** 2 / ratio
        av = [0.5 * visc * m[j] * (a / rho[i] + b / rho[j]) for a, b in zip(A, B)]
        mi, mj = m[j] * prho[i] * am, m[j] * prho[j] * bm
        return [mi * a + mj * b + x for a, b, x in zip(A, B, av)] + \
            [m[j] * am * sum(a * b for a, b in zip(v, A)), sum(a * b for a, b in zip(v, av))]

    t = S(me_terms, 5)
    du = K * (prho * t[3] + 0.5 * t[4].clamp(min=0.0))
    out = dict(zip(STD, [rho, p, c] + cs + [-K * a for a in t[:3]] + [du, h]), **none)
    out.update(zip(VE, [xm, kx, gradh, prho, divv, curlv, alpha]))
    out["minDtRho"] = 0.06 / abs(float(divv.max()))
    return out
