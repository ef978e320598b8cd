"""The FP64 loops that interpolate the fitted kernel table (long lists) against the loops
that read the table itself, one lane per target in list order (SPHX_OPT_LOOP_SHAPE_FP64 = 1),
on the same particles.

Tolerances, fixed by rounding: a sum of 800 positive terms regrouped, over weights that agree
to 2^-48, differs by at most 800 * 2^-52 + 2^-48 = 2e-13 relative (rho, xm, kx: 1e-12); the
other fields are differences of such sums, bounded at 1e-10 of their largest magnitude as in
the other FP64 tests.
"""
import numpy as np
import pytest
import torch

from tests.helpers import uniform_box

pytestmark = pytest.mark.gpu

POSITIVE = ("rho", "xm", "kx")
GROUPS = (("ax", "ay", "az"), ("c11", "c22", "c33", "c12", "c13", "c23"))
STD = ("rho", "c11", "c12", "c13", "c22", "c23", "c33", "ax", "ay", "az", "du")
VE = ("xm", "kx", "gradh", "c11", "c12", "c13", "c22", "c23", "c33", "divv", "curlv", "alpha", "ax", "ay", "az", "du")


def field(step, f):
    owner = step.ve if hasattr(step, "ve") and hasattr(step.ve, f) and getattr(step.ve, f) is not None else step.d
    return getattr(owner, f).double().clone()


# smooth: the kernel's own tables, every segment fitted.  rough: entries perturbed by 1e-3,
# no segment reproduced by the fit.  patch: one perturbed entry in the first, a middle and
# the last (shortened) segment.
@pytest.mark.parametrize("table", ["smooth", "rough", "patch"])
@pytest.mark.parametrize("kind", ["std", "ve"])
@pytest.mark.parametrize("periodic", [True, False])
def test_fitted_table_loops_equal_table_loops(kind, table, periodic):
    from sphexa_amd import hydro
    from sphexa_amd._lib import FP64

    print("case", kind, table, periodic, flush=True)
    inp, b = uniform_box(330_007, seed=11, periodic=periodic, ng=800)
    box = hydro.make_box([b.xmin, b.ymin, b.zmin], [b.xmax, b.ymax, b.zmax], [b.bx, b.by, b.bz])
    fields = STD if kind == "std" else VE
    out = []
    for shape in (0, 1):
        ctx = hydro.Context(0)
        try:
            ctx.set_loop_shape(FP64, shape)
            make = hydro.HydroStep if kind == "std" else hydro.VeHydroStep
            step = make(ctx, len(inp["x"]), box, FP64, ng0=800, ngmax=1200)
            tables = [step.d.wh] + ([step.ve.whd] if kind == "ve" else [])
            for k, t in enumerate(tables):
                n = t.numel()
                noise = torch.from_numpy(np.random.default_rng(k).uniform(-1e-3, 1e-3, n)).to(t.device)
                if table == "rough":
                    t.add_(noise * t.abs().max())
                elif table == "patch":
                    for e in (3, n // 2, n - 2):
                        t[e] += noise[e] * t.abs().max()
            d_inp = {k: torch.from_numpy(np.ascontiguousarray(v)).to("cuda") for k, v in inp.items()}
            if kind == "ve":
                d_inp["alpha"] = torch.full_like(d_inp["x"], 0.3)
            step.compute_forces(d_inp)
            assert ctx.candidate_tests() >= 5e8  # the lists are long enough for the fitted form
            out.append({f: field(step, f) for f in fields})
            out[-1]["dt"] = step.d.minDtCourant
        finally:
            ctx.close()
    got, ref = out
    for f in fields:
        assert torch.isfinite(ref[f]).all(), f
        err = (got[f] - ref[f]).abs()
        if f in POSITIVE:
            assert (err / ref[f].abs()).max().item() < 1e-12, f
        else:
            group = next((g for g in GROUPS if f in g), (f,))
            assert err.max().item() < 1e-10 * max(ref[g].abs().max().item() for g in group), f
    assert abs(got["dt"] - ref["dt"]) < 1e-12 * ref["dt"]


# The mixed loops' window lists (ORed into LDS for records up to 32 bytes): empty chunks and
# lists, full chunks and windows, unions of one entry and of several windows, against the
# FP64-exact loops (one lane per target, no windows) on the same particles.  A wrong or missing
# slot changes a sum by a whole term; tolerances are those of the other mixed tests (rho, xm,
# kx 1e-5 relative, IAD 1e-4 of its largest diagonal).
@pytest.mark.parametrize("n,ng", [(1, 10), (2, 10), (63, 20), (64, 64), (65, 65), (300, 300), (1500, 4), (2000, 30),
                                  (2000, 1900)])
@pytest.mark.parametrize("kind", ["std", "ve"])
def test_mixed_window_lists(kind, n, ng):
    from sphexa_amd import hydro
    from sphexa_amd._lib import FP64, MIXED

    print("case lists", kind, n, ng, flush=True)
    inp, b = uniform_box(n, seed=17, periodic=n < 3, ng=ng)  # (an open box is fitted to the particles: n >= 3)
    inp = {k: v if k in "xyz" else v.astype(np.float32).astype(np.float64) for k, v in inp.items()}
    box = hydro.make_box([b.xmin, b.ymin, b.zmin], [b.xmax, b.ymax, b.zmax], [b.bx, b.by, b.bz])
    out = []
    for prec in (MIXED, FP64):
        ctx = hydro.Context(0)
        try:
            ctx.set_fp64_exact(True)
            make = hydro.HydroStep if kind == "std" else hydro.VeHydroStep
            step = make(ctx, n, box, prec, ng0=4, ngmax=max(4, n))
            dt = torch.float64 if prec == FP64 else torch.float32
            d_inp = {k: torch.from_numpy(np.ascontiguousarray(v)).to("cuda", torch.float64 if k in "xyz" else dt)
                     for k, v in inp.items()}
            if kind == "ve":
                d_inp["alpha"] = torch.full((n,), 0.25, dtype=dt, device="cuda")
            step.compute_forces(d_inp)
            out.append({f: field(step, f) for f in (("rho", "c11", "c22", "c33") if kind == "std" else ("xm", "kx"))})
            out[-1]["nc"] = step.d.nc.clone()
        finally:
            ctx.close()
    got, ref = out
    assert torch.equal(got["nc"], ref["nc"])
    for f in POSITIVE:
        if f in got:
            assert ((got[f] - ref[f]).abs() <= 1e-5 * ref[f]).all(), f
    # the IAD inverts its sums; compared where they are well determined
    well = ref["nc"] > 30
    if kind == "std" and well.any():
        scale = max(ref[f][well].abs().max().item() for f in ("c11", "c22", "c33"))
        for f in ("c11", "c22", "c33"):
            assert ((got[f] - ref[f])[well].abs() <= 1e-4 * scale).all(), f


@pytest.mark.parametrize("clean", [False, True])
@pytest.mark.parametrize("length", [1e-3, 1.0, 1e3])
def test_ve_pairs(length, clean):
    """VE pairs with a reciprocal square root for the division by |r| and (mixed) 1/h^3 in the records, in
    units of h from 1e-4 to 100 and with coincident particles (r = 0), against the FP64-exact loops.
    Mixed: the mode's tolerances; FP64: the suite's 1e-10, times 10 for the poles of prho (gradh = 0)."""
    from sphexa_amd import hydro
    from sphexa_amd._lib import FP64, MIXED

    print("case mixed ve pairs", length, clean, flush=True)
    n = 4096
    inp, b = uniform_box(n, seed=23, ng=100, hi=length)
    for k in "xyz":
        inp[k][1:400:2] = inp[k][0:400:2]
    inp["alpha"] = np.random.default_rng(23).uniform(0.05, 1.0, n)
    inp = {k: v if k in "xyz" else v.astype(np.float32).astype(np.float64) for k, v in inp.items()}
    box = hydro.make_box([b.xmin, b.ymin, b.zmin], [b.xmax, b.ymax, b.zmax], [b.bx, b.by, b.bz])
    out = []
    for prec, exact in ((MIXED, False), (FP64, False), (FP64, True)):
        ctx = hydro.Context(0)
        try:
            ctx.set_fp64_exact(exact)
            step = hydro.VeHydroStep(ctx, n, box, prec, grad_v=True, av_clean=clean, ng0=100)
            d_inp = {k: torch.from_numpy(np.ascontiguousarray(v)).to("cuda", torch.float64 if k in "xyz" else step.d.dtype)
                     for k, v in inp.items()}
            step.compute_forces(d_inp, dt=1e-4 * length)
            out.append({f: field(step, f) for f in ("divv", "curlv", "alpha", "ax", "ay", "az", "du")})
            dt = step.d.minDtCourant
        finally:
            ctx.close()
        out[-1]["minDt"] = torch.tensor(dt, dtype=torch.float64)
    ref = out.pop()
    for got, tol in zip(out, (2e-3, 1e-9)):
        for f in ref:
            scale = max(ref[k].abs().max() for k in GROUPS[0]) if f in GROUPS[0] else ref[f].abs().max()
            assert ((got[f] - ref[f]).abs() <= tol * scale).all(), (f, tol)


@pytest.mark.parametrize("n,ng", [(4096, 100), (330_007, 800)])  # FP64: the table itself, the fitted table
def test_coincident_particles_std(n, ng):
    """Pairs at distance 0 (W(0), no direction, no approach speed) add nothing but to the sums of W: against the
    FP64-exact loops.  FP64: the suite's 1e-10; mixed: the mode's 1e-3 (both of the largest value)."""
    from sphexa_amd import hydro
    from sphexa_amd._lib import FP64, MIXED

    print("case coincident std", n, flush=True)
    inp, b = uniform_box(n, seed=29, ng=ng)
    for k in "xyz":
        inp[k][1:400:2] = inp[k][0:400:2]
    inp = {k: v if k in "xyz" else v.astype(np.float32).astype(np.float64) for k, v in inp.items()}
    box = hydro.make_box([b.xmin, b.ymin, b.zmin], [b.xmax, b.ymax, b.zmax], [b.bx, b.by, b.bz])
    out = []
    for prec, exact in ((FP64, False), (MIXED, False), (FP64, True)):
        ctx = hydro.Context(0)
        try:
            ctx.set_fp64_exact(exact)
            step = hydro.HydroStep(ctx, n, box, prec, ng0=ng, ngmax=ng + ng // 2)
            d_inp = {k: torch.from_numpy(np.ascontiguousarray(v)).to("cuda", torch.float64 if k in "xyz" else step.d.dtype)
                     for k, v in inp.items()}
            step.compute_forces(d_inp)
            assert (ctx.candidate_tests() >= 5e8) == (ng == 800)
            out.append({f: field(step, f) for f in STD})
            out[-1]["minDt"] = torch.tensor(step.d.minDtCourant, dtype=torch.float64)
        finally:
            ctx.close()
    ref = out.pop()
    for got, tol in zip(out, (1e-10, 1e-3)):
        for f in ref:
            assert torch.isfinite(got[f]).all(), (f, tol)
            group = next((g for g in GROUPS if f in g), (f,))
            assert ((got[f] - ref[f]).abs() <= tol * max(ref[g].abs().max() for g in group)).all(), (f, tol)


# particle mass, box length, specific energy: p / (kx m^2) and 1/h^3 are within the FP32 range, their product is not
@pytest.mark.parametrize("mass,length,u", [(1e-9, 1e-4, 0.4), (1e15, 1e6, 1.0), (1.0 / 4096, 1.0, 1.0)])
@pytest.mark.parametrize("clean", [False, True])
def test_mixed_ve_units(mass, length, u, clean):
    """Mixed VE accelerations and energy rates in systems of units with small and large particle masses, against
    the FP64 loops; tolerance of the mode, 2e-3 of the largest value, as test_ve_pairs."""
    from sphexa_amd import hydro
    from sphexa_amd._lib import FP64, MIXED

    print("case ve units", mass, length, clean, flush=True)
    n = 4096
    inp, b = uniform_box(n, seed=31, ng=100, hi=length)
    inp["m"] = np.full(n, mass)
    inp["u"] = np.full(n, u)
    for k in ("vx", "vy", "vz"):
        inp[k] = inp[k] * np.sqrt(u)
    inp["alpha"] = np.random.default_rng(31).uniform(0.05, 1.0, n)
    inp = {k: v if k in "xyz" else v.astype(np.float32).astype(np.float64) for k, v in inp.items()}
    box = hydro.make_box([b.xmin, b.ymin, b.zmin], [b.xmax, b.ymax, b.zmax], [b.bx, b.by, b.bz])
    out = []
    for prec in (MIXED, FP64):
        ctx = hydro.Context(0)
        try:
            step = hydro.VeHydroStep(ctx, n, box, prec, grad_v=True, av_clean=clean, ng0=100)
            d_inp = {k: torch.from_numpy(np.ascontiguousarray(v)).to("cuda", torch.float64 if k in "xyz" else step.d.dtype)
                     for k, v in inp.items()}
            step.compute_forces(d_inp, dt=1e-4 * length)
            out.append({f: field(step, f) for f in ("prho", "ax", "ay", "az", "du")})
        finally:
            ctx.close()
    got, ref = out
    assert torch.isfinite(got["prho"]).all() and (got["prho"] != 0).all()  # the field itself is in range
    for f in ("ax", "ay", "az", "du"):
        scale = max(ref[k].abs().max() for k in GROUPS[0]) if f in GROUPS[0] else ref[f].abs().max()
        assert ((got[f] - ref[f]).abs() <= 2e-3 * scale).all(), f


def test_loop_form_follows_the_lists():
    """The FP64 loops' form (the table, or its fit) depends on the lists that they run on, not on what else the
    context searched: a plain search in between, and one of no targets, leave every bit as it is; a second set's
    short lists take the table, also where h iterated to them over longer ones."""
    from sphexa_amd import hydro
    from sphexa_amd._lib import FP64

    def lists_of(ctx, n, ng, start=1.0):
        inp, b = uniform_box(n, seed=37, ng=ng)
        t = {k: torch.from_numpy(v).to("cuda") for k, v in inp.items()}
        keys = hydro.compute_sfc_keys(ctx, t["x"], t["y"], t["z"], box)
        order = hydro.sequence(ctx, n)
        hydro.sort_by_key(ctx, keys, order)
        d = hydro.ParticlesData(n, FP64, ng0=ng, ngmax=ng + ng // 2)
        for f in ("x", "y", "z", "h", "m"):
            setattr(d, f, hydro.gather(ctx, order, t[f]))
        d.h *= start ** (1 / 3)
        d.allocate("cuda")
        tree = hydro.tree_from_keys(ctx, keys, box, 64)
        hydro.find_neighbors_sfc(ctx, d, box, tree)
        return d, tree

    print("case loop form", flush=True)
    ctx = hydro.Context(0)
    try:
        box = hydro.make_box(0.0, 1.0, 1)
        d, tree = lists_of(ctx, 330_007, 800)
        ctx.set_timing(True)

        def density():
            ctx.timing_summary()
            hydro.compute_density(ctx, d, box)
            return d.rho.clone(), "tableFitKernel" in ctx.timing_summary()

        rho, fitted = density()
        assert fitted
        for last in (100, 0):
            hydro.find_neighbors(ctx, d.x, d.y, d.z, d.h, box, tree, 16, 0, last)
            again, fitted = density()
            assert fitted and torch.equal(rho, again), last
        d, _ = lists_of(ctx, 1000, 50)
        assert not density()[1]
        d, _ = lists_of(ctx, 100_000, 500, start=2.6)
        assert ctx.candidate_tests() >= 5e8 and not density()[1]
    finally:
        ctx.close()


@pytest.mark.parametrize("kind", ["std", "ve"])
def test_fitted_table_at_the_rim(kind):
    """Targets whose neighbors all lie at 1.985 to 1.995 h, where W is 1e-14 of W(0), beside a cloud whose long
    lists take the fitted table: sums of such weights keep the relative accuracy that the table itself has (1e-10
    of the largest value among these targets, as for the others in test_fitted_table_loops_equal_table_loops; a
    distance rounds W by 6 * 2^-53 * 200 = 1e-13 there).  Not gradh, and a and du by it: 1 minus the own terms'
    share, 5e-11, is what rounding leaves of it in either form."""
    from sphexa_amd import hydro
    from sphexa_amd._lib import FP64

    print("case rim", kind, flush=True)
    inp, b = uniform_box(330_007, seed=41, periodic=False, ng=800)
    rng, side, h = np.random.default_rng(41), 8, 0.25 * inp["h"][0]
    grid = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3) * 1.99 * h
    grid += rng.uniform(-0.001, 0.001, grid.shape) * h + [0.3, 0.3, 1.5]
    k = len(grid)
    more = dict(x=grid[:, 0], y=grid[:, 1], z=grid[:, 2], h=np.full(k, h), m=np.full(k, inp["m"][0]), u=np.ones(k),
                **{v: rng.normal(0, 0.1, k) for v in ("vx", "vy", "vz")})
    inp = {f: np.concatenate([inp[f], more[f]]) for f in inp}
    n = len(inp["x"])
    out = []
    for shape in (0, 1):
        ctx = hydro.Context(0)
        try:
            ctx.set_loop_shape(FP64, shape)
            make = hydro.HydroStep if kind == "std" else hydro.VeHydroStep
            step = make(ctx, n, hydro.make_box([0.0] * 3, [1.0, 1.0, 2.0], 0), FP64, ng0=16, ngmax=1200)
            d_inp = {f: torch.from_numpy(np.ascontiguousarray(v)).to("cuda") for f, v in inp.items()}
            if kind == "ve":
                d_inp["alpha"] = torch.full_like(d_inp["x"], 0.3)
            step.compute_forces(d_inp)
            assert ctx.candidate_tests() >= 5e8
            rim = step.d.z > 1.2
            nc = step.d.nc[rim]
            assert rim.sum() == k and nc.min() == 4 and nc.max() == 7
            fields = STD if kind == "std" else [f for f in VE if f not in ("gradh", "ax", "ay", "az", "du")]
            out.append({f: field(step, f)[rim] for f in fields})
        finally:
            ctx.close()
    got, ref = out
    for f in got:
        group = next((g for g in GROUPS if f in g), (f,))
        scale = max(ref[g].abs().max().item() for g in group)
        err = (got[f] - ref[f]).abs().max().item() / scale
        assert np.isfinite(scale) and err <= 1e-10, (f, err)
