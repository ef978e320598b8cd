"""The neighbor search where its FP32 test can go wrong, against the oracle, bit for bit: ties
at exactly d = 2h, coincident particles, positions far from the origin, extreme units, radii
mixed within a group, boxes without a single nearest image, lists cut at ngmax, and particle
counts around the sizes of quarters, batches and groups."""
import numpy as np
import pytest
import torch

import oracle
from tests.helpers import uniform_box

pytestmark = pytest.mark.gpu

CPU = oracle.Cpu("oracle")


@pytest.fixture(scope="module")
def ctx():
    from sphexa_amd import hydro

    c = hydro.Context(0)
    yield c
    c.close()


def u32(t):
    return t.cpu().numpy().view(np.uint32)


def dev(a, dtype=torch.float64):
    return torch.from_numpy(np.ascontiguousarray(a)).to(dtype).to("cuda")


def cloud(n, ng=60, periodic=True, lo=0.0, hi=1.0, seed=3):
    inp, box = uniform_box(n, seed=seed, ng=ng, periodic=periodic, lo=lo, hi=hi)
    return np.stack([inp["x"], inp["y"], inp["z"]], 1), inp["h"], box


def lattice(side, shift, radius_cells):
    c = (np.arange(side) + shift) / side
    p = np.stack(np.meshgrid(c, c, c, indexing="ij"), -1).reshape(-1, 3)
    return p, np.full(len(p), 0.5 * radius_cells / side), oracle.Box.cube(0.0, 1.0, oracle.BC_PERIODIC)


def make(case):
    rng = np.random.default_rng(5)
    kind, arg = case
    if kind == "n":
        return cloud(arg, ng=30, periodic=arg % 2 == 0)
    if kind == "ties":  # 1/16 cells: exact distances, spheres through many lattice points
        return lattice(16, 0.5, arg)
    if kind == "near_ties":  # the same, each distance off by its own rounding
        return lattice(15, 0.37, arg)
    if kind == "coincident":
        p, h, box = cloud(3000)
        p[1::3] = p[::3]
        return p, h, box
    if kind == "offset":
        return cloud(5000, lo=arg, hi=arg + 1.0)
    if kind == "units":
        return cloud(5000, lo=-0.5 * arg, hi=0.5 * arg)
    if kind == "mixed_h":
        p, h, box = cloud(5000)
        return p, h * 10.0 ** rng.uniform(-1.0, 0.4, len(h)), box
    if kind == "zero_h":
        p, h, box = cloud(2000)
        h[rng.random(len(h)) < 0.5] = 0.0
        return p, h, box
    if kind == "wide":  # 2h from a fifth of the box to over its half
        p, h, box = cloud(1500)
        return p, np.full(len(h), arg), box
    if kind == "blob":  # one dense blob: groups of few particles beside full ones
        p = np.clip(0.5 + 0.02 * rng.standard_normal((6000, 3)), 0.0, 1.0)
        return p, np.full(6000, 0.003), oracle.Box.cube(0.0, 1.0, oracle.BC_OPEN)
    if kind == "levels":  # density ~ r^-2: a group's candidate leaves are of many levels, and hundreds
        d = rng.standard_normal((20000, 3))
        r = 0.499 * rng.random((20000, 1))
        return 0.5 + r * d / np.linalg.norm(d, axis=1, keepdims=True), np.full(20000, arg), oracle.Box.cube(0.0, 1.0)


CASES = [("n", k) for k in (1, 2, 16, 17, 63, 64, 65, 130, 4097)] + [
    ("ties", 2.0), ("ties", 3.0), ("near_ties", 2.0), ("near_ties", 3.0), ("coincident", 0), ("offset", 1e3),
    ("offset", 1e8), ("units", 1e-18), ("units", 1e17), ("mixed_h", 0), ("zero_h", 0), ("wide", 0.1), ("wide", 0.2),
    ("wide", 0.24), ("wide", 0.3), ("blob", 0), ("levels", 0.005), ("levels", 0.03)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}-{c[1]}")
@pytest.mark.parametrize("entry", ["plain", "fp64", "mixed", "cut"])
def test_search_bit_exact(ctx, case, entry):
    from sphexa_amd import hydro
    from sphexa_amd._lib import FP64, MIXED

    print("case search", case, entry, flush=True)
    p, h, box = make(case)
    n = len(p)
    keys = CPU.sfc_keys(*(np.ascontiguousarray(p[:, d]) for d in range(3)), box)
    keys, order = CPU.sort_by_key(keys, np.arange(n, dtype=np.uint32))
    x, y, z = (np.ascontiguousarray(p[order, d]) for d in range(3))
    h = np.ascontiguousarray(h[order])
    if entry == "mixed":
        h = h.astype(np.float32).astype(np.float64)
    gbox = hydro.make_box([box.xmin, box.ymin, box.zmin], [box.xmax, box.ymax, box.zmax], [box.bx, box.by, box.bz])
    t = hydro.tree_from_keys(ctx, torch.from_numpy(keys.view(np.int64)).to("cuda"), gbox, 64)
    rt = CPU.tree(keys, box)
    ngmax = 12 if entry == "cut" else min(n, 3000)
    ref, ref_nc = CPU.find_neighbors(x, y, z, h, box, rt, ngmax)
    if entry in ("plain", "cut"):
        nb, nc = hydro.find_neighbors(ctx, dev(x), dev(y), dev(z), dev(h), gbox, t, ngmax)
        nb, nc = u32(nb), u32(nc)
        assert np.array_equal(nc, ref_nc)
    if entry in ("fp64", "mixed", "cut"):
        prec = MIXED if entry == "mixed" else FP64
        ng0 = min(4, ngmax)
        d = hydro.ParticlesData(n, prec, ng0=ng0, ngmax=ngmax)
        d.x, d.y, d.z, d.h = dev(x), dev(y), dev(z), dev(h, torch.float32 if prec == MIXED else torch.float64)
        d.allocate("cuda")
        hydro.find_neighbors_sfc(ctx, d, gbox, t)
        if entry == "cut":
            # the first check is of the plain entry; this one iterates h and keeps the first ngmax
            assert all(np.array_equal(nb[i, :c], ref[i, :c]) for i, c in enumerate(np.minimum(nc, ngmax)))
            ref, ref_nc, h = CPU.find_neighbors_sph(x, y, z, h, box, rt, ng0, ngmax)
            assert np.array_equal(d.h.cpu().numpy(), h)
            ref_nc = ref_nc - 1
        nb, nc = u32(hydro.export_neighbors(ctx, d)), u32(d.nc) - 1
        assert np.array_equal(nc, ref_nc)
    bad = [i for i, c in enumerate(np.minimum(nc, ngmax)) if not np.array_equal(nb[i, :c], ref[i, :c])]
    assert not bad, bad[:10]


def not_a_number(n, rng):
    """Particles whose values a test replaces: first, middle and last lanes of groups and quarters, a whole
    group, some at random; half of their NaN have the sign bit."""
    bad = np.zeros(n, bool)
    bad[[0, 5, 64 + 15, 64 + 16, 128 + 63, 192]] = True
    bad[256:320] = True
    bad |= rng.random(n) < 0.02
    nan = np.where(rng.random(n) < 0.5, np.nan, -np.nan)
    return bad, nan


def search_both(ctx, x, y, z, h, box, keys, entry, ngmax, ng0=4):
    """(lists, counts) of the device, of the oracle, for sorted particles with a tree from `keys`."""
    from sphexa_amd import hydro
    from sphexa_amd._lib import FP64, MIXED

    n = len(x)
    gbox = hydro.make_box([box.xmin, box.ymin, box.zmin], [box.xmax, box.ymax, box.zmax], [box.bx, box.by, box.bz])
    t = hydro.tree_from_keys(ctx, torch.from_numpy(keys.view(np.int64)).to("cuda"), gbox, 64)
    ref, ref_nc = CPU.find_neighbors(x, y, z, h, box, CPU.tree(keys, box), ngmax)
    if entry == "plain":
        nb, nc = hydro.find_neighbors(ctx, dev(x), dev(y), dev(z), dev(h), gbox, t, ngmax)
        return u32(nb), u32(nc), ref, ref_nc
    prec = MIXED if entry == "mixed" else FP64
    d = hydro.ParticlesData(n, prec, ng0=ng0, ngmax=ngmax)
    d.x, d.y, d.z, d.h = dev(x), dev(y), dev(z), dev(h, torch.float32 if prec == MIXED else torch.float64)
    d.allocate("cuda")
    hydro.find_neighbors_sfc(ctx, d, gbox, t)
    return u32(hydro.export_neighbors(ctx, d)), u32(d.nc) - 1, ref, ref_nc


def sorted_cloud(n, entry, **kw):
    p, h, box = cloud(n, **kw)
    keys, order = CPU.sort_by_key(CPU.sfc_keys(*(np.ascontiguousarray(p[:, d]) for d in range(3)), box),
                                  np.arange(n, dtype=np.uint32))
    x, y, z = (np.ascontiguousarray(p[order, d]) for d in range(3))
    h = h[order]
    return x, y, z, h.astype(np.float32).astype(np.float64) if entry == "mixed" else h, box, keys


def assert_same_lists(which, nb, nc, ref, ref_nc):
    assert np.array_equal(nc[which], ref_nc[which])
    bad = [i for i in np.flatnonzero(which) if not np.array_equal(nb[i, :nc[i]], ref[i, :nc[i]])]
    assert not bad, bad[:10]


@pytest.mark.parametrize("n", [60, 3000])  # a tree of one leaf, leaves of several levels
@pytest.mark.parametrize("entry", ["plain", "fp64", "mixed"])
def test_neighbors_of_targets_beside_nan_smoothing_lengths(ctx, entry, n):
    """A target with h = NaN leaves the lists of its group's other targets as they are."""
    print("case nan h", entry, n, flush=True)
    x, y, z, h, box, keys = sorted_cloud(n, entry, ng=40)
    bad, nan = not_a_number(3000, np.random.default_rng(2))
    bad, nan = bad[:n], nan[:n]
    h[bad] = nan[bad]
    assert_same_lists(~bad, *search_both(ctx, x, y, z, h, box, keys, entry, min(n, 400)))


@pytest.mark.parametrize("entry", ["plain", "fp64", "mixed"])
def test_targets_with_nan_smoothing_lengths_have_no_neighbors(ctx, entry):
    """h = NaN, of either sign: d^2 < (2h)^2 holds for no candidate."""
    print("case nan h targets", entry, flush=True)
    x, y, z, h, box, keys = sorted_cloud(3000, entry, ng=40)
    bad, nan = not_a_number(3000, np.random.default_rng(2))
    h[bad] = nan[bad]
    nb, nc, ref, ref_nc = search_both(ctx, x, y, z, h, box, keys, entry, 400)
    assert not ref_nc[bad].any()
    assert_same_lists(np.ones(3000, bool), nb, nc, ref, ref_nc)


@pytest.mark.parametrize("periodic", [False, True])
@pytest.mark.parametrize("entry", ["plain", "fp64", "mixed"])
def test_particles_with_nan_positions_are_no_neighbors(ctx, entry, periodic):
    """A NaN coordinate, of either sign, in the tree's range of some leaf: no target's neighbor, and none itself."""
    print("case nan positions", entry, periodic, flush=True)
    x, y, z, h, box, keys = sorted_cloud(3000, entry, ng=40, periodic=periodic)
    bad, nan = not_a_number(3000, np.random.default_rng(4))
    for d, a in enumerate((x, y, z)):
        some = np.flatnonzero(bad)[d::3]
        a[some] = nan[some]
    nb, nc, ref, ref_nc = search_both(ctx, x, y, z, h, box, keys, entry, 400)
    assert not ref_nc[bad].any()
    assert_same_lists(np.ones(3000, bool), nb, nc, ref, ref_nc)


@pytest.mark.parametrize("entry", ["plain", "fp64", "mixed"])
@pytest.mark.parametrize("kind", ["outside", "tiny"])
def test_folded_candidates(ctx, entry, kind):
    """Targets at the faces of a periodic box.  outside: some particles lie up to a third of h outside of it;
    the predicate folds offsets for the targets whose sphere leaves the box, and for those only.  tiny: all
    particles within 1e-13 of a face, where folding rounds at 1e-3 of their distances."""
    print("case fold", entry, kind, flush=True)
    rng, n = np.random.default_rng(7), 3000
    p = rng.random((n, 3))
    h = np.full(n, 0.5 * (40 / (4 / 3 * np.pi * n)) ** (1 / 3))
    if kind == "outside":
        for i in np.flatnonzero(rng.random(n) < 0.05):
            p[i, rng.integers(0, 3)] = 1.0 + 0.02 * rng.random() if rng.random() < 0.5 else -0.02 * rng.random()
    else:
        p[:, 0] -= 0.5
        p *= 1e-13
        p[:, 0] += np.where(p[:, 0] < 0, 1.0, 0.0)
        h *= 1e-13
    if entry == "mixed":
        h = h.astype(np.float32).astype(np.float64)
    box = oracle.Box.cube(0.0, 1.0, oracle.BC_PERIODIC)
    keys, order = CPU.sort_by_key(CPU.sfc_keys(*(np.ascontiguousarray(p[:, d]) for d in range(3)), box),
                                  np.arange(n, dtype=np.uint32))
    x, y, z = (np.ascontiguousarray(p[order, d]) for d in range(3))
    h = np.ascontiguousarray(h[order])
    nb, nc, _, _ = search_both(ctx, x, y, z, h, box, keys, entry, 400)
    for i in range(n):
        d = [a - a[i] for a in (x, y, z)]
        if not all(a[i] - 2.0 * h[i] >= 0.0 and a[i] + 2.0 * h[i] <= 1.0 for a in (x, y, z)):
            d = [a - np.rint(a) for a in d]
        hit = d[0] * d[0] + d[1] * d[1] + d[2] * d[2] < 4.0 * h[i] * h[i]
        hit[i] = False
        assert np.array_equal(nb[i, :nc[i]], np.flatnonzero(hit)), i


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_groups_searched_again_need_counts_only(ctx, prec):
    """Initial h of five times as many neighbors as ngmax takes: every target's count exceeds it for some
    iterations, and h follows the oracle; none of those lists is searched by the slower exact kernel."""
    from sphexa_amd import hydro
    from sphexa_amd._lib import FP64, MIXED

    print("case h iteration", prec, flush=True)
    n, ng0, ngmax = 20000, 60, 100
    x, y, z, h, box, keys = sorted_cloud(n, prec, ng=500, periodic=False)
    gbox = hydro.make_box([box.xmin, box.ymin, box.zmin], [box.xmax, box.ymax, box.zmax], [box.bx, box.by, box.bz])
    t = hydro.tree_from_keys(ctx, torch.from_numpy(keys.view(np.int64)).to("cuda"), gbox, 64)
    d = hydro.ParticlesData(n, MIXED if prec == "mixed" else FP64, ng0=ng0, ngmax=ngmax)
    d.x, d.y, d.z, d.h = dev(x), dev(y), dev(z), dev(h, d.dtype)
    d.allocate("cuda")
    ctx.set_timing(True)
    try:
        ctx.timing_summary()
        hydro.find_neighbors_sfc(ctx, d, gbox, t)
        launches = {k: v[0] for k, v in ctx.timing_summary().items()}
    finally:
        ctx.set_timing(False)
    rt = CPU.tree(keys, box)
    nb, nc = u32(hydro.export_neighbors(ctx, d)), u32(d.nc)
    if prec == "fp64":
        _, ref_nc, ref_h = CPU.find_neighbors_sph(x, y, z, h, box, rt, ng0, ngmax)
        assert np.array_equal(d.h.cpu().numpy(), ref_h) and np.array_equal(nc, ref_nc)
    assert (nc <= ngmax + 1).all() and launches["nsCandidates"] > 2
    final, _ = CPU.find_neighbors(x, y, z, d.h.double().cpu().numpy(), box, rt, ngmax)
    bad = [i for i in range(n) if not np.array_equal(nb[i, :nc[i] - 1], final[i, :nc[i] - 1])]
    assert not bad, bad[:10]
    assert launches.get("nsCandidatesExact", 0) == 0
