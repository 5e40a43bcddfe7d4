"""The workloads whose speed is measured, through the public Python interface.

A case is a dict of plain values; its "kind" picks what a pass does:

  frame      a whole small simulation step: index the moved points, radius
             neighbours of every point, k nearest of every point
  build      index new values, then a few thousand lookups in the new tree
  radius     neighbours of points within one radius (CSR), tree kept
  spheres    the same with a radius per query, queries that are not the
             indexed points
  nearest    k nearest of query points, with distances when asked for
  overlap    boxes against boxes (collision candidates)
  ray_first  the first k boxes along each ray
  ray_all    every box along each ray, ordered by distance
  energy     one molecular-dynamics step: neighbour list, Lennard-Jones
             energy and forces, backward included

Inputs are float32, made on the GPU from the seed alone: points uniform in
the unit cube or in 1000 Gaussian clusters, boxes with lognormal sides, rays
of which every fifth runs along an axis, jittered FCC lattices.

The number of results differs a little from seed to seed, so a pass returns
its CSR's offsets and the first and the last part of its indices, two views
of a length that the case fixes (about three quarters of what it expects),
which together are all of them.
"""
import math

import torch

import arborx_amd as ax

CENTRES, SIGMA = 1000, 0.01  # the Gaussian mixture
SIDE_MU, SIDE_SIGMA = math.log(0.002), 0.5  # lognormal box sides for 5M boxes
PROBES = 4096  # lookups that follow a build
CUTOFF, JITTER = 2.5, 0.05  # Lennard-Jones cutoff and lattice jitter (lattice distance 1)


def listed():
    return [
        # a small particle system rebuilt every step: launches and latency
        dict(name="frame_2k", kind="frame", n=1999, data="uniform", nodes="fp32", mean=32, k=8),
        # interactive picking in a kept scene: a handful of queries per call
        dict(name="nearest_300_of_1M", kind="nearest", n=1000003, nq=300, own=False,
             data="mixture", nodes="fp32", k=1, distances=True),
        # rebuilding the index of a large moving point set each step
        dict(name="build_points_10M", kind="build", n=10000000, geometry="points",
             data="uniform", nodes="q16"),
        # rebuilding a collision scene's index
        dict(name="build_boxes_1M", kind="build", n=1000000, geometry="boxes", data="uniform",
             nodes="fp32"),
        # fixed-radius neighbours of every point of a large uniform set
        dict(name="radius_10M", kind="radius", n=10000000, data="uniform", nodes="q16", mean=32),
        # clustered data with a smoothing length per query
        dict(name="spheres_clusters_700k", kind="spheres", n=1000003, nq=700001, data="mixture",
             nodes="fp32", mean=32),
        # k nearest of every point of a large set
        dict(name="nearest_10M_k16", kind="nearest", n=10000000, nq=10000000, own=True,
             data="uniform", nodes="q16", k=16, distances=False),
        # k nearest of other points, clustered, with distances (interpolation)
        dict(name="nearest_clusters_250k_k10", kind="nearest", n=300000, nq=250007, own=False,
             data="mixture", nodes="fp32", k=10, distances=True),
        # broad-phase collision detection
        dict(name="overlap_boxes_5M", kind="overlap", n=5000000, nq=5000000, nodes="q16"),
        # visibility: the first box along each ray
        dict(name="rays_first_1M", kind="ray_first", n=5000000, nq=1000000, nodes="fp32", k=1),
        # transmission: every box along each ray, in order
        dict(name="rays_all_200k", kind="ray_all", n=1000000, nq=200000, nodes="q16"),
        # a molecular-dynamics step on a 2M-atom crystal
        dict(name="md_step_2M", kind="energy", nx=80, ny=80, nz=78),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "build", "build", "radius", "radius", "spheres", "nearest",
                       "nearest", "overlap", "ray_first", "ray_all", "energy"])
    data = rng.choice(["uniform", "mixture"])
    nodes = rng.choice(["fp32", "q16"])
    if kind == "frame":
        return dict(kind=kind, n=_log_int(rng, 300, 30000), data="uniform", nodes=nodes,
                    mean=rng.choice([16, 32, 48]), k=rng.choice([1, 4, 8, 16]))
    if kind == "build":
        geometry = rng.choice(["points", "boxes"])
        return dict(kind=kind, n=_log_int(rng, 5000, 10000000 if geometry == "points" else 5000000),
                    geometry=geometry, data=data if geometry == "points" else "uniform",
                    nodes=nodes)
    if kind == "radius":
        return dict(kind=kind, n=_log_int(rng, 20000, 8000000), data=data, nodes=nodes,
                    mean=rng.choice([4, 16, 32, 60]) if data == "uniform" else 32)
    if kind == "spheres":
        n = _log_int(rng, 20000, 4000000)
        return dict(kind=kind, n=n, nq=_log_int(rng, 1000, n), data=data, nodes=nodes,
                    mean=rng.choice([8, 32]))
    if kind == "nearest":
        n = _log_int(rng, 20000, 5000000)
        own = rng.random() < 0.5
        return dict(kind=kind, n=n, nq=n if own else _log_int(rng, 100, n), own=own, data=data,
                    nodes=nodes, k=rng.choice([1, 3, 5, 8, 10, 16, 20, 32]),
                    distances=rng.random() < 0.5)
    if kind == "overlap":
        n = _log_int(rng, 20000, 5000000)
        return dict(kind=kind, n=n, nq=_log_int(rng, 1000, n), nodes=nodes)
    if kind == "ray_first":
        return dict(kind=kind, n=_log_int(rng, 20000, 5000000), nq=_log_int(rng, 1000, 500000),
                    nodes=nodes, k=rng.choice([1, 1, 4, 8]))
    if kind == "ray_all":
        return dict(kind=kind, n=_log_int(rng, 20000, 1000000), nq=_log_int(rng, 1000, 200000),
                    nodes=nodes)
    return dict(kind=kind, nx=rng.randint(8, 80), ny=rng.randint(8, 80), nz=rng.randint(8, 78))


# ------------------------------------------------------------ inputs
def _generator(seed, part):
    g = torch.Generator(device="cuda")
    g.manual_seed(1000003 * int(seed) + part)
    return g


def _rand(n, cols, g):
    return torch.rand((n, cols), generator=g, device="cuda", dtype=torch.float32)


def _points(data, n, seed, part):
    """n points; a mixture's centres depend on the seed only, so that queries
    and indexed points of one seed share their clusters."""
    g = _generator(seed, part)
    if data == "uniform":
        return _rand(n, 3, g)
    centres = _rand(CENTRES, 3, _generator(seed, 999))
    which = torch.arange(n, device="cuda") % CENTRES
    z = torch.randn((n, 3), generator=g, device="cuda", dtype=torch.float32)
    return (centres[which] + SIGMA * z).clamp_(0.0, 1.0)


def _radius(case):
    """Radius whose ball holds about case["mean"] of the case's points."""
    n, mean = case["n"], case["mean"]
    if case["data"] == "uniform":
        return (3.0 * mean / (4.0 * math.pi * n)) ** (1.0 / 3.0)
    per = n / CENTRES  # points of a cluster; density of the difference of two at 0
    return (3.0 * mean / (4.0 * math.pi * per)) ** (1.0 / 3.0) * math.sqrt(4.0 * math.pi) * SIGMA


def _box_scale(n):
    """Sides shrink with the spacing, so that the overlaps per box stay those
    of 5M boxes."""
    return (5000000.0 / n) ** (1.0 / 3.0)


def _boxes(n, of, seed, part):
    g = _generator(seed, part)
    c = _rand(n, 3, g)
    z = torch.randn((n, 3), generator=g, device="cuda", dtype=torch.float32)
    side = torch.exp(SIDE_MU + SIDE_SIGMA * z) * _box_scale(of)
    return torch.cat([c - 0.5 * side, c + 0.5 * side], dim=1).contiguous()


def _rays(n, seed, part):
    g = _generator(seed, part)
    o = _rand(n, 3, g) * 1.4 - 0.2
    d = torch.randn((n, 3), generator=g, device="cuda", dtype=torch.float32)
    i = torch.arange(n, device="cuda")
    along = i % 5 == 1
    other = torch.arange(3, device="cuda")[None, :] != ((i // 5) % 3)[:, None]
    d = torch.where(d == 0.0, torch.ones_like(d), d)  # no zero vectors
    d = torch.where(along[:, None] & other, torch.zeros_like(d), d)
    return ax.Rays(o, d)


def _lattice(case, seed):
    """FCC lattice (nx, ny, nz, 4, 3), nearest-neighbour distance 1, each
    coordinate moved by up to JITTER."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    edge = math.sqrt(2.0)
    basis = torch.tensor(_BASIS, device="cuda", dtype=torch.float64)
    axes = [torch.arange(m, device="cuda", dtype=torch.float64) for m in (nx, ny, nz)]
    cell = torch.stack(torch.meshgrid(*axes, indexing="ij"), dim=-1)
    p = (cell[:, :, :, None, :] + basis) * edge
    u = torch.rand(p.shape, generator=_generator(seed, 0), device="cuda", dtype=torch.float64)
    return (p + (2.0 * u - 1.0) * JITTER).to(torch.float32)


_BASIS = [[0.0, 0.0, 0.0], [0.5, 0.5, 0.0], [0.5, 0.0, 0.5], [0.0, 0.5, 0.5]]


def _ball(n, r):
    """Expected points of n uniform ones in the unit cube within r of another."""
    return n * (4.0 / 3.0 * math.pi * r ** 3 - 1.5 * math.pi * r ** 4 + 1.6 * r ** 5 - r ** 6 / 6.0)


def _neighbours(case, factor=1.0):
    """Expected neighbours of a query within factor times the case's radius."""
    n, r = case["n"], _radius(case) * factor
    if case["data"] == "uniform":
        return _ball(n, r)
    x = r / (2.0 * SIGMA)
    near = math.erf(x) - 2.0 * x / math.sqrt(math.pi) * math.exp(-x * x)
    return n / CENTRES * near + _ball(n, r)


def _overlaps(nq):
    """Expected overlaps of nq boxes: per axis the sides' sum is the chance."""
    return nq * 5000000 * (2.0 * math.exp(SIDE_MU + 0.5 * SIDE_SIGMA ** 2)) ** 3


def _ray_hits(case):
    """Expected boxes along case["nq"] rays, at most case["k"] each: a chord's
    hits are Poisson with the boxes' mean cross section, averaged over rays."""
    g = torch.Generator()
    g.manual_seed(1)
    m = 20000
    o = torch.rand((m, 3), generator=g, dtype=torch.float64) * 1.4 - 0.2
    d = torch.randn((m, 3), generator=g, dtype=torch.float64)
    i = torch.arange(m)
    other = torch.arange(3)[None, :] != ((i // 5) % 3)[:, None]
    d = torch.where((i % 5 == 1)[:, None] & other, torch.full_like(d, 1e-12), d)
    d = d / d.norm(dim=1, keepdim=True)
    a, b = (0.0 - o) / d, (1.0 - o) / d
    t0 = torch.minimum(a, b).amax(1).clamp(min=0.0)
    length = (torch.maximum(a, b).amin(1) - t0).clamp(min=0.0)
    side = math.exp(SIDE_MU + 0.5 * SIDE_SIGMA ** 2) * _box_scale(case["n"])
    mu = length * case["n"] * side ** 2 * d.abs().sum(1)
    if case["kind"] == "ray_all":
        return case["nq"] * float(mu.mean())
    hits, p, below = 0.0, torch.exp(-mu), torch.exp(-mu)
    for j in range(1, case["k"] + 1):  # sum of P(at least j hits)
        hits += float((1.0 - below).mean())
        p = p * mu / j
        below = below + p
    return case["nq"] * hits


def _results(case):
    """Expected length of the case's index array."""
    kind = case["kind"]
    if kind == "frame":
        return case["n"] * _neighbours(case)
    if kind == "build":
        return PROBES * 4 if case["geometry"] == "points" else _overlaps(PROBES)
    if kind == "radius":
        return case["n"] * _neighbours(case)
    if kind == "spheres":
        return case["nq"] * sum(_neighbours(case, 0.775 + 0.05 * j) for j in range(10)) / 10.0
    if kind == "nearest":
        return case["nq"] * case["k"]
    if kind == "overlap":
        return _overlaps(case["nq"])
    return _ray_hits(case)


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case)
    if kind != "energy":
        s["part"] = int(0.75 * _results(case))
    if kind == "frame":
        s["x"] = _points(case["data"], case["n"], seed, 0)
        s["r"] = _radius(case)
    elif kind == "build":
        if case["geometry"] == "points":
            s["x"] = _points(case["data"], case["n"], seed, 0)
            s["probe"] = ax.nearest(_points(case["data"], PROBES, seed, 1), 4)
        else:
            s["x"] = _boxes(case["n"], case["n"], seed, 0)
            s["probe"] = ax.intersects(ax.Boxes(_boxes(PROBES, case["n"], seed, 1)))
    elif kind == "radius":
        x = _points(case["data"], case["n"], seed, 0)
        s["tree"] = ax.BVH(x, node_format=case["nodes"])
        s["preds"] = ax.make_intersects(x, _radius(case))
    elif kind == "spheres":
        x = _points(case["data"], case["n"], seed, 0)
        q = _points(case["data"], case["nq"], seed, 1)
        r = _radius(case) * (0.75 + 0.5 * _rand(case["nq"], 1, _generator(seed, 2)))
        s["tree"] = ax.BVH(x, node_format=case["nodes"])
        s["preds"] = ax.intersects(ax.Spheres(torch.cat([q, r], dim=1)))
    elif kind == "nearest":
        x = _points(case["data"], case["n"], seed, 0)
        q = x if case["own"] else _points(case["data"], case["nq"], seed, 1)
        s["tree"] = ax.BVH(x, node_format=case["nodes"])
        s["preds"] = ax.make_nearest(q, case["k"])
    elif kind == "overlap":
        x = _boxes(case["n"], case["n"], seed, 0)
        s["tree"] = ax.BVH(x, node_format=case["nodes"])
        s["preds"] = ax.intersects(ax.Boxes(_boxes(case["nq"], case["n"], seed, 1)))
    elif kind in ("ray_first", "ray_all"):
        x = _boxes(case["n"], case["n"], seed, 0)
        rays = _rays(case["nq"], seed, 1)
        s["tree"] = ax.BVH(x, node_format=case["nodes"])
        s["preds"] = (ax.nearest(rays, case["k"]) if kind == "ray_first"
                      else ax.ordered_intersects(rays))
    else:
        s["x"] = _lattice(case, seed).reshape(-1, 3).contiguous()
    return s


def _csr(state, indices, offsets, **more):
    m = state["part"]
    return dict(offsets=offsets, first=indices[:m], last=indices[-m:], **more)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "frame":
        tree = ax.BVH(state["x"], node_format=case["nodes"])
        ri, ro = tree.query(ax.make_intersects(state["x"], state["r"]))
        ni, no, nd = tree.query(ax.make_nearest(state["x"], case["k"]), return_distances=True)
        return _csr(state, ri, ro, nearest=ni, nearest_offsets=no, distances=nd)
    if kind == "build":
        tree = ax.BVH(state["x"], node_format=case["nodes"])
        indices, offsets = tree.query(state["probe"])
        return _csr(state, indices, offsets,
                    bounds=torch.tensor(tree.bounds(), dtype=torch.float32))
    if kind == "energy":
        x = state["x"].detach().requires_grad_()
        e = ax.PairEnergy.apply(x, CUTOFF)
        e.backward()
        return dict(energy=e.detach(), gradient=x.grad)
    if kind == "nearest" and case["distances"]:
        indices, offsets, d = state["tree"].query(state["preds"], return_distances=True)
        return _csr(state, indices, offsets, distances=d)
    indices, offsets = state["tree"].query(state["preds"])
    return _csr(state, indices, offsets)


def work(case):
    """Inputs and indexed values (a float4 per point, two per box) read once,
    results written once; 8 operations per distance that is reported."""
    kind = case["kind"]
    if kind == "energy":
        n = 4 * case["nx"] * case["ny"] * case["nz"]
        return dict(bytes=24.0 * n + 8, flops=35.0 * 83 * n)
    n, found = case["n"], _results(case)
    if kind == "frame":
        found += n * case["k"]
        return dict(bytes=(12.0 + 16.0 + 16.0) * n + 4.0 * found + 4.0 * n * case["k"],
                    flops=8.0 * found)
    if kind == "build":
        value, node = (12, 16) if case["geometry"] == "points" else (24, 32)
        return dict(bytes=float((value + node) * n), flops=20.0 * n)
    value = 16.0 if kind in ("radius", "spheres", "nearest") else 32.0
    query = dict(radius=12, spheres=16, nearest=12).get(kind, 24)
    out = 8.0 if case.get("distances") else 4.0
    nq = case.get("nq", n)
    return dict(bytes=value * min(n, found) + (query + 8.0) * nq + out * found,
                flops=(8.0 if value == 16.0 else 12.0) * found)


# ------------------------------------------------------------ 64-bit results
def _nearest_distances(x, q, k):
    """Distances to the k nearest of x for every row of q, in 64 bits."""
    x, out = x.double(), []
    step = max(1, 200000000 // x.shape[0])
    for a in range(0, q.shape[0], step):
        b = q[a:a + step].double()
        d2 = torch.zeros((b.shape[0], x.shape[0]), device="cuda", dtype=torch.float64)
        for c in range(3):
            d2 += (b[:, c, None] - x[None, :, c]) ** 2
        out.append(torch.topk(d2, k, dim=1, largest=False, sorted=True).values.sqrt())
    return torch.cat(out).reshape(-1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "frame":
        x = _points(case["data"], case["n"], seed, 0)
        return dict(offsets=None, first=None, last=None, nearest=None, nearest_offsets=None,
                    distances=_nearest_distances(x, x, case["k"]))
    if kind == "build":
        if case["geometry"] == "points":
            lo = hi = _points(case["data"], case["n"], seed, 0).double()
        else:
            b = _boxes(case["n"], case["n"], seed, 0).double()
            lo, hi = b[:, :3], b[:, 3:]
        return dict(bounds=torch.cat([lo.amin(0), hi.amax(0)]), first=None, last=None,
                    offsets=None)
    if kind == "nearest" and case["distances"]:
        if case["n"] * case["nq"] > 80000000000:
            return None
        x = _points(case["data"], case["n"], seed, 0)
        q = x if case["own"] else _points(case["data"], case["nq"], seed, 1)
        return dict(first=None, last=None, offsets=None, distances=_nearest_distances(x, q, case["k"]))
    if kind == "energy":
        return _lattice_energy(case, seed)
    return None


def _lattice_energy(case, seed):
    """Energy and gradient over the lattice's own neighbour shells, in 64 bits.
    A pair counts when its distance in 32 bits is within the cutoff, which is
    what a neighbour list of 32-bit points holds."""
    x32 = _lattice(case, seed)
    x = x32.double()
    shape = x.shape[:3]
    grad = torch.zeros_like(x)
    energy = torch.zeros((), dtype=torch.float64, device="cuda")
    ic = 1.0 / CUTOFF ** 6
    phi_cut = 4.0 * (ic * ic - ic)
    reach = CUTOFF + 2.0 * math.sqrt(3.0) * JITTER
    for b in range(4):
        for c in range(4):
            for step in ((i, j, k) for i in range(-2, 3) for j in range(-2, 3)
                         for k in range(-2, 3)):
                if b == c and step == (0, 0, 0):
                    continue
                ideal = math.sqrt(2.0) * math.sqrt(sum(
                    (step[d] + _BASIS[c][d] - _BASIS[b][d]) ** 2 for d in range(3)))
                if ideal > reach or any(abs(step[d]) >= shape[d] for d in range(3)):
                    continue
                own = tuple(slice(max(0, -step[d]), shape[d] - max(0, step[d])) for d in range(3))
                far = tuple(slice(max(0, step[d]), shape[d] - max(0, -step[d])) for d in range(3))
                d32 = x32[far + (c,)] - x32[own + (b,)]
                s32 = d32[..., 0] * d32[..., 0]
                s32 = s32 + d32[..., 1] * d32[..., 1]
                s32 = s32 + d32[..., 2] * d32[..., 2]
                near = (s32.sqrt() <= CUTOFF).double()
                d = x[own + (b,)] - x[far + (c,)]
                i2 = 1.0 / (d * d).sum(-1)
                i6 = i2 ** 3
                energy += 0.5 * (near * (4.0 * i6 * (i6 - 1.0) - phi_cut)).sum()
                f = near * 24.0 * i2 * i6 * (1.0 - 2.0 * i6)
                grad[own + (b,)] += f[..., None] * d
    return dict(energy=energy, gradient=grad.reshape(-1, 3))
