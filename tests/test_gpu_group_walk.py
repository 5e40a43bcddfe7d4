"""Radius searches of point trees by 64 lanes together, against the oracle's
rope walk (rows equal in order): the sizes at the edges of leaf blocks, of the
levels above them and of wavefronts, radii and positions at which the
half-precision test of a pair is tightest or cannot be used, and wavefronts
whose predicates lie far apart and walk alone."""
import numpy as np
import pytest
import torch

import arborx_amd as ax
import oracle
from arborx_amd import synthetic

pytestmark = pytest.mark.gpu


def _check(points, spheres, fmt="q16", sort=True):
    t = oracle.Tree(points, 0)
    o_ref, i_ref = t.query_spatial(0, spheres)
    tree = ax.BVH(torch.from_numpy(points).cuda(), node_format=fmt)
    i, o = tree.query(ax.intersects(ax.Spheres(torch.from_numpy(spheres))),
                      ax.TraversalPolicy(0, sort))
    np.testing.assert_array_equal(o.cpu().numpy(), o_ref)
    np.testing.assert_array_equal(i.cpu().numpy(), i_ref)
    return o_ref[-1]


def _spheres(p, r):
    return np.concatenate([p, np.broadcast_to(np.float32(r), (len(p),)).reshape(-1, 1)],
                          1).astype(np.float32)


@pytest.mark.parametrize("fmt", ["fp32", "q16"])
@pytest.mark.parametrize("n", [2, 5, 63, 64, 65, 255, 4095, 4096, 4097, 20001, 262145])
def test_edges_of_blocks_and_levels(n, fmt):
    p = synthetic.uniform_points(n, n % 97)
    r = min(synthetic.radius_for_neighbours(n, 24), 0.6)
    nq = min(n, 20001)
    assert _check(p, _spheres(p[:nq], r), fmt) >= nq


@pytest.mark.parametrize("nq", [1, 63, 64, 65, 1000, 4001])
def test_edges_of_wavefronts_and_order(nq):
    p = synthetic.uniform_points(3000, 5)
    q = synthetic.uniform_points(nq, 6) * np.float32(1.2) - np.float32(0.1)
    g = np.random.default_rng(nq)
    s = _spheres(q, 0.0)
    s[:, 3] = g.uniform(0.0, 0.12, nq)
    for sort in (True, False):
        _check(p, s, sort=sort)


@pytest.mark.parametrize("scale,shift", [(1.0, 0.0), (1e-6, 0.0), (1e6, 0.0), (1.0, 1000.0),
                                         (1e-13, 0.0), (1e16, 0.0)])
def test_scales_and_offsets(scale, shift):
    # a grid whose spacing is the radius: hits and misses at the threshold
    a = np.arange(12, dtype=np.float64)
    p = np.stack(np.meshgrid(a, a, a, indexing="ij"), -1).reshape(-1, 3) / 12.0
    p = (p * scale + shift).astype(np.float32)
    for k in (1.0, np.sqrt(2.0), 2.0):
        r = np.float32(k * scale / 12.0)
        for rr in (np.nextafter(r, np.float32(0)), r, np.nextafter(r, np.float32(np.inf))):
            _check(p, _spheres(p, rr))


def test_radii_and_centres_without_hits_or_bounds():
    p = synthetic.uniform_points(5000, 1)
    s = _spheres(p, 0.08)
    s[::7, 3] = 0.0
    s[3::7, 3] = -1.0
    s[5::11, 3] = np.nan
    s[64:128, 3] = 1e-20
    s[777, 3] = np.inf
    s[1000, 0] = np.nan
    s[2000, 1] = np.inf
    s[3000, 2] = 1e30
    _check(p, s)
    p[::2] = p[0]  # many duplicates: rows longer than a scratch row
    _check(p, _spheres(p[:600], 0.01), "fp32")


@pytest.mark.parametrize("fmt", ["fp32", "q16"])
@pytest.mark.parametrize("sort", [True, False])
def test_infinite_radius_at_an_infinite_centre(fmt, sort):
    # sqrt(inf) <= inf: such a sphere lists every point, whatever the other
    # predicates of its wavefront are and whether there are any
    p = synthetic.uniform_points(500, 3)
    far = np.array([[np.inf, 0, 0, np.inf], [0.5, -np.inf, 0.5, np.inf]], np.float32)
    s = _spheres(synthetic.uniform_points(640, 4), 0.05)
    s[[5, 300]] = far  # among ordinary ones
    assert _check(p, s, fmt, sort) >= 1000
    assert _check(p, far[:1], fmt, sort) == 500  # alone
    s[64:128] = far[0]  # a wavefront of them
    s[130:190, 0] = np.inf  # infinite centres, finite radii
    s[200] = [np.nan, 0, 0, np.inf]  # no distance at all
    assert _check(p, s, fmt, sort) >= 66 * 500


def test_far_apart_predicates_walk_alone():
    # clusters at the corners of a large cube; wavefronts span several
    g = np.random.default_rng(3)
    c = np.array([[x, y, z] for x in (0, 1) for y in (0, 1) for z in (0, 1)], np.float64) * 1e4
    p = (c[np.arange(40000) % 8] + g.normal(size=(40000, 3))).astype(np.float32)
    _check(p, _spheres(p[g.permutation(40000)[:8000]], 0.15), sort=False)
    _check(p, _spheres(p[:6000], 30.0)[::40].copy(), sort=False)


@pytest.mark.parametrize("nq,grouped", [(100, False), (2499, False), (2500, True)])
def test_rows_written_again_go_the_way_of_their_batch(nq, grouped):
    p = synthetic.uniform_points(20000, 12)
    s = _spheres(p[:nq], synthetic.radius_for_neighbours(20000, 300))
    with ax.profile(timing=True) as prof:
        nnz = _check(p, s)
    assert nnz > 96 * nq  # rows longer than a scratch row
    kernels = [k for k in prof.kernels if "k_spatial" in k]
    assert len(kernels) == 2 and all(("k_spatial_group" in k) == grouped for k in kernels)


@pytest.mark.parametrize("n", [2, 65, 4097, 30000])
def test_neighbour_list_leaves_the_point_out(n):
    p = synthetic.uniform_points(n, 8)
    p[n // 2:n // 2 + 3] = p[0]  # duplicates of a point are its neighbours
    r = min(synthetic.radius_for_neighbours(n, 40), 0.5)
    # rows of the radius query without the point itself, in the same order
    o_all, i_all = oracle.Tree(p, 0).query_spatial(0, _spheres(p, r))
    own = np.repeat(np.arange(n), np.diff(o_all))
    o_ref, _ = oracle.neighbor_list(p, r, True)
    o, i = ax.find_full_neighbor_list(torch.from_numpy(p).cuda(), r)
    np.testing.assert_array_equal(o.cpu().numpy(), o_ref)
    np.testing.assert_array_equal(i.cpu().numpy(), i_all[i_all != own])


# ------------------------------------------------------------ nearest
def _check_nearest(points, queries, k, fmt="q16"):
    t = oracle.Tree(points, 0)
    o_ref, i_ref, d_ref = t.query_knn(queries, k)
    tree = ax.BVH(torch.from_numpy(points).cuda(), node_format=fmt)
    i, o, d = tree.query(ax.make_nearest(torch.from_numpy(queries), k), return_distances=True)
    np.testing.assert_array_equal(o.cpu().numpy(), o_ref)
    np.testing.assert_array_equal(i.cpu().numpy(), i_ref)
    np.testing.assert_array_equal(d.cpu().numpy().view(np.uint32), d_ref.view(np.uint32))


@pytest.mark.parametrize("fmt", ["fp32", "q16"])
@pytest.mark.parametrize("k", [1, 2, 3, 5, 8, 13, 16, 17, 32, 33, 64])
def test_nearest_uniform(k, fmt):
    p = synthetic.uniform_points(5000, k)
    _check_nearest(p, p, k, fmt)
    q = synthetic.uniform_points(1001, k + 100) * np.float32(1.5) - np.float32(0.25)
    _check_nearest(p, q, k, fmt)


@pytest.mark.parametrize("k", [1, 10, 40])
def test_nearest_uneven_density(k):
    g = np.random.default_rng(k)
    n = 12000
    # clusters of very different widths, a line, a plane, duplicates, outliers
    p = g.uniform(size=(n, 3))
    w = 10.0 ** g.uniform(-4, -1, 40)
    c = g.uniform(size=(40, 3))
    i = np.arange(6000) % 40
    p[:6000] = c[i] + w[i, None] * g.normal(size=(6000, 3))
    p[6000:7500, 1:] = 0.5
    p[7500:9000, 2] = 0.25
    p[9000:9200] = p[9000]
    p[9200:9210] *= 50.0
    p = p.astype(np.float32)
    _check_nearest(p, p, k)
    _check_nearest(p, np.roll(p, 1, axis=1)[:3000].copy(), k)
    _check_nearest(p, np.repeat(p[8990:9010], 200, axis=0), k)


def test_nearest_ties_and_lists_of_queries_left():
    a = np.arange(18, dtype=np.float32)
    p = np.stack(np.meshgrid(a, a, a, indexing="ij"), -1).reshape(-1, 3)
    _check_nearest(p, p, 16)  # a grid: the 16th is tied with others
    q = synthetic.uniform_points(4000, 2)
    q[::9, 0] = np.nan
    q[1::9] = 3e18
    ref = ax.BruteForce(torch.from_numpy(p).cuda()).query(
        ax.make_nearest(torch.from_numpy(q), 6), return_distances=True)
    tree = ax.BVH(torch.from_numpy(p).cuda())
    for kw in (dict(), dict(knn_batch_max=777), dict(knn_rounds=1), dict(knn_rounds=-1)):
        with ax.debug_limits(**kw):
            got = tree.query(ax.make_nearest(torch.from_numpy(q), 6), return_distances=True)
        keep = torch.from_numpy(~np.isnan(q[:, 0])).cuda()
        for x, y in zip(got, ref):
            if x.numel() == 6 * len(q):
                x, y = x.reshape(-1, 6)[keep], y.reshape(-1, 6)[keep]
            assert torch.equal(x, y), kw


# ------------------------------------------- what is left to the lanes' walks
def _leaves_per_query(points, spheres, sort):
    tree = ax.BVH(torch.from_numpy(points).cuda(), node_format="q16")
    q = ax.intersects(ax.Spheres(torch.from_numpy(spheres)))
    with ax.profile(timing=False, visits=True) as prof:
        tree.query(q, ax.TraversalPolicy(0, sort))
    _check(points, spheres, sort=sort)
    return prof.visits["leaf"] / len(spheres)


def test_groups_that_do_not_pay_walk_alone():
    # visits count blocks of 64 leaves for a group's lanes, leaves for a lane
    # alone: a group over all leaves looks at n / 64 blocks
    n = 16000
    g = np.random.default_rng(1)
    p = synthetic.uniform_points(n, 3)
    r = synthetic.radius_for_neighbours(n, 30)
    assert _leaves_per_query(p, _spheres(p[g.permutation(n)], r), False) < 200  # not 250
    assert _leaves_per_query(p, _spheres(p, r), True) < 40  # close together: groups
    # on a line every cell of the query order holds thousands of points
    line = np.full((1 << 20, 3), 0.5, np.float32)
    line[:, 0] = synthetic.uniform01(7, 1 << 20)
    assert _leaves_per_query(line, _spheres(line, 8.0 / (1 << 20)), True) < 40  # not 64


@pytest.mark.parametrize("scale", [1e-11, 1e-4, 1e8, 1e13])
def test_cost_of_a_group_at_any_scale(scale):
    p = (synthetic.uniform_points(20000, 3) * np.float32(scale)).astype(np.float32)
    r = np.float32(synthetic.radius_for_neighbours(20000, 30) * scale)
    assert _leaves_per_query(p, _spheres(p, r), True) < 40


def _knn_kernels(points, k, nq=None):
    tree = ax.BVH(torch.from_numpy(points).cuda(), node_format="q16")
    q = ax.make_nearest(torch.from_numpy(points[:nq]), k)
    with ax.profile(timing=True) as prof:
        tree.query(q)
    return [n for n in prof.kernels if "k_knn_collect" in n]


@pytest.mark.parametrize("k,grouped", [(2, "uniform"), (5, "uniform"), (8, "uniform sphere"),
                                       (24, "uniform sphere")])
def test_nearest_in_groups_where_leaves_fill_space(k, grouped):
    n = 40000
    g = np.random.default_rng(5)
    u = g.normal(size=(n, 3))
    t = g.uniform(0, 40, n)
    line = np.full((n, 3), 0.5)
    line[:, 0] = g.uniform(size=n)
    centres = g.uniform(size=(20, 3))
    sets = dict(uniform=g.uniform(size=(n, 3)), sphere=u / np.linalg.norm(u, axis=1)[:, None],
                helix=np.stack([np.cos(t), np.sin(t), t / 40], 1), line=line,
                clusters=centres[np.arange(n) % 20] + 0.001 * u)
    for name, p in sets.items():
        p = p.astype(np.float32)
        kernels = _knn_kernels(p, k)
        assert len(kernels) == 1
        assert ("k_knn_collect_group" in kernels[0]) == (name in grouped.split()), name
        _check_nearest(p, p[:2000].copy(), k)
        _check_nearest(p, p, k)


def test_nearest_of_queries_outside_the_points():
    # far outside, the leaves' density is no guide to a radius: such lanes
    # walk alone (135 records per query, 270 where they search as a group)
    n = 200000
    p = synthetic.uniform_points(n, 1)
    q = synthetic.uniform_points(n, 2) * np.float32(1.5) - np.float32(0.25)
    tree = ax.BVH(torch.from_numpy(p).cuda(), node_format="q16")
    with ax.profile(timing=False, visits=True) as prof:
        tree.query(ax.make_nearest(torch.from_numpy(q), 5))
    assert prof.visits["leaf"] < 200 * n
    _check_nearest(p, q, 5)


@pytest.mark.parametrize("k,n,group", [(4, 1000000, False), (5, 999999, False),
                                       (5, 1000000, True), (8, 400000, True),
                                       (16, 400000, True)])
def test_nearest_of_many_uneven_queries_in_groups(k, n, group):
    g = np.random.default_rng(6)
    p = g.uniform(size=(1000, 3))[np.arange(n) % 1000] + 0.01 * g.normal(size=(n, 3))
    p = p.astype(np.float32)
    kernels = _knn_kernels(p, k)
    assert ["k_knn_collect_group" in name for name in kernels] == [group]
    _check_nearest(p, p, k)


@pytest.mark.parametrize("fill", [0, 1, 2, 3])
@pytest.mark.parametrize("k", [2, 3, 5, 8, 13, 16, 17, 24, 32, 33, 64])
def test_nearest_over_every_route(k, fill):
    # uneven density, duplicates, ties and queries without an answer, through
    # each guess of the radius and as small and as large launches
    g = np.random.default_rng(k)
    p = g.uniform(size=(7000, 3))
    p[:3000] = g.uniform(size=(30, 3))[np.arange(3000) % 30]
    p[:3000] += 10.0 ** g.uniform(-4, -1, (3000, 1)) * g.normal(size=(3000, 3))
    p[3000:3500, 1:] = 0.5
    p[3500:3600] = p[3500]
    a = np.arange(12) / 12.0
    p[4000:4000 + 1728] = np.stack(np.meshgrid(a, a, a, indexing="ij"), -1).reshape(-1, 3)
    p = p.astype(np.float32)
    q = np.concatenate([p, synthetic.uniform_points(999, k) * np.float32(2) - np.float32(0.5)])
    t = oracle.Tree(p, 0)
    o_ref, i_ref, d_ref = t.query_knn(q, k)
    bad = q.copy()
    bad[::37, 1] = np.nan
    bad[5::41, 2] = np.inf
    ref_bad = ax.BruteForce(torch.from_numpy(p).cuda()).query(
        ax.make_nearest(torch.from_numpy(bad), k))[0].reshape(-1, k)
    keep = torch.from_numpy(np.isfinite(bad).all(1)).cuda()
    tree = ax.BVH(torch.from_numpy(p).cuda(), node_format="fp32" if k % 2 else "q16")
    for large in (1, 1 << 30):
        for limits in (dict(), dict(knn_batch_max=777)):
            with ax.debug_search(knn_large=large, fill=fill), ax.debug_limits(**limits):
                i, o, d = tree.query(ax.make_nearest(torch.from_numpy(q), k),
                                     return_distances=True)
                b = tree.query(ax.make_nearest(torch.from_numpy(bad), k))[0].reshape(-1, k)
            np.testing.assert_array_equal(i.cpu().numpy(), i_ref)
            np.testing.assert_array_equal(d.cpu().numpy().view(np.uint32), d_ref.view(np.uint32))
            assert torch.equal(b[keep], ref_bad[keep])
