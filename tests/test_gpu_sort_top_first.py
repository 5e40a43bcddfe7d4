"""Large builds sort their 63-bit Morton codes by the top 32 bits first: the
permutation equals a stable sort of the whole codes for points whose codes
differ in the top half, for close groups (short runs put right one by one),
for duplicates, and for points squeezed into a few cells by an outlier (the
full sort runs)."""
import numpy as np
import pytest
import torch

import arborx_amd as ax
import oracle
from arborx_amd import synthetic

pytestmark = pytest.mark.gpu

N = (1 << 19) + 77


def _points(kind):
    p = synthetic.uniform_points(N, 4)
    g = np.random.default_rng(1)
    if kind == "pairs":  # neighbours closer than a cell of the top half
        p[1::2][: N // 2] = p[0::2][: N // 2] + g.normal(size=(N // 2, 3)).astype(np.float32) * 1e-5
        p = p[g.permutation(N)]
    elif kind == "runs":  # groups of 1 to 90 in one cell: some longer than a short run
        at = np.sort(g.integers(0, N // 40, N))
        p = (p[at] + g.uniform(size=(N, 3)).astype(np.float32) * 2e-6)[g.permutation(N)]
    elif kind == "long_runs":  # cells of hundreds of points, up to thousands
        at = np.minimum(g.exponential(400.0, N).astype(np.int64) ** 2 // 300, N - 1)
        p = (p[at] + g.uniform(size=(N, 3)).astype(np.float32) * 3e-6)[g.permutation(N)]
    elif kind == "late_inversion":  # duplicates with a smaller code after many
        p[:] = p[g.integers(0, N // 100, N)]
        p[N // 2:N // 2 + 100] = p[7] - np.float32(1e-6)
    elif kind == "short_runs":
        p = (p[np.arange(N) // 30] + g.uniform(size=(N, 3)).astype(np.float32) * 1e-6)
        p = p[g.permutation(N)]
    elif kind == "duplicates":
        p = p[g.integers(0, 500, N)]
    elif kind == "outlier":
        p[N // 3] = 3e4
    return np.ascontiguousarray(p, np.float32)


@pytest.mark.parametrize("kind", ["uniform", "pairs", "short_runs", "runs", "duplicates",
                                  "long_runs", "late_inversion", "outlier"])
def test_permutation_is_the_stable_sort(kind):
    p = _points(kind)
    codes = oracle.morton64_values(p, oracle.scene_box(p))
    perm = np.argsort(codes, kind="stable")
    tree = ax.BVH(torch.from_numpy(p).cuda(), keep_topology=True)
    e = tree.export_topology()
    np.testing.assert_array_equal(e["perm"].cpu().numpy().view(np.uint32), perm)
    np.testing.assert_array_equal(e["keys"].cpu().numpy().view(np.uint64), codes[perm])


@pytest.mark.parametrize("longest", [4096, 4097, 400000])
def test_runs_at_the_edges_of_their_kernels(longest):
    # groups of exactly so many points in a cell of the top half of the codes
    # among many more far from them; 4097 takes the full sort after the one by
    # the top halves, 400000 instead of it
    n = 10_000_000
    g = np.random.default_rng(longest)
    sizes = [2, 3, 7, 8, 9, 10, 31, 32, 33, 63, 64, 65, 66, 127, 128, 129, 1000, 4095, longest]
    sizes = sizes + [s for s in sizes if s < 1000] * 40
    at = g.permutation(100 ** 3)[:len(sizes)]
    cell = np.stack([at // 10000, at // 100 % 100, at % 100], 1) * 0.005 + 0.0025
    p = synthetic.uniform_points(n, 4) * np.float32(0.45) + np.float32(0.55)
    members = np.repeat(cell, sizes, axis=0) + g.uniform(-1, 1, (sum(sizes), 3)) * 2e-5
    p[g.permutation(n)[:len(members)]] = members
    p = np.ascontiguousarray(p, np.float32)
    codes = oracle.morton64_values(p, oracle.scene_box(p))
    perm = np.argsort(codes, kind="stable")
    runs = np.unique(codes[perm] >> np.uint64(31), return_counts=True)[1]
    # (the largest group may lie on a cell's edge)
    assert set(sizes) <= set(runs.tolist()) or (longest == 400000 and runs.max() > 50000)
    tree = ax.BVH(torch.from_numpy(p).cuda(), keep_topology=True)
    e = tree.export_topology()
    np.testing.assert_array_equal(e["perm"].cpu().numpy().view(np.uint32), perm)
    np.testing.assert_array_equal(e["keys"].cpu().numpy().view(np.uint64), codes[perm])
