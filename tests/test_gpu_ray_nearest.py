"""nearest(ray, k) for small k against the oracle's brute force: tiny trees,
boxes that overlap so much that the walk's stack leaves the LDS, ties of
distance (origins inside many boxes), and directions whose components are
zero or so small that their reciprocals overflow."""
import numpy as np
import pytest
import torch

import arborx_amd as ax
import oracle
from arborx_amd import synthetic
from tests.helpers import ray_inputs

pytestmark = pytest.mark.gpu


def _soup(n, side, seed):
    g = np.random.default_rng(seed)
    c = g.uniform(size=(n, 3))
    h = 0.5 * side * g.uniform(size=(n, 3))
    return np.concatenate([c - h, c + h], 1).astype(np.float32)


def _check(boxes, rays, k, fmt, buffer=0):
    o_ref, i_ref = oracle.bruteforce_rays_ordered(boxes, rays, k)
    tree = ax.BVH(torch.from_numpy(boxes).cuda(), geometry="boxes", node_format=fmt)
    i, o = tree.query(ax.nearest(ax.Rays.from_normalized(torch.from_numpy(rays)), k),
                      ax.TraversalPolicy(buffer))
    np.testing.assert_array_equal(o.cpu().numpy(), o_ref)
    np.testing.assert_array_equal(i.cpu().numpy(), i_ref)


@pytest.mark.parametrize("fmt", ["fp32", "q16"])
@pytest.mark.parametrize("k", [1, 2, 4, 5, 8, 9])
def test_first_boxes_of_a_soup(k, fmt):
    boxes = _soup(3000, 0.4, k)
    boxes[1000:1100] = boxes[5]  # ties of distance
    o, d = ray_inputs(500, k, boxes)
    rays = oracle.make_rays(o, d)
    _check(boxes, rays, k, fmt)
    _check(boxes, rays, k, fmt, buffer=2)


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 8, 9, 17])
def test_tiny_trees(n):
    boxes = _soup(n, 0.8, n)
    rays = oracle.make_rays(*ray_inputs(300, n, boxes))
    for k in (1, 3, 8):
        _check(boxes, rays, k, "fp32")
        _check(boxes, rays, k, "q16")


def test_directions_with_tiny_components():
    boxes = synthetic.lognormal_boxes(20000, 3, mu=np.log(0.03))
    rays = oracle.make_rays(*ray_inputs(400, 9, boxes))
    for j, t in enumerate((1e-40, -1e-40, 1e-38, -3e-39, 1e-30)):
        # (every fifth ray runs along an axis: its direction would not stay a unit vector)
        at = np.arange(j, 400, 10)
        rays[at[at % 5 != 1], 3 + j % 3] = np.float32(t)
    rays[9::10, :3] *= np.float32(1e6)  # far away: entries with few bits
    for fmt in ("fp32", "q16"):
        _check(boxes, rays, 4, fmt)
        o_ref, i_ref = oracle.bruteforce_rays_ordered(boxes, rays)
        tree = ax.BVH(torch.from_numpy(boxes).cuda(), geometry="boxes", node_format=fmt)
        r = ax.Rays.from_normalized(torch.from_numpy(rays))
        i, o = tree.query(ax.ordered_intersects(r))
        np.testing.assert_array_equal(o.cpu().numpy(), o_ref)
        np.testing.assert_array_equal(i.cpu().numpy(), i_ref)


@pytest.mark.parametrize("fmt", ["fp32", "q16"])
@pytest.mark.parametrize("k", [1, 4, 8])
def test_stack_past_its_entries(k, fmt):
    # 19 scales times three axes, eight equal boxes each, split one after the
    # other from the rest of the tree, and 65536 equal boxes at its end: the
    # way down to them passes more than 64 nodes, all around the rays' origins
    boxes = []
    for i in range(1, 20):
        for a in range(3):
            c = np.zeros(3)
            c[a] = 2.0 ** -i
            boxes += [np.concatenate([c - 1.5 * 2.0 ** -i, c + 1.5 * 2.0 ** -i])] * 8
    tip = 1.5 * 2.0 ** -20
    boxes += [np.array([-tip] * 3 + [tip] * 3)] * 65536
    boxes = np.array(boxes, np.float32)[np.random.default_rng(k).permutation(len(boxes))]
    g = np.random.default_rng(1)
    rays = oracle.make_rays(np.zeros((5, 3), np.float32), g.normal(size=(5, 3)).astype(np.float32))
    with ax.profile(timing=True) as prof:
        _check(boxes, rays, k, fmt)
    # the rows were taken from the whole ordered ones instead
    assert any("k_row_prefix_copy" in n for n in prof.kernels)
