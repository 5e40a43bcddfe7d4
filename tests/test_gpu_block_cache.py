"""Blocks that the library keeps between calls: trees and queries of changing
sizes, from several threads on streams of their own, with trees destroyed
while others are built, give the rows of a run that keeps nothing."""
import ctypes
import threading

import numpy as np
import pytest
import torch

import arborx_amd as ax
from arborx_amd import synthetic

pytestmark = pytest.mark.gpu


def _rows(n, seed, fmt):
    x = torch.from_numpy(synthetic.uniform_points(n, seed)).cuda()
    r = synthetic.radius_for_neighbours(n, 12)
    tree = ax.BVH(x, node_format=fmt)
    i, o = tree.query(ax.make_intersects(x, r))
    ki, _, kd = tree.query(ax.make_nearest(x, 5), return_distances=True)
    return [t.cpu() for t in (i, o, ki, kd)]


@pytest.mark.parametrize("fmt", ["fp32", "q16"])
def test_kept_blocks_on_threads_and_streams(fmt):
    sizes = [1, 2, 700, 4097, 20000, 4096, 650, 20001]
    want = {}
    for j, n in enumerate(sizes):
        ax.trim_memory()
        want[n] = _rows(n, j, fmt)
    errors = []

    def work(shift):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(3):
                    for j in range(len(sizes)):
                        j = (j + shift) % len(sizes)
                        for a, b in zip(_rows(sizes[j], j, fmt), want[sizes[j]]):
                            assert torch.equal(a, b), (shift, sizes[j])
        except BaseException as e:  # reported by the main thread
            errors.append(e)

    threads = [threading.Thread(target=work, args=(s,)) for s in (0, 3, 5)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors


def test_trim_gives_kept_blocks_back():
    _rows(500000, 1, "q16")
    torch.cuda.empty_cache()
    ax.trim_memory()
    free = torch.cuda.mem_get_info()[0]
    rows = _rows(500000, 1, "q16")
    torch.cuda.empty_cache()
    assert torch.cuda.mem_get_info()[0] < free  # blocks and workspaces are kept ...
    ax.trim_memory()
    # ... and given back (the runtime keeps up to a few megabytes of its own)
    assert torch.cuda.mem_get_info()[0] > free - (32 << 20)
    assert rows[0].numel() > 0


def test_kept_blocks_give_way_to_allocations_that_fail():
    # every allocation fails while blocks are kept, as on a full device:
    # trees, scratch rows, candidate rows, results and energies get memory all
    # the same
    n = 30000
    x = torch.from_numpy(synthetic.uniform_points(n, 1)).cuda()
    r = synthetic.radius_for_neighbours(n, 12)  # as in _rows
    want = _rows(n, 1, "q16")
    L = ax.lib()

    def call(fn, *args):
        assert fn(*args) == 0, L.axb_last_error()

    def kept():  # something in the lists, and no workspace from earlier calls
        ax.trim_memory()
        ax.BVH(x[:5000])
        assert ax.debug_cached_bytes() > 0

    with ax.debug_memory(scarce=True):
        kept()
        tree = ax.BVH(x, node_format="q16")
        kept()
        i, o = tree.query(ax.make_intersects(x, r))
        kept()
        ki, _, kd = tree.query(ax.make_nearest(x, 5), return_distances=True)
        for a, b in zip((i, o, ki, kd), want):
            assert torch.equal(a.cpu(), b)
        kept()
        off, idx = ax.energy.neighbour_csr(x, r)
        kept()
        e = torch.zeros((), dtype=torch.float64, device="cuda")
        call(L.axb_pair_energy, ax._ptr(x), n, ax._ptr(off), ax._ptr(idx), ctypes.c_float(r),
             ctypes.c_void_p(e.data_ptr()), None, ax._stream())
        # results from the library's own allocator (creating a BVH object
        # sets torch's again), and the per-thread stream (handle 2), whose
        # blocks are never kept
        per_thread = ctypes.c_void_p(2)
        h, ind, nnz = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_int64()
        offsets = torch.empty(n + 1, dtype=torch.int64, device="cuda")
        kept()
        torch.cuda.synchronize()
        call(L.axb_bvh_create, ax._ptr(x), n, ax.GEOMETRY_POINTS, ax.NODES_Q16, 0, per_thread,
             ctypes.byref(h))
        for stream in (ax._stream(), per_thread):
            kept()
            call(L.axb_set_output_allocator, ax._ALLOC_FN(0), ax._FREE_FN(0), None)
            try:
                call(L.axb_bvh_query_intersects_radius, h, ax._ptr(x), n, ctypes.c_float(r),
                     ax.TraversalPolicy()._c(), ax._ptr(offsets), ctypes.byref(ind),
                     ctypes.byref(nnz), stream)
            finally:
                ax._use_torch_allocator()
            assert ind.value not in ax._live_outputs  # not torch's memory
            call(L.axb_free, ind, stream)
            assert nnz.value == int(want[1][-1])
        L.axb_bvh_destroy(h)
    assert np.isfinite(e.item())


def test_full_lists_let_the_oldest_blocks_go():
    # sizes that drift through the size classes, and streams that come and
    # go: the lists stay within their limit and the newest sizes stay in them
    limit = 8 << 20
    ax.trim_memory()
    points = torch.from_numpy(synthetic.uniform_points(60000, 2)).cuda()
    want = {}
    for n in range(9000, 60000, 5100):
        tree = ax.BVH(points[:n], node_format="q16")
        want[n] = [t.cpu() for t in tree.query(ax.make_nearest(points[:n], 3))]
        del tree
    ax.trim_memory()
    with ax.debug_memory(cache_bytes=limit):
        for turn in range(2):
            for n in want:
                with torch.cuda.stream(torch.cuda.Stream()):
                    tree = ax.BVH(points[:n], node_format="q16")
                    got = tree.query(ax.make_nearest(points[:n], 3))
                    for a, b in zip(got, want[n]):
                        assert torch.equal(a.cpu(), b), n
                    del tree
                assert 0 < ax.debug_cached_bytes() <= limit
        # small blocks of the default stream are kept although others filled
        # the lists before
        for _ in range(3):
            tree = ax.BVH(points[:700])
            full = ax.debug_cached_bytes()
            del tree
            assert full < ax.debug_cached_bytes() <= limit
            with ax.profile(timing=True) as p:
                ax.BVH(points[:700])
            assert "host:pool_alloc" not in p.kernels and "host:pool_free" not in p.kernels
    ax.trim_memory()
