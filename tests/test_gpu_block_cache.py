"""Blocks that the library keeps between calls: trees and queries of changing
sizes, from several threads on streams of their own, with trees destroyed
while others are built, give the rows of a run that keeps nothing."""
import threading

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
