"""Trees are built through pageable memory in one piece, and queried through a
context's small pinned halves; finders go on through the halves of the default
context, which grow.  The sizes at which an array no longer fits the 1536 bytes
of a new context's halves (384 node ids, 192 coordinates), and an invalid node
on both sides."""
import numpy as np
import pytest

import oracle_lib as O
from libsupermesh_amd import gpu, meshgen

pytestmark = pytest.mark.gpu


def strips(n):
    x = np.arange(n, dtype=np.float64)[:, None]
    pos = np.stack([x + [0.0, 0.4, 0.0], np.broadcast_to([0.0, 0.0, 1.0], (n, 3))], 2).reshape(-1, 2)
    return np.ascontiguousarray(pos), np.arange(3 * n, dtype=np.int64).reshape(n, 3)


@pytest.mark.parametrize("n", [1, 32, 33, 64, 65, 127, 128, 129, 341, 342, 174763])
def test_trees(n):
    pos, enl = strips(n)
    tree = gpu.DeviceTree(pos, enl)
    for e in sorted({0, n // 2, n - 1}):
        assert np.array_equal(tree.query(pos[enl[e]]), [e])
    everything = np.array([[-1.0, -1.0], [2.0 * n, -1.0], [-1.0, 2.0]])
    assert np.array_equal(tree.query(everything), np.arange(n))
    indptr, indices = gpu.tree_intersection_finder(pos, enl, pos, enl)
    assert np.array_equal(indptr, np.arange(n + 1)) and np.array_equal(indices, np.arange(n))
    assert np.array_equal(tree.query(pos[enl[0]]), [0])
    tree.close()


@pytest.mark.parametrize("n,at", [(20, 0), (20, 59), (1000, 0), (1000, 2999)])
@pytest.mark.parametrize("node", [-1, "n", 2**32])
def test_invalid_node(n, at, node):
    pos, enl = strips(n)
    bad = enl.copy()
    bad.reshape(-1)[at] = len(pos) if node == "n" else node
    with pytest.raises(gpu.GpuError, match="Invalid node"):
        gpu.DeviceTree(pos, bad)
    tree = gpu.DeviceTree(pos, enl)
    assert np.array_equal(tree.query(pos[enl[n - 1]]), [n - 1])
    tree.close()


def test_many_trees():
    pa, ea = meshgen.split_grid(3, 3, 1)
    pb, eb = meshgen.split_grid(3, 2, 2, mesh_id=1)
    ip, ix = O.brute_force(pb, eb, pa, ea)
    trees = [gpu.DeviceTree(pa, ea) for _ in range(40)]
    for k, tree in enumerate(trees):
        e = k % len(eb)
        assert np.array_equal(tree.query(pb[eb[e]]), ix[ip[e]:ip[e + 1]])
    for tree in trees:
        tree.close()
