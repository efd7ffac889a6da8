"""The host-array finders pass their arrays through pinned memory in chunks of
2 MiB (524 288 node ids or results, 262 144 coordinates): the pair set on both
sides of a chunk's end, an invalid node in the first and in a later chunk, and
results that wait while another finder uses the context."""
import ctypes

import numpy as np
import pytest

import oracle_lib as O
from libsupermesh_amd import gpu, meshgen

pytestmark = pytest.mark.gpu


def strips(n):
    """n triangles in a row, 0.4 wide and one apart."""
    x = np.arange(n, dtype=np.float64)[:, None]
    pos = np.stack([x + [0.0, 0.4, 0.0], np.broadcast_to([0.0, 0.0, 1.0], (n, 3))], 2).reshape(-1, 2)
    return np.ascontiguousarray(pos), np.arange(3 * n, dtype=np.int64).reshape(n, 3)


# 174 763 triangles hold the first node id of the second chunk; 524 288 pairs
# fill a chunk of results; 43 691 triangles' 262 146 coordinates pass one
@pytest.mark.parametrize("n", [1, 341, 342, 43690, 43691, 174762, 174763, 524288, 524289])
def test_chunk_edges(n):
    pos, enl = strips(n)
    indptr, indices = gpu.tree_intersection_finder(pos, enl, pos, enl)
    assert np.array_equal(indptr, np.arange(n + 1)) and np.array_equal(indices, np.arange(n))


@pytest.mark.parametrize("at", [0, 524287, 524288, 600000])
@pytest.mark.parametrize("node", [-1, -2**63, "n", 2**63 - 1, 2**32])
def test_invalid_node(at, node):
    pos, enl = strips(200001)
    good = enl.copy()
    enl.reshape(-1)[at] = len(pos) if node == "n" else node
    with pytest.raises(Exception, match="Invalid node"):
        gpu.tree_intersection_finder(pos, enl, pos[:300], good[:100])
    indptr, indices = gpu.tree_intersection_finder(pos[:300], good[:100], pos[:300], good[:100])
    assert np.array_equal(indices, np.arange(100))


def test_results_wait_for_get_output():
    lib = gpu.lib()
    L, D, I = ctypes.c_long, ctypes.POINTER(ctypes.c_double), ctypes.c_int
    PL = ctypes.POINTER(L)
    pa, ea = meshgen.split_grid(2, 9, 1)
    pb, eb = meshgen.split_grid(2, 8, 2, mesh_id=1, diagonal=1)
    ea, eb = (np.ascontiguousarray(e, dtype=np.int64) for e in (ea, eb))

    def call(kind, name, *a):
        f = getattr(lib, f"libsupermesh_{kind}_intersection_finder_{name}")
        f.restype = None
        f(*a)

    def set_input(kind, p, e, q, f):
        r = ctypes.byref
        call(kind, "set_input", r(L(len(p))), r(I(2)), r(L(len(e))), r(I(3)), r(L(len(q))), r(I(2)), r(L(len(f))), r(I(3)),
             p.ctypes.data_as(D), e.ctypes.data_as(PL), q.ctypes.data_as(D), f.ctypes.data_as(PL))

    def output(kind, ne):
        n = L()
        call(kind, "query_output", ctypes.byref(n))
        indices, indptr = np.zeros(n.value, dtype=np.int64), np.zeros(ne + 1, dtype=np.int64)
        call(kind, "get_output", ctypes.byref(L(ne)), ctypes.byref(n), indices.ctypes.data_as(PL), indptr.ctypes.data_as(PL))
        return indptr, indices

    for _ in range(2):
        set_input("tree", pa, ea, pb, eb)
        set_input("rtree", pb, eb, pa, ea)
        t, r = output("tree", len(ea)), output("rtree", len(eb))
        for got, want in ((t, O.brute_force(pa, ea, pb, eb)), (r, O.brute_force(pb, eb, pa, ea, closed=True))):
            assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
        set_input("tree", pa, ea, pb, eb)  # nobody asks for these
