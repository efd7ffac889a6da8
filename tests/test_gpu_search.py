"""The candidate search at the edges of its shapes: query waves of 32 with one
element fewer and more, hierarchies of one node, of exactly full groups of
eight and of one more, and rows on both sides of the row sort's 256 entries --
against the brute-force set of the oracle (Intersection_Finder.F90:1032-1050),
strict and closed."""
import numpy as np
import pytest

import oracle_lib as O
from libsupermesh_amd import gpu, meshgen

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = gpu.Context()
    yield c
    c.close()


def _simplices(rng, n, dim, size):
    """n separate simplices with a vertex in the unit cube and edges up to `size`."""
    t = rng.uniform(0, 1, (n, 1, dim)) + np.concatenate([np.zeros((n, 1, dim)), rng.uniform(0, size, (n, dim, dim))], 1)
    return np.ascontiguousarray(t.reshape(-1, dim)), np.arange(n * (dim + 1), dtype=np.int32).reshape(n, dim + 1)


def _check(ctx, pa, ea, pb, eb):
    A, B = gpu.DeviceMesh(pa, ea), gpu.DeviceMesh(pb, eb)
    for finder, closed in ((gpu.FINDER_TREE, False), (gpu.FINDER_RTREE, True)):
        ip, ix = O.brute_force(pa, ea, pb, eb, closed=closed)
        out = gpu.fetch(ctx.intersection_finder(A, B, finder=finder, flags=gpu.SORTED), 2, ("indptr", "indices", "rows"))
        assert np.array_equal(out["indptr"], ip) and np.array_equal(out["indices"], ix)
        assert np.array_equal(out["rows"], np.repeat(np.arange(len(ea)), np.diff(ip)))
        plain = gpu.fetch(ctx.intersection_finder(A, B, finder=finder), 2, ("indptr", "indices"))
        assert np.array_equal(plain["indptr"], ip)
        order = np.lexsort((plain["indices"], np.repeat(np.arange(len(ea)), np.diff(ip))))
        assert np.array_equal(plain["indices"][order], ix)
    return int(np.diff(ip).max(initial=0))


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("na", [1, 31, 32, 33, 700])
@pytest.mark.parametrize("nb", [1, 7, 8, 9, 64, 65, 512, 513])
def test_sizes(ctx, dim, na, nb):
    rng = np.random.default_rng(1000 * na + nb)
    print(f"[search] {dim}D {na} x {nb}", flush=True)
    _check(ctx, *_simplices(rng, na, dim, 0.3), *_simplices(rng, nb, dim, 0.2))


@pytest.mark.parametrize("nb", [256, 257, 5000])
def test_long_rows(ctx, nb):
    # a few elements over the whole domain: rows of (nearly) all of B; 700 of
    # them keep the search in the direction it was asked for
    rng = np.random.default_rng(nb)
    pa, ea = _simplices(rng, 700, 2, 0.05)
    pa[:9] = np.array([[-1.0, -1.0], [4.0, -1.0], [-1.0, 4.0]] * 3)
    assert _check(ctx, pa, ea, *_simplices(rng, nb, 2, 0.02)) == nb


def test_uneven_batch(ctx):
    # one batch of meshes of 2 and of thousands of elements, either way round
    sizes = [(1, 40), (40, 1), (3, 3), (1, 1), (25, 30), (2, 33)]
    meshes = [(meshgen.split_grid(2, a, 3, mesh_id=2 * k), meshgen.split_grid(2, b, 3, mesh_id=2 * k + 1, diagonal=1))
              for k, (a, b) in enumerate(sizes)]
    r, br = ctx.supermesh_batched(gpu.DeviceMeshBatch([m[0] for m in meshes]), gpu.DeviceMeshBatch([m[1] for m in meshes]),
                                  flags=gpu.SORTED)
    out = gpu.fetch(r, 2, ("indices",))
    offs, sums = gpu.fetch_batch(br)
    first = 0
    for k, ((pa, ea), (pb, eb)) in enumerate(meshes):
        _, ix = O.brute_force(pa, ea, pb, eb)
        assert np.array_equal(out["indices"][offs[k]:offs[k + 1]] - first, ix), k
        first += len(eb)
    assert np.all(np.abs(sums - 1.0) <= 1e-12)   # both meshes cover the unit square
