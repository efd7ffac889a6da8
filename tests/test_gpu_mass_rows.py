"""The 3D mixed-mass rows where their kernel changes path: nodes of 64 tets and
more (the node's list no longer fits the wave), rows of few columns, of more
than 64 and 128, and of more than 256 (the global sort); against the oracle's
blocks summed with scipy."""
import numpy as np
import pytest

import oracle_lib as O
from libsupermesh_amd import gpu, meshgen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb", [2, 4, 5, 7, 9])
@pytest.mark.parametrize("points", [12, 34, 35, 70])
def test_fan_of_tets(points, nb):
    import scipy.sparse as sp
    from scipy.spatial import ConvexHull
    # 2 points - 4 tets around one node: the triangles of a convex hull of
    # points on a sphere inside the unit cube, each joined to its centre
    rng = np.random.default_rng(points)
    x = rng.normal(size=(points, 3))
    x = 0.5 + 0.45 * x / np.linalg.norm(x, axis=1, keepdims=True)
    tri = ConvexHull(x).simplices
    assert len(tri) == 2 * points - 4
    pa = np.vstack([x, [[0.5, 0.5, 0.5]]])
    ea = np.hstack([tri, np.full((len(tri), 1), points)]).astype(np.int32)
    pb, eb = meshgen.split_grid(3, nb, 3, mesh_id=1)
    ctx = gpu.Context()
    r = ctx.supermesh(gpu.DeviceMesh(pa, ea), gpu.DeviceMesh(pb, eb), flags=gpu.MASS)
    out = gpu.fetch(r, 3, ("rows", "indices", "counts"))
    indptr, indices, values = gpu.fetch_mass(r, pa.shape[0])
    want = O.mass_pairs(pa, ea, pb, eb, out["rows"], out["indices"])
    ne = out["counts"] > 0
    rr = np.repeat(ea[out["rows"][ne]], 4, axis=1).ravel()
    cc = np.tile(eb[out["indices"][ne]], (1, 4)).ravel()
    W = sp.coo_matrix((want[ne].ravel(), (rr, cc)), shape=(pa.shape[0], pb.shape[0])).tocsr()
    W.sum_duplicates()
    W.sort_indices()
    print(f"[mass] {len(tri)} tets at the node, longest row {np.diff(indptr).max()} columns", flush=True)
    assert np.array_equal(indptr, W.indptr) and np.array_equal(indices, W.indices)
    # entries are sums of up to a few thousand products, each good to a few
    # ulps of the largest block entry that it was summed from
    assert np.abs(values - W.data).max() <= 1e-12 * np.abs(want).max() * max(1, len(tri))
    ctx.close()
