"""The 2D mixed-mass rows by their number of columns: 64 and fewer are placed
by counting and summed in 64 / columns parts, more go through the bitonic
network; a node without pairs has none.  Against the oracle's blocks summed
with scipy."""
import numpy as np
import pytest

import oracle_lib as O
from libsupermesh_amd import gpu, meshgen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("na,nb", [(40, 3), (17, 16), (9, 14), (7, 17), (6, 18), (5, 19), (4, 17), (8, 30)])
def test_rows_by_columns(na, nb):
    import scipy.sparse as sp
    pa, ea = meshgen.split_grid(2, na, 11)
    pb, eb = meshgen.split_grid(2, nb, 12, mesh_id=1)
    pa = np.vstack([pa, [[0.5, 0.5]]])  # a node of no element
    ctx = gpu.Context()
    r = ctx.supermesh(gpu.DeviceMesh(pa, ea), gpu.DeviceMesh(pb, eb), flags=gpu.MASS)
    out = gpu.fetch(r, 2, ("rows", "indices", "counts"))
    indptr, indices, values = gpu.fetch_mass(r, pa.shape[0])
    want = O.mass_pairs(pa, ea, pb, eb, out["rows"], out["indices"])
    ne = out["counts"] > 0
    rr = np.repeat(ea[out["rows"][ne]], 3, axis=1).ravel()
    cc = np.tile(eb[out["indices"][ne]], (1, 3)).ravel()
    W = sp.coo_matrix((want[ne].ravel(), (rr, cc)), shape=(pa.shape[0], pb.shape[0])).tocsr()
    W.sum_duplicates()
    W.sort_indices()
    n = np.diff(indptr)
    print(f"[mass] rows of {n[:-1].min()} to {n.max()} columns", flush=True)
    assert np.array_equal(indptr, W.indptr) and np.array_equal(indices, W.indices)
    # sums of up to a few hundred products, each good to a few ulps of the
    # largest block entry
    assert np.abs(values - W.data).max() <= 1e-12 * np.abs(want).max()
    ctx.close()
