"""The 3D mass adds a row's entries in LDS, several lanes to one column in one
instruction: the same call has to give the same bits again, on rows of a few and
of hundreds of columns, whatever ran on the context before."""
import numpy as np
import pytest

from libsupermesh_amd import gpu, meshgen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("na,nb", [(8, 3), (12, 11), (6, 9), (20, 19)])
def test_same_bits(na, nb):
    A = gpu.DeviceMesh(*meshgen.split_grid(3, na, 1))
    B = gpu.DeviceMesh(*meshgen.split_grid(3, nb, 2, mesh_id=1, diagonal=1))
    ctx = gpu.Context()
    first = None
    for k in range(6):
        r = ctx.supermesh(A, B, flags=gpu.MASS | gpu.SORTED)
        got = gpu.fetch_mass(r, A.nnodes)
        if first is None:
            first = got
            print(f"[repeat] rows of up to {np.diff(got[0]).max()} columns", flush=True)
        for x, y in zip(got, first):
            assert np.array_equal(x, y)
        if k % 2:
            ctx.close()
            ctx = gpu.Context()
        ctx.supermesh(B, A, flags=gpu.ELEMENTS)
    ctx.close()
