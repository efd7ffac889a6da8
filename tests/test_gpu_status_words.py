"""The status words that a context keeps from call to call: what a refused call
leaves in them must not be taken for the next call's."""
import numpy as np
import pytest

from libsupermesh_amd import gpu, meshgen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("bad", [(0, -1), (-1, 0), (0, 10**6)])
@pytest.mark.parametrize("refusals", [1, 2, 3])
def test_refused_pair_list_then_other_calls(dim, bad, refusals):
    # on a new context, where the numbers of the stagings are still small
    A = gpu.DeviceMesh(*meshgen.split_grid(dim, 3, 1))
    B = gpu.DeviceMesh(*meshgen.split_grid(dim, 2, 1, mesh_id=1))
    pa, pb = (gpu.DeviceArray(np.array([0, x], dtype=np.int32)) for x in bad)
    ctx = gpu.Context()
    for _ in range(refusals):
        with pytest.raises(gpu.GpuError, match="pair id out of range"):
            ctx.clip_pairs(A, B, pa, pb)
    for _ in range(4):
        r = ctx.supermesh(A, B)
        assert abs(r.sum - 1.0) <= 1e-12
    good = gpu.DeviceArray(np.zeros(2, dtype=np.int32))
    assert ctx.clip_pairs(A, B, good, good).npairs == 2
    ctx.close()
