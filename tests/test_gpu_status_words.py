"""The status words that a context keeps from call to call: what a refused call
leaves in them must not be taken for the next call's."""
import ctypes

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


def test_new_context_beside_a_busy_null_stream():
    # the first calls of a context, made while the null stream still has tens
    # of milliseconds of work queued: whatever clears the context's words has
    # to be done before its first kernel, not when the null stream gets to it
    A, B = gpu.DeviceMesh(*meshgen.split_grid(3, 16, 1)), gpu.DeviceMesh(*meshgen.split_grid(3, 15, 2, mesh_id=1))
    finder = gpu.Context()
    r = finder.intersection_finder(A, B)
    counts, measure, total = (gpu.DeviceArray(np.zeros(n, t)) for n, t in
                              ((r.npairs, np.int32), (r.npairs, float), (1, float)))
    f = gpu.lib().libsupermesh_gpu_clip_pairs_noalloc
    f.argtypes = [ctypes.c_int, ctypes.c_void_p, ctypes.POINTER(gpu.Mesh), ctypes.POINTER(gpu.Mesh), ctypes.c_long] + [ctypes.c_void_p] * 5
    f.restype = ctypes.c_int
    pos, enl = meshgen.split_grid(3, 4, 1)
    bad = enl.copy()
    bad[7, 2] = len(pos)
    S, Q, X = (gpu.DeviceMesh(*m) for m in ((pos, enl), meshgen.split_grid(3, 3, 2, mesh_id=1), (pos, bad)))
    want = finder.supermesh(S, Q, flags=gpu.SORTED)
    npairs, nout = want.npairs, want.nout
    r = finder.intersection_finder(A, B)
    for _ in range(40):
        gpu._check(f(0, None, ctypes.byref(A.struct), ctypes.byref(B.struct), r.npairs, r.rows, r.indices, counts.ptr,
                     measure.ptr, total.ptr))
    contexts = []
    for _ in range(6):
        ctx = gpu.Context()
        contexts.append(ctx)
        with pytest.raises(gpu.GpuError, match="Invalid node"):
            ctx.supermesh(X, Q)
        got = ctx.supermesh(S, Q, flags=gpu.SORTED)
        assert (got.npairs, got.nout) == (npairs, nout) and got.sum == want.sum
    gpu.synchronize()
    for ctx in contexts:
        ctx.close()
    finder.close()
