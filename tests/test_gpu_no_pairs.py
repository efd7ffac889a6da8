"""Calls that find no candidate pair: meshes apart from each other, empty
meshes, empty pair lists and batches of such, in 2D and 3D and with every
output.  (In 3D the clip used to read the length of a work list that is only
made for at least one pair: a null pointer.)"""
import os

import numpy as np
import pytest

from libsupermesh_amd import gpu, meshgen

pytestmark = pytest.mark.gpu

DATA = os.path.join(os.path.dirname(os.path.abspath(gpu.__file__)), "data", "tet_counts_mlp.f32")
FLAGS = [0, gpu.SORTED, gpu.ELEMENTS, gpu.MASS, gpu.MASS | gpu.BLOCKS, gpu.GRAPH, gpu.TIMING,
         gpu.ELEMENTS | gpu.LEARNED, gpu.ELEMENTS | gpu.LEARNED | gpu.DENSE]


def _meshes(dim, kind):
    pos, enl = meshgen.split_grid(dim, 3, 1)
    empty = pos, enl[:0]
    return {"apart": ((pos, enl), (pos + 5.0, enl)), "no A": (empty, (pos, enl)), "no B": ((pos, enl), empty),
            "neither": (empty, empty)}[kind]


def _check(r, dim, flags, nnodes):
    assert r.npairs == 0 and r.sum == 0.0 and r.nonempty == 0 and r.nout == 0 and r.max_count == 0
    assert not np.any(gpu.device_to_numpy(r.indptr, r.nelements_a + 1, np.int64))
    if flags & gpu.ELEMENTS:
        assert gpu.device_to_numpy(r.offsets, 1, np.int64)[0] == 0 and r.elements_size == 0
    if flags & gpu.MASS:
        assert r.mass_nnz == 0 and not np.any(gpu.fetch_mass(r, nnodes)[0])


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("kind", ["apart", "no A", "no B", "neither"])
def test_supermesh(dim, kind):
    a, b = _meshes(dim, kind)
    A, B = gpu.DeviceMesh(*a), gpu.DeviceMesh(*b)
    ctx = gpu.Context()
    ctx.predictor_set(np.fromfile(DATA, dtype=np.float32))
    for flags in FLAGS:
        print(f"[no pairs] {dim}D {kind} flags {flags}", flush=True)
        _check(ctx.supermesh(A, B, flags=flags), dim, flags, a[0].shape[0])
    # the context goes on
    C = gpu.DeviceMesh(*meshgen.split_grid(dim, 3, 1))
    r = ctx.supermesh(C, gpu.DeviceMesh(*meshgen.split_grid(dim, 2, 1, mesh_id=1)))
    assert abs(r.sum - 1.0) <= 1e-12
    ctx.close()


@pytest.mark.parametrize("dim", [2, 3])
def test_pair_list(dim):
    A = gpu.DeviceMesh(*meshgen.split_grid(dim, 2, 1))
    none = gpu.DeviceArray(np.zeros(0, dtype=np.int32))
    ctx = gpu.Context()
    for flags in (0, gpu.ELEMENTS, gpu.MASS):
        print(f"[no pairs] {dim}D list flags {flags}", flush=True)
        r = ctx.clip_pairs(A, A, none, none, flags=flags)
        assert r.npairs == 0 and r.sum == 0.0 and r.nout == 0
    ctx.close()


@pytest.mark.parametrize("dim", [2, 3])
def test_batch(dim):
    pairs = [_meshes(dim, kind) for kind in ("apart", "no A", "no B")]
    A, B = (gpu.DeviceMeshBatch([p[k] for p in pairs]) for k in (0, 1))
    ctx = gpu.Context()
    for flags in (0, gpu.ELEMENTS, gpu.MASS, gpu.GRAPH):
        print(f"[no pairs] {dim}D batch flags {flags}", flush=True)
        r, br = ctx.supermesh_batched(A, B, flags=flags)
        assert r.npairs == 0 and r.sum == 0.0
        offsets, sums = gpu.fetch_batch(br)
        assert not np.any(offsets) and not np.any(sums)
    ctx.close()


def test_predictor_samples():
    a, b = _meshes(3, "apart")
    ctx = gpu.Context()
    assert ctx.predictor_collect(gpu.DeviceMesh(*a), gpu.DeviceMesh(*b), 100) == 0
    ctx.close()
