"""The quad clipper (csrc/tet_quad.hpp) against the oracle where it can go
wrong: lists that fill a wave's sixteen quads, one less and one more; tets on
a coarse dyadic lattice, whose vertices lie exactly on the other's planes
(every split case of Tetrahedron_Intersection.F90:292-434 and both ways a
plane can leave a tet whole); and the mass of pairs whose elements differ
much in size."""
import numpy as np
import pytest

import oracle_lib as O
from libsupermesh_amd import gpu

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = gpu.Context()
    yield c
    c.close()


def _tets(rng, n, lattice, vmin=0.0):
    t = rng.integers(0, lattice + 1, (8 * n + 64, 4, 3)) / lattice if lattice else rng.uniform(0, 1, (8 * n + 64, 4, 3))
    v = np.abs(np.einsum("ni,ni->n", t[:, 1] - t[:, 0], np.cross(t[:, 2] - t[:, 0], t[:, 3] - t[:, 0])))
    return np.ascontiguousarray(t[v > vmin][:n])


def _mesh(t):
    return t.reshape(-1, 3), np.arange(4 * len(t), dtype=np.int64).reshape(-1, 4)


@pytest.mark.parametrize("lattice", [0, 2, 4])
@pytest.mark.parametrize("n", [1, 3, 4, 15, 16, 17, 63, 64, 65, 2000])
def test_pair_lists_match_the_oracle(ctx, n, lattice):
    rng = np.random.default_rng(100 * n + lattice)
    pa, ea = _mesh(_tets(rng, n, lattice))
    pb, eb = _mesh(_tets(rng, n, lattice))
    ids = np.arange(n, dtype=np.int32)
    A, B = gpu.DeviceMesh(pa, ea), gpu.DeviceMesh(pb, eb)
    print(f"[quad] {n} pairs, lattice {lattice}", flush=True)
    r = ctx.clip_pairs(A, B, gpu.DeviceArray(ids), gpu.DeviceArray(ids), flags=gpu.ELEMENTS)
    out = gpu.fetch(r, 3, ("counts", "measure", "offsets", "elements"))
    cnt, meas = O.clip_pairs(pa, ea, pb, eb, ids, ids)
    assert np.array_equal(out["counts"], cnt)
    assert np.array_equal(out["measure"], meas)
    for p in range(min(n, 100)):
        got = out["elements"][out["offsets"][p]:out["offsets"][p + 1]]
        assert np.array_equal(got, O.intersect_tets(pa[ea[p]], pb[eb[p]])), p


@pytest.mark.parametrize("ratio", [1.0, 0.05, 20.0])
def test_mass_of_uneven_pairs(ctx, ratio):
    rng = np.random.default_rng(7)
    n = 500
    # well-shaped (six times the volume over 0.05): the basis functions of a
    # flat tet lose digits in either program
    a = _tets(rng, n, 0, 0.05)
    b = a.mean(axis=1, keepdims=True) + (_tets(rng, n, 0, 0.05) - 0.5) * ratio   # around A's centre
    (pa, ea), (pb, eb) = _mesh(a), _mesh(b)
    ids = np.arange(n, dtype=np.int32)
    r = ctx.clip_pairs(gpu.DeviceMesh(pa, ea), gpu.DeviceMesh(pb, eb), gpu.DeviceArray(ids), gpu.DeviceArray(ids),
                       flags=gpu.MASS)
    got = gpu.fetch(r, 3, ("blocks",))["blocks"]
    want = O.mass_pairs(pa, ea, pb, eb, ids, ids)
    # both sum a few hundred products of numbers of at most the pair's measure
    # (basis functions lie in [0, 1] in the overlap): 1e-12 of the largest entry
    scale = np.abs(want).max(axis=(1, 2), keepdims=True)
    assert (scale > 0).sum() > 100
    assert np.all(np.abs(got - want) <= 1e-12 * scale + 1e-300)
