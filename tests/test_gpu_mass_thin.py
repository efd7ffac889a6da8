"""The 3D mass of thin, tilted tets, where the barycentric maps are large and
the products of two of them must not lose the digits of both.

The blocks are compared with the same integrals in extended precision: over the
kept tets as the library gives them, with the barycentric maps and the volumes
as 64-bit arithmetic makes them (staging is bit exact), so that what differs is
how the basis functions are evaluated and multiplied.  With u = 2^-53, a value
Minv (x - v1) is off by at most 4 u k, k = the largest sum_k |Minv_rk| |x_k - v1_k|
over the pair's vertices and maps, the fourth, one minus the others, by at most
16 u k; a product of two by 16 u (k_A + k_B) times the largest value.  The closed
form V/20 (sum_v f_v g_v + (sum f)(sum g)) adds five terms per tet to a sum of at
most V, and what is left is some 32 operations on values of at most V:
(5 n + 32) u V over n tets."""
import numpy as np
import pytest

from libsupermesh_amd import gpu, meshgen

pytestmark = pytest.mark.gpu

U = 2.0 ** -53


def _affine(v):
    """v1 and Minv of tets v[n, 4, 3], in the operations of the staging."""
    m = (v[:, 1:] - v[:, :1]).transpose(0, 2, 1)  # m[:, r, c]: coordinate r of edge c
    a, b, c = m[:, 0], m[:, 1], m[:, 2]
    minv = np.empty_like(m)
    for r, (i, j) in enumerate(((1, 2), (2, 0), (0, 1))):
        minv[:, r, 0] = b[:, i] * c[:, j] - b[:, j] * c[:, i]
        minv[:, r, 1] = c[:, i] * a[:, j] - c[:, j] * a[:, i]
        minv[:, r, 2] = a[:, i] * b[:, j] - a[:, j] * b[:, i]
    det = a[:, 0] * minv[:, 0, 0] + a[:, 1] * minv[:, 1, 0] + a[:, 2] * minv[:, 2, 0]
    return v[:, 0], minv / det[:, None, None]


def _volumes(t):
    e1, e2, e3 = t[:, 1] - t[:, 0], t[:, 2] - t[:, 0], t[:, 3] - t[:, 0]
    d = e1[:, 0] * (e2[:, 1] * e3[:, 2] - e2[:, 2] * e3[:, 1])
    d = d + e1[:, 1] * (e2[:, 2] * e3[:, 0] - e2[:, 0] * e3[:, 2])
    d = d + e1[:, 2] * (e2[:, 0] * e3[:, 1] - e2[:, 1] * e3[:, 0])
    return (1.0 / 6.0) * np.abs(d)


def _basis(affine, pair, tets):
    """Basis functions [tet, vertex, 4] in extended precision, and k per tet."""
    v1, minv = (x[pair].astype(np.longdouble) for x in affine)
    d = tets.astype(np.longdouble) - v1[:, None]
    f = (minv[:, None] * d[:, :, None]).sum(3)
    k = (np.abs(minv)[:, None] * np.abs(d)[:, :, None]).sum(3).max((1, 2))
    return np.concatenate([1 - f.sum(2, keepdims=True), f], 2), k


@pytest.mark.parametrize("shift", [0.0, 1000.0])
@pytest.mark.parametrize("thin", [(1.0, 1.0), (1e-2, 1e-2), (1e-3, 1e-3), (1e-4, 1e-4), (1e-3, 0.3)])
@pytest.mark.parametrize("crossed", [False, True])
def test_blocks(thin, shift, crossed):
    q, _ = np.linalg.qr(np.random.default_rng(7).normal(size=(3, 3)))
    pa, ea = meshgen.split_grid(3, 4, 1)
    pb, eb = meshgen.split_grid(3, 3, 2, mesh_id=1, diagonal=1)
    sa, sb = np.array([1.0, 1.0, thin[0]]), np.array([1.0, 1.0, thin[1]])
    pa, pb = (pa * sa) @ q + shift, (pb * (sb[[2, 0, 1]] if crossed else sb)) @ q + shift
    ctx = gpu.Context()
    A, B = gpu.DeviceMesh(pa, ea), gpu.DeviceMesh(pb, eb)
    r = ctx.supermesh(A, B, flags=gpu.MASS | gpu.BLOCKS | gpu.SORTED)
    out = gpu.fetch(r, 3, ("rows", "indices", "counts", "blocks"))
    el = gpu.fetch(ctx.supermesh(A, B, flags=gpu.ELEMENTS | gpu.SORTED), 3, ("counts", "elements"))
    ctx.close()
    assert np.array_equal(el["counts"], out["counts"]) and el["counts"].sum() > 50
    pair = np.repeat(np.arange(len(out["counts"])), out["counts"])
    tets = el["elements"]
    va, vb = pa[ea[out["rows"]]], pb[eb[out["indices"]]]
    fa, ka = _basis(_affine(va), pair, tets)
    fb, kb = _basis(_affine(vb), pair, tets)
    vol = _volumes(tets)
    sums = np.matmul(fa.transpose(0, 2, 1), fb) + fa.sum(1)[:, :, None] * fb.sum(1)[:, None]
    want = np.zeros((len(out["counts"]), 4, 4), dtype=np.longdouble)
    np.add.at(want, pair, sums * vol[:, None, None].astype(np.longdouble) / 20)
    top = np.maximum(1, np.maximum(np.abs(fa).max((1, 2)), np.abs(fb).max((1, 2))))
    bound = np.zeros(len(want), dtype=np.longdouble)
    np.add.at(bound, pair, U * vol * (16 * (ka + kb) * top + 32 * top ** 2 + 5 * out["counts"][pair]))
    err = np.abs(out["blocks"] - want).max((1, 2))
    live = out["counts"] > 0
    print(f"[thin] {thin} {shift} {crossed}: k up to {float(max(ka.max(), kb.max())):.1e}, "
          f"error / bound up to {float((err[live] / bound[live]).max()):.3f}", flush=True)
    assert np.all(err <= 1.01 * bound)
