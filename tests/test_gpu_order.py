"""The sort of the elements by Morton code: rows of an unsorted search come in
the order of the hierarchy's leaves, which numpy's stable sort of the same
codes gives, for element counts at the edges of the one-block sort (1024 keys), of
the sort by counting (64 keys a block, up to 8192),
of the tiles (2048 keys) and groups of tiles of the other, of the
hierarchy's blocks (512 leaves) and of the one-block scan (16384 rows)."""
import numpy as np
import pytest

import oracle_lib as O
from libsupermesh_amd import gpu

pytestmark = pytest.mark.gpu


def spread(x, step, bits):
    out = np.zeros_like(x)
    for b in range(bits):
        out |= ((x >> np.uint64(b)) & np.uint64(1)) << np.uint64(step * b)
    return out


def morton_rank(pos, enl):
    """Place of every element in the order of the leading 32 bits of the
    Morton code of its box centre, ties by element id."""
    v = pos[enl]
    c = 0.5 * (v.min(1) + v.max(1))
    lo, hi = c.min(0), c.max(0)
    dim = pos.shape[1]
    bits = 32 if dim == 2 else 21
    code = np.zeros(len(enl), dtype=np.uint64)
    for d in range(dim):
        t = (c[:, d] - lo[d]) / (hi[d] - lo[d]) if hi[d] > lo[d] else np.zeros(len(enl))
        code |= spread((np.clip(t, 0.0, 1.0) * float((1 << bits) - 1)).astype(np.uint64), dim, bits) << np.uint64(d)
    key = code >> np.uint64(32 if dim == 2 else 31)
    rank = np.empty(len(enl), dtype=np.int64)
    rank[np.argsort(key, kind="stable")] = np.arange(len(enl))
    return rank


def loose(dim, n, seed, ties):
    """n small elements of any place; with `ties`, at 40 places only."""
    rng = np.random.default_rng(seed)
    at = rng.random((40, dim))[rng.integers(0, 40, n)] if ties else rng.random((n, dim))
    size = 2.0 * n ** (-1.0 / dim)
    pos = (at[:, None] + size * np.concatenate([np.zeros((1, dim)), np.eye(dim)])[None]).reshape(-1, dim)
    return pos, np.arange(n * (dim + 1), dtype=np.int64).reshape(n, dim + 1)


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("na, nb", [
    # one block each (to 1024), counting (to 8192)
    (1, 1), (3, 8), (20, 63), (21, 64), (22, 65), (200, 511), (200, 512), (200, 513), (1025, 1023), (400, 1024),
    (1024, 1025), (1024, 1024), (300, 1025), (2000, 4095), (3000, 8191), (8192, 8192),
    # one beyond
    (9000, 1), (9000, 513), (9000, 2047), (9000, 2048), (9000, 2049), (3000, 8193), (2049, 8 * 2048 + 5),
    (16384, 4096 + 1), (16385, 4096), (20000, 33 * 2048 - 1)])
def test_rows_come_in_leaf_order(dim, na, nb):
    ctx = gpu.Context(0)
    pb, eb = loose(dim, nb, nb, False)
    pa, ea = loose(dim, na, nb + 1, False)
    r = ctx.supermesh(gpu.DeviceMesh(pa, ea), gpu.DeviceMesh(pb, eb), flags=0)
    out = gpu.fetch(r, dim)
    rank = morton_rank(pb, eb)
    rows, cols = O.csr_to_pairs(out["indptr"], out["indices"])
    same = rows[1:] == rows[:-1]
    assert (np.diff(rank[cols])[same] > 0).all()
    if nb <= 20000:
        ip, ix = O.brute_force(pa, ea, pb, eb)
        assert np.array_equal(out["indptr"], ip)
        order = np.lexsort((cols, rows))
        assert np.array_equal(cols[order], ix)
    ctx.close()


@pytest.mark.parametrize("n", [700, 3000])
def test_equal_codes_keep_element_order(n):
    ctx = gpu.Context(0)
    pb, eb = loose(2, n, 5, True)
    pa, ea = loose(2, n // 2, 6, False)
    out = gpu.fetch(ctx.supermesh(gpu.DeviceMesh(pa, ea), gpu.DeviceMesh(pb, eb), flags=0), 2)
    rank = morton_rank(pb, eb)
    rows, cols = O.csr_to_pairs(out["indptr"], out["indices"])
    assert len(cols) > 0 and (np.diff(rank[cols])[rows[1:] == rows[:-1]] > 0).all()
    ctx.close()
