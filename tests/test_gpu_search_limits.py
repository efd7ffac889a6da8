"""The candidate search where it changes its way at a limit of its buffers, of the
order's sort or of its rules: more tasks than the arrays of the first try hold (in
one mesh pair and in a batch), meshes of 2^23 elements and one more, and query
waves on both sides of the number from which walks are not cut."""
import numpy as np
import pytest

import oracle_lib as O
from libsupermesh_amd import gpu, meshgen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [2, 3])
def test_more_tasks_than_room(dim):
    # 250 query waves make room for 20 384 tasks; a large element in most of
    # them sends those waves to each of the 250 nodes of 64 elements
    rng = np.random.default_rng(dim)
    na, nb = 8000, 16000
    def simplices(n, size):
        t = rng.uniform(0, 1, (n, 1, dim)) + np.concatenate([np.zeros((n, 1, dim)), rng.uniform(0, size, (n, dim, dim))], 1)
        return t, np.arange(n * (dim + 1), dtype=np.int32).reshape(n, dim + 1)
    ta, ea = simplices(na, 0.01)
    tb, eb = simplices(nb, 0.01)
    large = rng.permutation(na)[: na // 32]
    box = np.concatenate([np.full((1, dim), -3.0), -3.0 + 6.0 * np.eye(dim)])  # its middle is 0
    ta[large] = ta[large][:, :1] + box
    pa, pb = ta.reshape(-1, dim), tb.reshape(-1, dim)
    ip, ix = O.brute_force(pa, ea, pb, eb)
    assert np.all(np.diff(ip)[large] == nb)
    ctx = gpu.Context()
    A, B = gpu.DeviceMesh(pa, ea), gpu.DeviceMesh(pb, eb)
    for _ in range(2):
        out = gpu.fetch(ctx.intersection_finder(A, B, flags=gpu.SORTED), dim, ("indptr", "indices", "rows"))
        assert np.array_equal(out["indptr"], ip) and np.array_equal(out["indices"], ix)
        assert np.array_equal(out["rows"], np.repeat(np.arange(na), np.diff(ip)))
    ctx.close()


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("na", [32 * 2047 - 1, 32 * 2047, 32 * 2047 + 1, 32 * 2048 + 1])
def test_waves_about_the_cut(dim, na):
    rng = np.random.default_rng(na)
    def simplices(n, size):
        t = rng.uniform(0, 1, (n, 1, dim)) + np.concatenate([np.zeros((n, 1, dim)), rng.uniform(0, size, (n, dim, dim))], 1)
        return np.ascontiguousarray(t.reshape(-1, dim)), np.arange(n * (dim + 1), dtype=np.int32).reshape(n, dim + 1)
    pa, ea = simplices(na, 0.05)
    pb, eb = simplices(900, 0.1)
    ip, ix = O.brute_force(pa, ea, pb, eb)
    ctx = gpu.Context()
    out = gpu.fetch(ctx.intersection_finder(gpu.DeviceMesh(pa, ea), gpu.DeviceMesh(pb, eb), flags=gpu.SORTED), dim,
                    ("indptr", "indices", "rows"))
    assert np.array_equal(out["indptr"], ip) and np.array_equal(out["indices"], ix)
    assert np.array_equal(out["rows"], np.repeat(np.arange(na), np.diff(ip)))
    ctx.close()


def test_more_tasks_than_room_in_a_batch():
    # 200 meshes of one triangle over 45 000: 88 nodes of 512 elements each,
    # 17 600 tasks, where 7 query waves make room for 16 496
    n, m = 200, 150
    one = np.array([[-1.0, -1.0], [4.0, -1.0], [-1.0, 4.0]]), np.array([[0, 1, 2]], dtype=np.int32)
    many = meshgen.split_grid(2, m, 1)
    ctx = gpu.Context()
    r, br = ctx.supermesh_batched(gpu.DeviceMeshBatch([one] * n), gpu.DeviceMeshBatch([many] * n), flags=gpu.SORTED)
    per = 2 * m * m
    assert r.npairs == n * per
    out = gpu.fetch(r, 2, ("indptr", "indices", "rows"))
    assert np.array_equal(out["indptr"], per * np.arange(n + 1))
    assert np.array_equal(out["indices"], np.arange(n * per)) and np.array_equal(out["rows"], np.repeat(np.arange(n), per))
    offsets, sums = gpu.fetch_batch(br)
    assert np.array_equal(offsets, per * np.arange(n + 1)) and np.all(np.abs(sums - 1.0) <= 1e-12)
    ctx.close()


@pytest.mark.parametrize("n", [1 << 23, (1 << 23) + 1])
def test_order_of_eight_million(n):
    # triangles in a row, 0.4 wide and one apart: each meets itself
    pos = np.zeros((n, 3, 2))
    pos[:, :, 0] = np.arange(n, dtype=np.float64)[:, None] + [0.0, 0.4, 0.0]
    pos[:, 2, 1] = 1.0
    enl = np.arange(3 * n, dtype=np.int32).reshape(n, 3)
    ctx = gpu.Context()
    A = gpu.DeviceMesh(pos.reshape(-1, 2), enl)
    small = gpu.DeviceMesh(pos[-5:].reshape(-1, 2), enl[:5])
    out = gpu.fetch(ctx.intersection_finder(A, A), 2, ("indptr", "indices"))
    assert np.array_equal(out["indptr"], np.arange(n + 1)) and np.array_equal(out["indices"], np.arange(n))
    # one mesh beyond the limit and a small one, either way round
    out = gpu.fetch(ctx.intersection_finder(A, small, flags=gpu.SORTED), 2, ("indptr", "indices"))
    assert np.array_equal(out["indices"], np.arange(5)) and np.array_equal(np.diff(out["indptr"])[-6:], [0, 1, 1, 1, 1, 1])
    out = gpu.fetch(ctx.intersection_finder(small, A, flags=gpu.SORTED), 2, ("indptr", "indices"))
    assert np.array_equal(out["indices"], np.arange(n - 5, n)) and np.array_equal(out["indptr"], np.arange(6))
    ctx.close()
