"""Workloads of the supermesher's public entry points, for timing.

Every case is one call (or, for a batch, one call per dimension) of
libsupermesh_amd.gpu as a program makes it: meshes resident in device memory
(host arrays for the drop-in finder), a context that the program keeps, and
all arrays that the call computes, as views of the context's buffers.

Meshes are jittered split grids of the unit square / cube (the kind of
libsupermesh_amd.meshgen, made here on the GPU so that large ones are quick):
``n`` cells per side give 2 n^2 triangles, 6 n^3 tetrahedra, n^2
quadrilaterals or n^3 hexahedra.  The case fixes the geometry and the seed the
numbering of nodes and elements (contiguous parts of the grid in any order, as
a partitioned mesh is numbered; a batch's mesh pairs in any order), so that
every seed has as many candidate pairs and output elements.
"""
import math
import os
import random

import numpy as np
import torch

from libsupermesh_amd import gpu

CUDA = "cuda" if torch.cuda.is_available() else "cpu"


# ---------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # the smallest call: the element-intersector meshes a user starts with,
        # 50 against 32 triangles; launches and host latency
        {"name": "tri_tiny", "call": "count", "dim": 2, "na": 5, "nb": 4, "sorted": True},
        # one call per mesh pair of a multi-mesh program, ~8 000 elements each
        {"name": "tri_small", "call": "count", "dim": 2, "na": 63, "nb": 61, "sorted": True},
        {"name": "tet_small", "call": "count", "dim": 3, "na": 11, "nb": 10, "sorted": True},
        # the reference's C finder on host arrays (set_input .. get_output)
        {"name": "finder_host_tri", "call": "finder", "dim": 2, "na": 257, "nb": 240, "sorted": True},
        # materialised supermesh, a coarse mesh over a fine one
        {"name": "tri_elements_coarse", "call": "elements", "dim": 2, "na": 150, "nb": 601, "sorted": False},
        # Galerkin projection: supermesh and P1 x P1 mixed mass matrix
        {"name": "tri_mass", "call": "mass", "dim": 2, "na": 1024, "nb": 1000, "sorted": False},
        {"name": "tet_mass", "call": "mass", "dim": 3, "na": 32, "nb": 30, "sorted": False},
        # counts, measures and the total overlap of two large tet meshes
        {"name": "tet_count", "call": "count", "dim": 3, "na": 64, "nb": 60, "sorted": False},
        # materialised tet supermesh, count then fill, and the single pass sized
        # by the learned predictor in the same (dense) layout
        {"name": "tet_elements", "call": "elements", "dim": 3, "na": 32, "nb": 29, "sorted": False},
        {"name": "tet_learned", "call": "learned", "dim": 3, "na": 48, "nb": 45, "sorted": False},
        # simplices against quadrilaterals / hexahedra
        {"name": "tet_hex", "call": "mixed", "dim": 3, "na": 40, "nb": 37, "sorted": False},
        # many mesh pairs of uneven sizes (50 to 50 000 elements) in one call per dimension
        {"name": "batch", "call": "batch", "dim": 0, "na": 192, "nb": 50000, "sorted": False},
    ]


#: per call and dimension: range of cells per side (for a batch: of mesh
#: pairs) and range of nb / na
RANGES = {
    ("count", 2): (4, 1024, 0.8, 1.25), ("count", 3): (4, 60, 0.85, 1.1), ("finder", 2): (24, 320, 0.8, 1.25),
    ("elements", 2): (12, 400, 0.25, 4.0), ("elements", 3): (6, 36, 0.6, 1.2), ("mass", 2): (24, 1000, 0.8, 1.1),
    ("mass", 3): (6, 32, 0.7, 1.1), ("learned", 3): (16, 46, 0.8, 1.1), ("mixed", 2): (24, 800, 0.8, 1.25),
    ("mixed", 3): (6, 38, 0.8, 1.1), ("batch", 0): (8, 192, 1.0, 1.0),
}


def draw(rng):
    call, dim = rng.choice([k for k in RANGES for _ in range(3 if k[0] == "count" else 1)])
    lo, hi, r0, r1 = RANGES[call, dim]
    na = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    nb = max(3, int(round(na * math.exp(rng.uniform(math.log(r0), math.log(r1))))))
    if call == "batch":
        nb = int(round(math.exp(rng.uniform(math.log(2000), math.log(50000)))))
    return {"call": call, "dim": dim, "na": na, "nb": nb,
            "sorted": call == "finder" or (call in ("count", "elements") and rng.random() < 0.5)}


def _batch_sizes(case):
    """(dim, na, nb) of every mesh pair of a batch: element counts
    log-uniform in [50, nb], 2D or 3D with equal odds, fixed by the case."""
    rng = random.Random(1000003 * case["na"] + case["nb"])
    out = []
    for _ in range(case["na"]):
        dim = 2 if rng.random() < 0.5 else 3
        n = []
        for _ in range(2):
            e = math.exp(rng.uniform(math.log(50), math.log(case["nb"])))
            n.append(max(1, round(math.sqrt(e / 2) if dim == 2 else (e / 6) ** (1 / 3))))
        out.append((dim, *n))
    return out


def _pairs(call, dim, na, nb):
    """Candidate pairs, nearly: boxes of jittered elements are 1.1 cells wide."""
    if call == "mixed":
        return 1.245 * 2 * (na + nb) ** 2 if dim == 2 else 1.192 * 6 * (na + nb) ** 3
    return 4.83 * (na + nb) ** 2 if dim == 2 else 51.1 * (na + nb) ** 3


def _one_work(call, dim, na, nb):
    loc = dim + 1
    locb = 2 ** dim if call == "mixed" else loc
    ne = {(2, False): 2, (3, False): 6}.get((dim, False))
    ea, eb = ne * na ** dim, (1 if call == "mixed" else ne) * nb ** dim
    va, vb = (na + 1) ** dim, (nb + 1) ** dim
    p = _pairs(call, dim, na, nb)
    read = 8 * dim * (va + vb) + 4 * (loc * ea + locb * eb)
    if call == "finder":
        return 8 * dim * (va + vb) + 8 * (loc * ea + loc * eb) + 8 * (ea + 1) + 8 * p, 4 * dim * p
    write = 8 * (ea + 1) + 4 * p + 4 * p + 4 * p + 8 * p  # indptr, indices, rows, counts, measures
    per_out = {(2, False): 1.09, (3, False): 2.27, (2, True): 1.3, (3, True): 6.38}[dim, call == "mixed"]
    flops = (108.6 if dim == 2 else 544.6 * (3 if call == "mixed" else 1)) * p
    if call in ("elements", "learned"):
        write += 8 * p + 8 * loc * dim * per_out * p
    if call == "mass":
        nnz = 3.64 * (na + nb) ** 2 if dim == 2 else 15 * (na + nb) ** 3
        write += 8 * va + 12 * nnz
        flops += (268.0 if dim == 2 else 900.0) * p
    return read + write, flops


def work(case):
    if case["call"] == "batch":
        each = [_one_work("count", *s) for s in _batch_sizes(case)]
        return {"bytes": sum(e[0] for e in each), "flops": sum(e[1] for e in each)}
    b, f = _one_work(case["call"], case["dim"], case["na"], case["nb"])
    return {"bytes": b, "flops": f}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

def _rand(shape, seed):
    g = torch.Generator(device=CUDA)
    g.manual_seed(int(seed))
    return torch.rand(shape, generator=g, device=CUDA, dtype=torch.float64)


def _measures(pos, enl):
    p = pos[enl.long()]
    e = p[:, 1:] - p[:, :1]
    if pos.shape[1] == 2:
        return 0.5 * (e[:, 0, 0] * e[:, 1, 1] - e[:, 0, 1] * e[:, 1, 0])
    return (e[:, 0] * torch.linalg.cross(e[:, 1], e[:, 2])).sum(1) / 6.0


def _grid(dim, n):
    """(positions, interior mask, node id of every cell's low corner)."""
    t = torch.arange(n + 1, device=CUDA, dtype=torch.float64) / n
    i = torch.arange(n + 1, device=CUDA)
    x = torch.stack([c.reshape(-1) for c in torch.meshgrid(*([t] * dim), indexing="ij")][::-1], 1)
    inner = torch.stack([((c > 0) & (c < n)).reshape(-1) for c in torch.meshgrid(*([i] * dim), indexing="ij")], 1).all(1)
    low = torch.zeros((n,) * dim, device=CUDA, dtype=torch.int64)
    for c in torch.meshgrid(*([i[:n]] * dim), indexing="ij"):
        low = low * (n + 1) + c
    return x, inner, low.reshape(-1)


def _simplices(dim, n, seed, diagonal):
    """Jittered split grid; the jitter of every vertex of an element that
    comes out below a tenth of its size is halved until none is."""
    pos, inner, low = _grid(dim, n)
    sx, sy = 1, n + 1
    if dim == 2:
        tris = ((0, sx, sx + sy), (0, sx + sy, sy)) if diagonal == 0 else ((0, sx, sy), (sx, sx + sy, sy))
        enl = torch.stack([torch.stack([low + o for o in t], 1) for t in tris], 1).reshape(-1, 3)
    else:
        s = (1, n + 1, (n + 1) ** 2)
        perms = ((0, 1), (0, 2), (1, 0), (1, 2), (2, 0), (2, 1))
        enl = torch.stack([torch.stack([low, low + s[a], low + s[a] + s[b], low + sum(s)], 1) for a, b in perms], 1)
        enl = enl.reshape(-1, 4)
    d = (2 * _rand(pos.shape, seed) - 1) * ((0.3 if dim == 2 else 0.25) / n) * inner[:, None]
    ref = _measures(pos, enl)
    while True:
        bad = _measures(pos + d, enl) / ref < 0.1
        if not bool(bad.any()):
            return pos + d, enl.int()
        d[torch.unique(enl[bad])] *= 0.5


def _cells(dim, n, seed):
    """Quadrilaterals (vertices jittered) or hexahedra (grid planes jittered)."""
    pos, inner, low = _grid(dim, n)
    s = (1, n + 1, (n + 1) ** 2)
    if dim == 2:
        pos = pos + (2 * _rand(pos.shape, seed) - 1) * (0.2 / n) * inner[:, None]
        ring = (0, s[0], s[0] + s[1], s[1])
    else:
        t = torch.arange(n + 1, device=CUDA, dtype=torch.float64) / n
        ax = t + (2 * _rand((3, n + 1), seed) - 1) * (0.2 / n) * ((t > 0) & (t < 1))
        z, y, x = torch.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
        pos = torch.stack([x.reshape(-1), y.reshape(-1), z.reshape(-1)], 1)
        ring = tuple(k + o for k in (0, s[2]) for o in (0, s[0], s[0] + s[1], s[1]))
    return pos, torch.stack([low + o for o in ring], 1).int()


def _parts(n, rng):
    """0 .. n-1 cut into up to 16 contiguous parts, in any order."""
    cuts = sorted(rng.randrange(n + 1) for _ in range(15))
    parts = [(lo, hi) for lo, hi in zip([0, *cuts], [*cuts, n]) if lo < hi]
    rng.shuffle(parts)
    return torch.cat([torch.arange(lo, hi, device=CUDA) for lo, hi in parts])


def _renumber(mesh, rng):
    pos, enl = mesh
    nodes, elements = _parts(pos.shape[0], rng), _parts(enl.shape[0], rng)
    place = torch.empty_like(nodes)
    place[nodes] = torch.arange(nodes.numel(), device=CUDA)
    return pos[nodes], place[enl[elements].long()].int()


def _meshes(case, seed):
    """(positions, element node ids) of A and of B."""
    dim, na, nb = case["dim"], case["na"], case["nb"]
    rng = random.Random(seed)
    a = _simplices(dim, na, 1, 0)
    b = _cells(dim, nb, 2) if case["call"] == "mixed" else _simplices(dim, nb, 2, 1)
    return _renumber(a, rng), _renumber(b, rng)


def _batch_meshes(case, seed):
    """{dim: (A's meshes, B's meshes)}."""
    out, rng = {}, random.Random(seed)
    sizes = list(enumerate(_batch_sizes(case)))
    rng.shuffle(sizes)
    for k, (dim, na, nb) in sizes:
        pair = out.setdefault(dim, ([], []))
        pair[0].append(_renumber(_simplices(dim, na, 2 * k + 1, 0), rng))
        pair[1].append(_renumber(_simplices(dim, nb, 2 * k + 2, 1), rng))
    return out


def _host(m):
    return m[0].cpu().numpy(), m[1].cpu().numpy()


def prepare(case, seed):
    s = {"case": dict(case)}
    if case["call"] == "finder":
        (pa, ea), (pb, eb) = (_host(m) for m in _meshes(case, seed))
        s["arrays"] = pa, ea.astype(np.int64), pb, eb.astype(np.int64)
        return s
    if case["call"] == "batch":
        # a context's results last until its next call: one for each dimension
        s["batches"] = [(gpu.Context(0), dim, *(gpu.DeviceMeshBatch([_host(m) for m in side]) for side in sides))
                        for dim, sides in sorted(_batch_meshes(case, seed).items())]
        return s
    s["context"] = gpu.Context(0)
    s["meshes"] = [gpu.DeviceMesh(*_host(m)) for m in _meshes(case, seed)]
    if case["call"] == "learned":
        data = os.path.join(os.path.dirname(os.path.abspath(gpu.__file__)), "data", "tet_counts_mlp.f32")
        s["context"].predictor_set(np.fromfile(data, dtype=np.float32))
    return s


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------

class _Device:
    """Device memory of a context; a tensor made of it keeps the context alive."""

    def __init__(self, ctx, ptr, shape, kind):
        self.owner = ctx
        self.__cuda_array_interface__ = {"data": (int(ptr), False), "shape": shape, "typestr": kind, "version": 2}


def _view(ctx, ptr, shape, kind):
    """A tensor on the context's own memory: no copy."""
    if 0 in shape or not ptr:
        return torch.empty((0,) * len(shape), device=CUDA, dtype={"<i4": torch.int32, "<i8": torch.int64}.get(kind, torch.float64))
    return torch.as_tensor(_Device(ctx, ptr, shape, kind), device=CUDA)


def _outputs(ctx, r, dim, nnodes_a):
    n, loc = r.npairs, dim + 1
    out = {"sum": float(r.sum), "nonempty": int(r.nonempty), "nout": int(r.nout), "max_count": int(r.max_count),
           "indptr": _view(ctx, r.indptr, (r.nelements_a + 1,), "<i8"), "indices": _view(ctx, r.indices, (n,), "<i4"),
           "rows": _view(ctx, r.rows, (n,), "<i4"), "counts": _view(ctx, r.counts, (n,), "<i4"),
           "measure": _view(ctx, r.measure, (n,), "<f8")}
    if r.elements:
        out["offsets"] = _view(ctx, r.offsets, (n + 1,), "<i8")
        out["elements"] = _view(ctx, r.elements, (r.elements_size, loc, dim), "<f8")
    if r.mass_indptr:
        out["mass_indptr"] = _view(ctx, r.mass_indptr, (nnodes_a + 1,), "<i8")
        out["mass_indices"] = _view(ctx, r.mass_indices, (r.mass_nnz,), "<i4")
        out["mass_values"] = _view(ctx, r.mass_values, (r.mass_nnz,), "<f8")
    return out


FLAGS = {"count": 0, "mixed": 0, "elements": gpu.ELEMENTS, "mass": gpu.MASS,
         "learned": gpu.ELEMENTS | gpu.LEARNED | gpu.DENSE}


def run(state):
    case = state["case"]
    if case["call"] == "finder":
        indptr, indices = gpu.tree_intersection_finder(*state["arrays"])
        return {"indptr": indptr, "indices": indices}
    if case["call"] == "batch":
        out = []
        for ctx, dim, a, b in state["batches"]:
            r, br = ctx.supermesh_batched(a, b)
            out.append(_outputs(ctx, r, dim, 0))
            out[-1]["pair_offsets"] = _view(ctx, br.pair_offsets, (br.nmeshes + 1,), "<i8")
            out[-1]["sums"] = _view(ctx, br.sums, (br.nmeshes,), "<f8")
        return out
    ctx = state["context"]
    a, b = state["meshes"]
    flags = FLAGS[case["call"]] | (gpu.SORTED if case["sorted"] else 0)
    r = (ctx.supermesh_mixed if case["call"] == "mixed" else ctx.supermesh)(a, b, flags=flags)
    return _outputs(ctx, r, case["dim"], a.nnodes)


# ---------------------------------------------------------------------------
# The same values by other means, in 64 bits
# ---------------------------------------------------------------------------

def _halfspaces(v):
    """Points on and outward normals of the faces of simplices v[n, d+1, d]."""
    n, loc, d = v.shape
    pts, nrm = [], []
    for k in range(loc):
        f = [j for j in range(loc) if j != k]
        p = v[:, f[0]]
        if d == 2:
            e = v[:, f[1]] - p
            m = torch.stack([e[:, 1], -e[:, 0]], 1)
        else:
            m = torch.linalg.cross(v[:, f[1]] - p, v[:, f[2]] - p)
        out = ((v[:, k] - p) * m).sum(1, keepdim=True) > 0
        pts.append(p)
        nrm.append(torch.where(out, -m, m))
    return torch.stack(pts, 1), torch.stack(nrm, 1)


def _distance(p, pts, nrm):
    """Scaled distances from planes; 0 where rounding alone parts a point from its plane."""
    d = ((p - pts) * nrm).sum(-1)
    return torch.where(d.abs() <= 1e-15 * nrm.abs().sum(-1), 0.0, d)


def _clip(poly, count, pts, nrm):
    """Convex polygons poly[n, V, d] (the first count[n] vertices) within the
    closed half-spaces."""
    for k in range(pts.shape[1]):
        n, cap, d = poly.shape
        at = torch.arange(cap, device=poly.device)
        nxt = torch.where(at[None] + 1 < count[:, None], at[None] + 1, 0)
        live = at[None] < count[:, None]
        dist = _distance(poly, pts[:, k, None], nrm[:, k, None])
        other = torch.gather(poly, 1, nxt[..., None].expand(-1, -1, d))
        dn = torch.gather(dist, 1, nxt)
        keep = live & (dist <= 0)
        cross = live & (((dist < 0) & (dn > 0)) | ((dist > 0) & (dn < 0)))
        t = torch.where(cross, dist / torch.where(cross, dist - dn, 1.0), 0.0)[..., None]
        new = poly + t * (other - poly)
        both = torch.stack([poly, new], 2).reshape(n, 2 * cap, d)
        mask = torch.stack([keep, cross], 2).reshape(n, 2 * cap)
        order = torch.argsort((~mask).int(), dim=1, stable=True)[:, : cap + 1]
        poly = torch.gather(both, 1, order[..., None].expand(-1, -1, d))
        count = mask.sum(1).clamp(max=cap + 1)
    return poly, count


def _overlap(a, b):
    """Areas / volumes of the intersections of the simplices a[n] and b[n]."""
    n, loc, d = a.shape
    count = torch.full((n,), 3, device=a.device)
    if d == 2:
        p, c = _clip(a, count, *_halfspaces(b))
        e = p[:, 1:] - p[:, :1]
        live = torch.arange(e.shape[1] - 1, device=a.device)[None] + 2 < c[:, None]
        return (0.5 * (e[:, :-1, 0] * e[:, 1:, 1] - e[:, :-1, 1] * e[:, 1:, 0]) * live).sum(1).abs()
    # the faces of the intersection are the parts of each one's faces within
    # the other; one that both have (on the domain's boundary) counts once
    total = torch.zeros(n, device=a.device, dtype=a.dtype)
    origin = a.mean(1)
    for v, w, first in ((a, b, True), (b, a, False)):
        pts, nrm = _halfspaces(v)
        wp, wn = _halfspaces(w)
        for k in range(loc):
            f = v[:, [j for j in range(loc) if j != k]]
            p, c = _clip(f, count, wp, wn)
            e = p[:, 1:] - p[:, :1]
            live = torch.arange(e.shape[1] - 1, device=a.device)[None] + 2 < c[:, None]
            area = (torch.linalg.cross(e[:, :-1], e[:, 1:]) * live[..., None]).sum(1)
            side = torch.sign((area * nrm[:, k]).sum(1))
            if not first:
                on = (_distance(f[:, :, None], wp[:, None], wn[:, None]) == 0).all(1)
                side = torch.where((on & ((wn * nrm[:, k, None]).sum(2) > 0)).any(1), 0.0, side)
            total += side * (area * (pts[:, k] - origin)).sum(1) / 6.0
    return total


def _candidates(a, b):
    """Pairs of elements whose boxes overlap, by A's element, then B's."""
    alo, ahi, blo, bhi = a.amin(1), a.amax(1), b.amin(1), b.amax(1)
    rows, cols = [], []
    step = max(1, (1 << 26) // b.shape[0])
    for k in range(0, a.shape[0], step):
        hit = torch.ones((min(step, a.shape[0] - k), b.shape[0]), dtype=torch.bool, device=a.device)
        for d in range(a.shape[2]):
            hit &= (ahi[k:k + step, None, d] > blo[None, :, d]) & (alo[k:k + step, None, d] < bhi[None, :, d])
        r, c = hit.nonzero(as_tuple=True)
        rows.append(r + k)
        cols.append(c)
    return torch.cat(rows), torch.cat(cols)


def _total(m):
    """Sum of the measures of A's elements: the domain, which B covers too."""
    return float(_measures(*m).abs().sum())


def exact(case, seed):
    if case["call"] == "finder":
        return None
    if case["call"] == "batch":
        sums = [np.array([_total(m) for m in side[0]]) for _, side in sorted(_batch_meshes(case, seed).items())]
        return [{"sum": float(s.sum()), "sums": s} for s in sums]
    a, b = _meshes(case, seed)
    out = {"sum": _total(a)}
    if case["sorted"] and a[1].shape[0] * b[1].shape[0] < 4e9:
        va, vb = a[0][a[1].long()], b[0][b[1].long()]
        rows, cols = _candidates(va, vb)
        parts = [_overlap(va[rows[k:k + (1 << 20)]], vb[cols[k:k + (1 << 20)]]) for k in range(0, rows.numel(), 1 << 20)]
        out["measure"] = torch.cat(parts)
    return out
