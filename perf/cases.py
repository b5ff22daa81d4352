"""The work that users of this framework have it do, as measurable cases.

Four kinds of call, each through the public entry points of manifolddmc_amd:

* ``extract``  a float32 field resident on the GPU -> the repaired halfedge mesh in the caller's
  device buffers (DualMarchingCubes.extract_raw, then copy_device);
* ``host``     a numpy field -> the mesh, its triangle list and its render vertices in a viewer's
  host buffers (DualMarchingCubes.run, triangles, render_vertices);
* ``batch``    many small grids at several iso-values each in one call
  (DualMarchingCubes.extract_batch_raw, then copy_device and batch_offsets);
* ``adjoint``  a training step's share: dual vertices of a field with grad, a loss on them and
  its gradient (manifolddmc_amd.autograd.dual_marching_cubes, loss.backward).

A program keeps one context per GPU for all its extractions, and buffers with room for any mesh
it expects; so do the cases.
"""
import functools
import json
import math

import numpy as np
import torch

import manifolddmc_amd as mdmc
from manifolddmc_amd.autograd import dual_marching_cubes

# the option sets in use: the reference's defaults, everything on, the dual mesh alone
FLAGS = {
    "default": mdmc.DEFAULT_FLAGS,
    "all": mdmc.PAD1 | mdmc.SURF_ITER | mdmc.ALL_POST,
    "dual": mdmc.PAD1 | mdmc.SURF_ITER,
    "all_unpadded": mdmc.SURF_ITER | mdmc.ALL_POST,
}


def listed():
    return [
        # the smallest call: one small object of a scene; launches and read-backs are all of it
        {"name": "blobs16", "kind": "extract", "field": "blobs", "nx": 16, "ny": 16, "nz": 16, "n": 8, "flags": "default", "refinement": 0},
        # an ordinary small volume with every post-process on
        {"name": "blobs64_all", "kind": "extract", "field": "blobs", "nx": 64, "ny": 64, "nz": 64, "n": 8, "flags": "all", "refinement": 0},
        # a field full of ambiguous faces: many non-manifold edges, so the repair is the work
        {"name": "lattice128_all", "kind": "extract", "field": "lattice", "nx": 128, "ny": 128, "nz": 128, "n": 4, "flags": "all", "refinement": 0},
        # a noisy scan cut to a ragged box, the reference's default options
        {"name": "gyroid201x77x131", "kind": "extract", "field": "gyroid", "nx": 201, "ny": 77, "nz": 131, "n": 3, "flags": "default", "refinement": 0},
        # a smooth object in a large volume: few cells meet the surface, reading the field is the work
        {"name": "blobs256", "kind": "extract", "field": "blobs", "nx": 256, "ny": 256, "nz": 256, "n": 8, "flags": "default", "refinement": 0},
        # a coarse field refined by two cuts per cell before extraction
        {"name": "lattice48_refined", "kind": "extract", "field": "lattice", "nx": 48, "ny": 48, "nz": 48, "n": 4, "flags": "default", "refinement": 2},
        # the benchmark's workload: a large noisy volume, every post-process
        {"name": "gyroid512_all", "kind": "extract", "field": "gyroid", "nx": 512, "ny": 512, "nz": 512, "n": 8, "flags": "all", "refinement": 0},
        # a viewer that loads a volume from disk and draws it
        {"name": "host_blobs128", "kind": "host", "field": "blobs", "nx": 128, "ny": 128, "nz": 128, "n": 8, "flags": "default", "refinement": 0},
        # a few small volumes at a time, as a service answers them
        {"name": "batch16x2", "kind": "batch", "grids": 16, "isos": 2, "lo": 16, "hi": 48, "shapes": 1, "flags": "all"},
        # a data set's worth of volumes of all sizes
        {"name": "batch64x4", "kind": "batch", "grids": 64, "isos": 4, "lo": 16, "hi": 192, "shapes": 5, "flags": "all"},
        # shape optimisation: a small field in an inner loop, and the benchmark's distance field
        {"name": "adjoint_spheres65", "kind": "adjoint", "field": "spheres", "nx": 65, "ny": 65, "nz": 65, "n": 8, "pad": True, "refinement": 0},
        {"name": "adjoint_spheres256", "kind": "adjoint", "field": "spheres", "nx": 256, "ny": 256, "nz": 256, "n": 32, "pad": True, "refinement": 0},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_dims(rng, lo, hi):
    side = _log_uniform(rng, lo, hi)
    dims = [max(lo, int(round(side * rng.uniform(0.6, 1.0)))) for _ in range(3)]
    dims = dims if rng.random() < 0.7 else [side, side, side]
    return dict(zip(("nx", "ny", "nz"), dims))


def _dims(case):
    return [case["nx"], case["ny"], case["nz"]]


def draw(rng):
    """One more case of the ranges above."""
    kind = rng.choices(["extract", "host", "batch", "adjoint"], [10, 2, 4, 4])[0]
    if kind == "batch":
        lo = 16
        hi = rng.choice([32, 48, 96, 160])
        return {"kind": kind, "grids": rng.randint(3, 48), "isos": rng.randint(1, 4), "lo": lo, "hi": hi,
                "shapes": rng.randrange(1 << 20), "flags": rng.choice(["default", "all"])}
    if kind == "adjoint":
        field = rng.choice(["spheres", "blobs"])
        refinement = rng.choice([0, 0, 0, 1])
        return {"kind": kind, "field": field, "n": rng.randint(4, 32), "pad": rng.random() < 0.7, "refinement": refinement,
                **_draw_dims(rng, 16, 240 if not refinement else 96)}
    field = rng.choice(["blobs", "blobs", "gyroid", "gyroid", "lattice"])
    refinement = rng.choice([0, 0, 0, 0, 1, 2]) if kind == "extract" else 0
    hi = {"blobs": 400, "gyroid": 400, "lattice": 200}[field]
    if kind == "host":
        hi = 160
    if refinement:
        hi = 72
    dims = _draw_dims(rng, 16, hi)
    n = {"blobs": rng.randint(1, 32), "gyroid": rng.randint(1, max(1, min(8, min(dims.values()) // 10))), "lattice": rng.randint(3, 6)}[field]
    return {"kind": kind, "field": field, "n": n, "flags": rng.choice(["default", "default", "all", "all", "dual", "all_unpadded"]),
            "refinement": refinement, **dims}


# ---------------------------------------------------------------------------- fields
def _device():
    return torch.device("cuda") if torch.cuda.is_available() else torch.device("cpu")


def _axes(dims, dev):
    """Sample positions of the three axes in [0, 1], as broadcastable (z, y, x)."""
    nx, ny, nz = dims
    t = [torch.arange(k, device=dev, dtype=torch.float32) / max(k - 1, 1) for k in (nz, ny, nx)]
    return t[0][:, None, None], t[1][None, :, None], t[2][None, None, :]


def _field(kind, dims, n, seed, dev, noise=0.1):
    """A float32 field [z][y][x] and the iso-value it is looked at with."""
    rng = np.random.default_rng(seed)
    nx, ny, nz = dims
    z, y, x = _axes(dims, dev)
    if kind == "blobs":  # a sum of Gaussians in the unit cube
        f = torch.zeros((nz, ny, nx), device=dev)
        for _ in range(n):
            c = rng.uniform(0.2, 0.8, 3)
            k = -0.5 / rng.uniform(0.05, 0.15) ** 2
            f += torch.exp(k * (z - c[2]) ** 2) * torch.exp(k * (y - c[1]) ** 2) * torch.exp(k * (x - c[0]) ** 2)
        return f, 0.5
    if kind == "gyroid":  # n periods along the longest axis, plus noise of a measured volume
        g = torch.Generator(device=dev)
        g.manual_seed(int(rng.integers(1 << 31)))
        m = max(dims)
        w = 2.0 * math.pi * n / m
        x, y, z = x * (w * (nx - 1)), y * (w * (ny - 1)), z * (w * (nz - 1))
        f = torch.sin(x) * torch.cos(y) + torch.sin(y) * torch.cos(z) + torch.sin(z) * torch.cos(x)
        f += noise * torch.randn((nz, ny, nx), device=dev, generator=g)
        return f, 0.0
    if kind == "lattice":  # uniform random values every n samples, trilinear in between
        lat = torch.from_numpy(rng.uniform(-1.0, 1.0, [k // n + 2 for k in (nz, ny, nx)]).astype(np.float32)).to(dev)
        for axis, k in enumerate((nz, ny, nx)):
            p = torch.arange(k, device=dev, dtype=torch.float32) * ((k // n) / k)
            i = p.long()
            u = (p - i).reshape([-1 if a == axis else 1 for a in range(3)])
            lat = lat.index_select(axis, i) * (1.0 - u) + lat.index_select(axis, i + 1) * u
        return lat.contiguous(), 0.0
    if kind == "spheres":  # signed distance to a union of spheres
        f = torch.full((nz, ny, nx), float("inf"), device=dev)
        for _ in range(n):
            c = rng.uniform(0.15, 0.85, 3)
            r = rng.uniform(0.03, 0.12)
            torch.minimum(f, torch.sqrt((z - c[2]) ** 2 + (y - c[1]) ** 2 + (x - c[0]) ** 2) - r, out=f)
        return f, 0.0
    raise ValueError(kind)


def _delta(dims):
    return tuple(1.0 / max(k - 1, 1) for k in dims)


def _batch_fields(case, seed, dev):
    """(field, dims, delta, iso-values) of every grid: even ones blobs, odd ones noisy gyroids, sides
    log-uniform per axis, iso-values between the field's 10% and 90% quantiles.  The sides belong to
    the case (a service sees the same volumes' shapes again), the values to the seed."""
    shapes = np.random.default_rng(case["shapes"])
    rng = np.random.default_rng(seed)
    out = []
    for i in range(case["grids"]):
        dims = [int(round(math.exp(shapes.uniform(math.log(case["lo"]), math.log(case["hi"]))))) for _ in range(3)]
        n = int(shapes.integers(4, 33)) if i % 2 == 0 else int(shapes.integers(1, max(2, min(12, max(dims) // 10))))
        f, _ = _field("blobs" if i % 2 == 0 else "gyroid", dims, n, int(rng.integers(1 << 31)), dev, noise=0.05)
        sample = f.reshape(-1)[:: max(1, f.numel() // 100000)]
        q = torch.quantile(sample, torch.tensor([0.1, 0.9], device=dev)).tolist()
        out.append((f, dims, _delta(dims), sorted(float(v) for v in rng.uniform(q[0], q[1], case["isos"]))))
    return out


# ---------------------------------------------------------------------------- what a program has in hand
_contexts = {}


def _context():
    dev = torch.cuda.current_device()
    if dev not in _contexts:
        _contexts[dev] = mdmc.DualMarchingCubes(device=dev)
    return _contexts[dev]


@functools.lru_cache(maxsize=None)
def _room(case_text):
    """Vertices (and faces) the program's buffers hold: a few times those of the fields it has seen."""
    case = json.loads(case_text)
    most = max(_count_quads(case, seed) for seed in range(3))
    blobs = case["kind"] != "batch" and case["field"] == "blobs"
    return (8 if blobs else 3 if case["kind"] == "batch" and case["grids"] < 12 else 2) * most + 20000


def _buffers(room, dev):
    """The mesh as mesh_torch and mesh_numpy lay it out, with room for `room` vertices and faces."""
    shapes = {"positions": ((room, 3), torch.float32), "normals": ((room, 3), torch.float32), "halfedges": ((4 * room, 4), torch.int32),
              "face_halfedge": ((room,), torch.int32), "face_attr": ((room,), torch.int16), "vertex_flags": ((room,), torch.uint8),
              "vertex_halfedge": ((room,), torch.int32)}
    return {k: torch.zeros(shape, dtype=t, device=dev) for k, (shape, t) in shapes.items()}


def prepare(case, seed):
    dev = _device()
    state = {"case": case, "dmc": _context()}
    if case["kind"] != "adjoint":
        room = _room(json.dumps({k: v for k, v in case.items() if k != "name"}, sort_keys=True))
        state["room"] = room
        state["mesh"] = _buffers(room, "cpu" if case["kind"] == "host" else dev)
    if case["kind"] == "batch":
        grids = _batch_fields(case, seed, dev)
        state["fields"] = [f for f, _, _, _ in grids]
        state["grids"] = [(f.data_ptr(), tuple(dims), (0.0, 0.0, 0.0), delta, True) for f, dims, delta, _ in grids]
        state["isos"] = [isos for _, _, _, isos in grids]
    else:
        f, state["iso"] = _field(case["field"], _dims(case), case["n"], seed, dev)
        state["field"] = f.cpu().numpy() if case["kind"] == "host" else f
        state["delta"] = _delta(_dims(case))
        if case["kind"] == "adjoint":
            state["centre"] = torch.tensor([0.5, 0.5, 0.5], device=dev)
    if case["kind"] == "host":
        state["mesh"] = {k: v.numpy() for k, v in state["mesh"].items()}
        state["mesh"]["face_attr"] = state["mesh"]["face_attr"].view(np.uint16)
        state["triangles"] = np.zeros((room, 6), np.uint32)
        state["render"] = np.zeros((room, 10), np.float32)
    torch.cuda.synchronize()
    return state


def _counts(st):
    return np.array([st.n_vertices, st.n_halfedges, st.n_faces, st.n_dmc_vertices, st.n_dmc_quads, st.nm_edges4, st.nm_edges3, st.n_edges,
                     st.nm_vertices, st.split_iterations, st.anomalies] + list(st.quads_with_nm), np.int64)


def _copy_mesh(d, st, state):
    if max(st.n_vertices, st.n_faces) > state["room"]:
        raise RuntimeError("the mesh is larger than the buffers")
    if st.n_vertices:
        d.copy_device(**{k: v.data_ptr() for k, v in state["mesh"].items()})
    return state["mesh"]


def _loss(positions, centre):
    """Mean squared distance of the vertices to a sphere."""
    return ((torch.linalg.norm(positions - centre, dim=1) - 0.3) ** 2).mean()


def run(state):
    case, d = state["case"], state["dmc"]
    kind = case["kind"]
    if kind == "extract":
        st = d.extract_raw(state["field"].data_ptr(), _dims(case), (0.0, 0.0, 0.0), state["delta"], state["iso"], FLAGS[case["flags"]],
                           case["refinement"], True)
        return {"mesh": _copy_mesh(d, st, state), "counts": _counts(st)}
    if kind == "batch":
        st = d.extract_batch_raw(state["grids"], state["isos"], FLAGS[case["flags"]])
        return {"mesh": _copy_mesh(d, st, state), "offsets": d.batch_offsets(), "counts": _counts(st)}
    if kind == "host":
        flags = FLAGS[case["flags"]]
        d.enable_surface_to_vertex_iteration = bool(flags & mdmc.SURF_ITER)
        d.simplify_p3x3y_color = bool(flags & mdmc.P3X3Y_COLOR)
        d.simplify_p3x3y_old = bool(flags & mdmc.P3X3Y_OLD)
        d.simplify_p3333 = bool(flags & mdmc.P3333)
        d.split_non_manifold_halfedges = bool(flags & mdmc.SPLIT_NM)
        d.detect_non_manifold_vertices = bool(flags & mdmc.DETECT_NM_VERTS)
        m = d.run(state["iso"], state["field"], (0.0, 0.0, 0.0), state["delta"], case["refinement"], bool(flags & mdmc.PAD1))
        for k, buf in state["mesh"].items():
            v = getattr(m, k)
            buf[:len(v)] = v
        t, r = d.triangles(), d.render_vertices()
        state["triangles"][:len(t)] = t
        state["render"][:len(r)] = r
        return {"mesh": state["mesh"], "triangles": state["triangles"].view(np.int32), "render": state["render"], "counts": _counts(d.last_stats)}
    if kind == "adjoint":
        f = state["field"].detach().requires_grad_(True)
        pos, quads = dual_marching_cubes(f, state["iso"], (0.0, 0.0, 0.0), state["delta"], pad=case["pad"], refinement=case["refinement"])
        loss = _loss(pos, state["centre"])
        loss.backward()
        return {"loss": loss.detach(), "grad": f.grad}
    raise ValueError(kind)


# ---------------------------------------------------------------------------- the work of a pass
def _refined(f, refinement):
    """The field sampled with `refinement` more points between neighbours (trilinear)."""
    if refinement:
        f = torch.nn.functional.interpolate(f[None, None], size=[(k - 1) * (refinement + 1) + 1 for k in f.shape], mode="trilinear",
                                            align_corners=True)[0, 0]
    return f


def _quads(f, iso, pad):
    """Quads of the dual mesh: one per grid edge across the surface with four cells around it."""
    s = f >= iso
    n = 0
    for axis in range(3):
        k = s.shape[axis]
        c = s.narrow(axis, 1, k - 1) != s.narrow(axis, 0, k - 1)
        if not pad:  # without the duplicated border, edges on the grid's faces carry no quad
            for other in range(3):
                if other != axis:
                    c = c.narrow(other, 1, max(c.shape[other] - 2, 0))
        n += int(c.sum())
    return n


# one quad's share of the mesh: a vertex (position, normal, flag, halfedge), four halfedge
# records, a face (first halfedge, attribute); the repaired mesh has about as many
_MESH_BYTES = (12 + 12 + 1 + 4) + 4 * 16 + (4 + 2)
# a dual vertex: four crossings averaged, the corner gradients, one interpolated normal
_VERTEX_FLOPS = 4 * 8 + 24 * 2 + 3 * 14 + 12


def _count_quads(case, seed):
    dev = _device()
    if case["kind"] == "batch":
        return sum(_quads(f, iso, True) for f, _, _, isos in _batch_fields(case, seed, dev) for iso in isos)
    f, iso = _field(case["field"], _dims(case), case["n"], seed, dev)
    pad = case["pad"] if case["kind"] == "adjoint" else bool(FLAGS[case["flags"]] & mdmc.PAD1)
    return _quads(_refined(f, case["refinement"]), iso, pad)


def work(case):
    """Each input read once and each output written once; seed 0 stands for all seeds."""
    q = _count_quads(case, 0)
    if case["kind"] == "batch":
        return {"bytes": sum(4 * f.numel() for f, _, _, _ in _batch_fields(case, 0, _device())) + _MESH_BYTES * q, "flops": _VERTEX_FLOPS * q}
    field = 4 * case["nx"] * case["ny"] * case["nz"]
    if case["kind"] == "adjoint":  # field in, positions and quads out, gradient of the positions in, of the field out
        return {"bytes": field + (12 + 32) * q + 12 * q + field, "flops": 2 * 4 * 8 * q + 30 * q}
    out = _MESH_BYTES * q
    if case["kind"] == "host":  # the same, then triangles and render vertices
        out += (24 + 40) * q
    return {"bytes": field + out, "flops": _VERTEX_FLOPS * q}


# ---------------------------------------------------------------------------- 64-bit values
# A cube's corner k is at (k & 1, k >> 1 & 1, k >> 2 & 1); its edges as corner pairs, its faces as
# four corners (two by two, so that corners 0 and 3 are opposite).
_EDGES = [(0, 1), (1, 3), (2, 3), (0, 2), (4, 5), (5, 7), (6, 7), (4, 6), (0, 4), (1, 5), (3, 7), (2, 6)]
_FACES = [(0, 1, 2, 3), (4, 5, 6, 7), (0, 1, 4, 5), (2, 3, 6, 7), (0, 2, 4, 6), (1, 3, 5, 7)]


def _edge(a, b):
    return _EDGES.index((min(a, b), max(a, b)))


def _contours(s, iso):
    """Cells' corner values [N, 8] -> for every surface contour of every cell, in order of (cell,
    smallest edge), its cell and the edges it crosses [V, 12].  On a face crossed four times the
    contour goes as the bilinear interpolant's saddle says."""
    n = s.shape[0]
    inside = s >= iso
    link = torch.zeros((n, 12, 12), dtype=torch.bool, device=s.device)

    def connect(a, b, where):
        link[:, a, b] |= where
        link[:, b, a] |= where

    for c in _FACES:
        v = [s[:, k] for k in c]
        i = [inside[:, k] for k in c]
        ring = [_edge(c[0], c[1]), _edge(c[1], c[3]), _edge(c[2], c[3]), _edge(c[0], c[2])]
        across = [i[0] != i[1], i[1] != i[3], i[2] != i[3], i[0] != i[2]]
        four = across[0] & across[1] & across[2] & across[3]
        for a in range(4):
            for b in range(a):
                connect(ring[a], ring[b], across[a] & across[b] & ~four)
        saddle = (v[0] * v[3] - v[1] * v[2]) / (v[0] + v[3] - v[1] - v[2]) >= iso
        # corners 0 and 3 are cut off when they lie on the other side than the saddle, else 1 and 2
        cut03 = four & (i[0] != saddle)
        cut12 = four & (i[0] == saddle)
        connect(ring[0], ring[3], cut03)
        connect(ring[1], ring[2], cut03)
        connect(ring[0], ring[1], cut12)
        connect(ring[2], ring[3], cut12)
    crossed = torch.stack([inside[:, a] != inside[:, b] for a, b in _EDGES], 1)
    index = torch.arange(12, dtype=torch.int8, device=s.device)
    label = torch.where(crossed, index, torch.full_like(index, 12))
    for _ in range(6):  # a contour has at most 12 edges: its smallest reaches all within 6 steps
        near = torch.where(link, label[:, None, :], torch.full_like(label, 12)[:, None, :]).amin(2)
        label = torch.minimum(label, near)
    first = (label == index) & crossed
    cell, edge = torch.nonzero(first, as_tuple=True)
    return cell, (label[cell] == edge[:, None].to(torch.int8)) & crossed[cell]


def exact(case, seed):
    """Only the adjoint's outputs have a 64-bit value: the loss on the means of the contours' edge
    crossings and its gradient, with the topology of the float32 field.  The other calls move vertices
    along a branching search and merge or split them, so a change of precision changes the mesh
    itself; for those the float32 result is the definition."""
    if case["kind"] != "adjoint":
        return None
    dev = _device()
    field, iso = _field(case["field"], _dims(case), case["n"], seed, dev)
    f = field.double().requires_grad_(True)
    r, pad, dims = case["refinement"], int(case["pad"]), _dims(case)
    delta = np.array([np.float32(v) for v in _delta(dims)]).astype(np.float64) / (r + 1)

    def processed(t):
        """The refined and padded grid: trilinear between the samples, its border duplicated."""
        for axis, k in enumerate((dims[2], dims[1], dims[0])):
            p = torch.arange(-pad, (k - 1) * (r + 1) + 1 + pad, device=dev).clamp(0, (k - 1) * (r + 1))
            i = torch.div(p, r + 1, rounding_mode="floor")
            if r == 0:
                t = t.index_select(axis, i)
                continue
            u = ((p - i * (r + 1)).to(t.dtype) / (r + 1)).reshape([-1 if a == axis else 1 for a in range(3)])
            t = t.index_select(axis, i) * (1 - u) + t.index_select(axis, (i + 1).clamp(max=k - 1)) * u
        return t

    proc = processed(f)
    nz, ny, nx = proc.shape
    with torch.no_grad():
        inside = (processed(field) if r else proc) >= iso
        corner = lambda k: inside[k >> 2 & 1:nz - 1 + (k >> 2 & 1), k >> 1 & 1:ny - 1 + (k >> 1 & 1), k & 1:nx - 1 + (k & 1)]
        n_in = sum(corner(k).to(torch.int8) for k in range(8))
        cz, cy, cx = torch.nonzero((n_in > 0) & (n_in < 8), as_tuple=True)
    at = [((cz + (k >> 2 & 1)) * ny + cy + (k >> 1 & 1)) * nx + cx + (k & 1) for k in range(8)]
    s = torch.stack([proc.reshape(-1)[i] for i in at], 1)
    with torch.no_grad():
        cell, member = _contours(s.detach(), iso)
    s = s[cell]
    m = member.double()
    local = torch.zeros((len(cell), 3), dtype=torch.float64, device=dev)
    for e, (a, b) in enumerate(_EDGES):
        t = torch.where(member[:, e], (iso - s[:, a]) / torch.where(member[:, e], s[:, b] - s[:, a], torch.ones_like(s[:, a])), 0.0)
        axis = (b - a).bit_length() - 1
        cross = [t if k == axis else torch.full_like(t, float(a >> k & 1)) for k in range(3)]
        cross[axis] = t + float(a >> axis & 1)
        local = local + torch.stack(cross, 1) * m[:, e:e + 1]
    local = local / m.sum(1, keepdim=True)
    ijk = torch.stack([cx[cell], cy[cell], cz[cell]], 1).double()
    pos = torch.from_numpy(-pad * delta).to(dev) + (ijk + local) * torch.from_numpy(delta).to(dev)
    loss = _loss(pos, torch.tensor([0.5, 0.5, 0.5], dtype=torch.float64, device=dev))
    loss.backward()
    return {"loss": loss.detach(), "grad": f.grad}
