"""Timed workloads of the implicit-modeling library, through its Python API.

A case is a dict of plain values: what is done (``do``), the mesh it is done to
(``mesh``, and its size: ``level`` subdivisions of a displaced icosphere, or
``major`` x ``minor`` segments of a noisy torus), and ``span``, the number of
voxels along the mesh's largest extent.  Meshes are made on the GPU from the
seed alone and are closed and outward oriented.

``listed`` names the workloads, ``draw`` gives one more of the same ranges,
``prepare`` makes what a program holds before the call, ``run`` is one pass,
``work`` its compulsory bytes and operations, ``exact`` its result in 64 bits
where the result has a value that does not depend on the library.

How many leaves or triangles come out depends on the mesh.  Like a program
that takes many meshes, a state holds buffers large enough for any mesh of its
case, and a pass leaves its result at their start (the rest stays zero).
"""
import math
import random

import numpy as np
import torch

import baby_shark_amd as bs

LEAF_BYTES = 16 + 64 + 2048  # origin, mask and values of one 8^3 leaf
ISO_EXTENT = 2.06            # largest extent of a displaced icosphere of radius 1
TORUS_R, TORUS_r = 1.0, 0.35


def listed():
    return [
        # the small end-to-end workload's conversion: one part, a coarse grid; latency and launches
        {"name": "convert_torus_16k", "do": "convert", "mesh": "torus", "major": 128, "minor": 64, "span": 135,
         "band": 3, "signs": "voxel"},
        # the headline conversion: a 1.3 M triangle scan at a fine grid
        {"name": "convert_icosphere_1310k", "do": "convert", "mesh": "icosphere", "level": 8, "span": 1050,
         "band": 3, "signs": "voxel"},
        # the same mesh, known to be closed: shared signs
        {"name": "convert_shared_1310k", "do": "convert", "mesh": "icosphere", "level": 8, "span": 1050,
         "band": 3, "signs": "shared"},
        # a library of parts voxelized in one call
        {"name": "batch_20_parts", "do": "batch", "count": 20, "lo": 1000, "hi": 200000, "span": 256, "band": 3},
        # the voxel remesher on a scan of the bunny's size, host soup in, host soup out
        {"name": "remesh_13k", "do": "remesh", "mesh": "torus", "major": 114, "minor": 57, "span": 500,
         "method": "manifold"},
        # the small workload's union with a primitive, which leaves tiles
        {"name": "union_torus_sphere", "do": "csg", "op": "union", "mesh": "torus", "major": 128, "minor": 64,
         "span": 135, "with": "sphere"},
        # two large parts, one cut from the other
        {"name": "subtract_2x328k", "do": "csg", "op": "subtract", "mesh": "icosphere", "level": 7, "span": 2060,
         "with": "mesh"},
        # a large part grown by 20 voxels
        {"name": "offset_out_328k", "do": "offset", "mesh": "icosphere", "level": 7, "span": 2060, "voxels": 20.0},
        # a small scan shrunk by 5 voxels, as before hollowing it
        {"name": "offset_in_13k", "do": "offset", "mesh": "torus", "major": 114, "minor": 57, "span": 250,
         "voxels": -5.0},
        # both meshers on a large volume
        {"name": "dual_contour_328k", "do": "mesh", "method": "feature", "mesh": "icosphere", "level": 7,
         "span": 2060, "band": 3},
        {"name": "marching_cubes_328k", "do": "mesh", "method": "manifold", "mesh": "icosphere", "level": 7,
         "span": 2060, "band": 3},
        # a whole program: a scan hollowed, filled with an IWP lattice, clipped and meshed
        {"name": "lightweighting_20k", "do": "lightweight", "mesh": "icosphere", "level": 5, "span": 250},
    ]


def _log_uniform(rng, lo, hi):
    return lo * (hi / lo) ** rng.random()


def _draw_mesh(rng, most_tris, lo_span, hi_span):
    c = {"span": round(_log_uniform(rng, lo_span, hi_span), 3)}
    if rng.random() < 0.5:
        level = rng.randint(3, 8)
        while 20 * 4 ** level > most_tris:
            level -= 1
        c.update(mesh="icosphere", level=level)
    else:
        tris = _log_uniform(rng, 1000.0, most_tris)
        minor = max(8, int(math.sqrt(tris / 4.0)) + rng.randint(-3, 3))
        c.update(mesh="torus", minor=minor, major=2 * minor + rng.randint(-5, 5))
    return c


def draw(rng):
    do = rng.choice(["convert", "convert", "batch", "remesh", "csg", "csg", "offset", "offset", "mesh", "mesh",
                     "lightweight"])
    if do == "convert":
        c = _draw_mesh(rng, 1.4e6, 64, 1050)
        c.update(band=rng.randint(0, 3), signs=rng.choice(["voxel", "shared"]))
    elif do == "batch":
        c = {"count": rng.randint(3, 20), "lo": 1000, "hi": rng.choice([20000, 200000]),
             "span": rng.randint(64, 256), "band": rng.randint(1, 3)}
    elif do == "remesh":
        c = _draw_mesh(rng, 4e4, 64, 500)
        c.update(method=rng.choice(["manifold", "feature"]))
    elif do == "csg":
        c = _draw_mesh(rng, 3.5e5, 100, 2060)
        c.update(op=rng.choice(["union", "subtract", "intersect"]), **{"with": rng.choice(["mesh", "sphere"])})
    elif do == "offset":
        c = _draw_mesh(rng, 3.5e5, 100, 2060)
        c.update(voxels=round(rng.choice([1, -1]) * _log_uniform(rng, 1.0, 20.0), 3))
        if c["voxels"] < 0:
            c["voxels"] = max(c["voxels"], -10.0)
    elif do == "mesh":
        c = _draw_mesh(rng, 3.5e5, 64, 2060)
        c.update(method=rng.choice(["manifold", "feature"]), band=rng.randint(0, 3))
    else:
        c = _draw_mesh(rng, 4e4, 120, 250)
    return {"do": do, **c}


# ---------------------------------------------------------------- meshes
def _unit_icosphere(level):
    """(20 * 4^level, 3, 3) float64 soup on the GPU; an edge's midpoint is the same value from both sides."""
    t = (1.0 + 5.0 ** 0.5) / 2.0
    v = torch.tensor([[-1, t, 0], [1, t, 0], [-1, -t, 0], [1, -t, 0], [0, -1, t], [0, 1, t], [0, -1, -t],
                      [0, 1, -t], [t, 0, -1], [t, 0, 1], [-t, 0, -1], [-t, 0, 1]], dtype=torch.float64)
    f = torch.tensor([[0, 11, 5], [0, 5, 1], [0, 1, 7], [0, 7, 10], [0, 10, 11], [1, 5, 9], [5, 11, 4], [11, 10, 2],
                      [10, 7, 6], [7, 1, 8], [3, 9, 4], [3, 4, 2], [3, 2, 6], [3, 6, 8], [3, 8, 9], [4, 9, 5],
                      [2, 4, 11], [6, 2, 10], [8, 6, 7], [9, 8, 1]])
    s = (v / v.norm(dim=1, keepdim=True)).cuda()[f.cuda()]
    for _ in range(level):
        a, b, c = s[:, 0], s[:, 1], s[:, 2]
        ab, bc, ca = a + b, b + c, c + a
        ab, bc, ca = (m / torch.sqrt(m[:, 0:1] ** 2 + m[:, 1:2] ** 2 + m[:, 2:3] ** 2) for m in (ab, bc, ca))
        s = torch.stack([torch.stack([a, ab, ca], 1), torch.stack([b, bc, ab], 1), torch.stack([c, ca, bc], 1),
                         torch.stack([ab, bc, ca], 1)], 1).reshape(-1, 3, 3)
    return s


def _displaced_icosphere(level, seed):
    """Radius 1 + 0.05 * three octaves of random waves (frequencies about 4, 8 and 16)."""
    rng = np.random.default_rng(seed)
    p = _unit_icosphere(level)
    x, y, z = p[..., 0], p[..., 1], p[..., 2]
    d = torch.zeros_like(x)
    for octave, gain in enumerate((0.57, 0.29, 0.14)):
        w = rng.normal(size=(6, 3)) * 4.0 * 2 ** octave
        for (wx, wy, wz), phase in zip(w.tolist(), rng.uniform(0, 2 * math.pi, 6).tolist()):
            d += gain / 6 * 2 * torch.sin(wx * x + wy * y + wz * z + phase)
    return p * (1.0 + 0.05 * d.clamp(-1, 1))[..., None]


def _torus(major, minor, seed):
    """2 * major * minor triangles about the z axis, the tube's radius noisy by 0.01."""
    rng = np.random.default_rng(seed)
    u = torch.arange(major, dtype=torch.float64, device="cuda") * (2 * math.pi / major)
    v = torch.arange(minor, dtype=torch.float64, device="cuda") * (2 * math.pi / minor)
    u, v = torch.meshgrid(u, v, indexing="ij")
    r = TORUS_r + torch.from_numpy(rng.uniform(-0.01, 0.01, (major, minor))).cuda()
    q = TORUS_R + r * torch.cos(v)
    p = torch.stack([q * torch.cos(u), q * torch.sin(u), r * torch.sin(v)], -1)
    p10, p01 = p.roll(-1, 0), p.roll(-1, 1)
    p11 = p10.roll(-1, 1)
    return torch.cat([torch.stack([p, p10, p11], 2).reshape(-1, 3, 3), torch.stack([p, p11, p01], 2).reshape(-1, 3, 3)])


def _mesh(case, seed):
    """(soup in float64 on the GPU, its nominal extent)."""
    if case["mesh"] == "torus":
        return _torus(case["major"], case["minor"], seed), 2.0 * (TORUS_R + TORUS_r)
    return _displaced_icosphere(case["level"], seed), ISO_EXTENT


def _f32(soup):
    return soup.to(torch.float32).contiguous()


def _batch_meshes(case, seed):
    """(soup, voxel size) of each part: triangle counts log-uniform in [lo, hi], tori and icospheres in turn."""
    rng = random.Random(case["count"] * 1000003 + case["hi"])  # the sizes belong to the case, the shapes to the seed
    out = []
    for i in range(case["count"]):
        tris = _log_uniform(rng, case["lo"], case["hi"])
        if i % 2 == 0:
            minor = max(3, round(math.sqrt(tris / 4.0)))
            soup, ext = _mesh({"mesh": "torus", "major": 2 * minor, "minor": minor}, seed * 1000 + i)
        else:
            level = min(6, max(3, round(math.log(tris / 20.0, 4))))
            soup, ext = _mesh({"mesh": "icosphere", "level": level}, seed * 1000 + i)
        out.append((_f32(soup), ext / case["span"]))
    return out


# ---------------------------------------------------------------- prepare and run
def _convert(soup, h, band, signs="voxel"):
    return bs.MeshToVolume().with_voxel_size(h).with_narrow_band_width(band).with_shared_signs(
        signs == "shared").convert(soup)


def _mesher(method, h):
    m = bs.MarchingCubesMesher() if method == "manifold" else bs.DualContouringMesher()
    return m.with_voxel_size(h)


def _leaf_room(n):
    n = int(n)
    return {"origins": torch.zeros((n, 4), dtype=torch.int32, device="cuda"),
            "masks": torch.zeros((n, 8), dtype=torch.int64, device="cuda"),
            "values": torch.zeros((n, 512), dtype=torch.float32, device="cuda")}


def _room(case):
    """Leaves that any mesh of the case fits."""
    do, area = case["do"], _area(case["mesh"], case["span"])
    n = _leaves(area, case.get("band", 3))
    if do == "csg":
        n = 2 * n if case["with"] == "mesh" else n + _ball_leaves(case)
    elif do == "offset":
        n = _leaves(area, 3 + abs(case["voxels"]))
    elif do == "lightweight":
        n = (case["span"] / 8 + 4) ** 3  # the lattice fills the part
    return 1.5 * n + 500


def _triangle_room(case):
    if case["do"] == "lightweight":
        return int(40 * _area(case["mesh"], case["span"]) + 20000)
    return int(4.5 * _area(case["mesh"], case["span"]) + 5000)


def prepare(case, seed):
    do = case["do"]
    if do == "batch":
        parts = _batch_meshes(case, seed)
        room = 1.5 * _leaves(_area("icosphere", case["span"]), case["band"]) + 500
        return {"case": case, "soups": [s for s, _ in parts], "h": [h for _, h in parts],
                "leaves": [_leaf_room(room) for _ in parts]}
    soup, ext = _mesh(case, seed)
    h = ext / case["span"]
    st = {"case": case, "h": h}
    if do not in ("remesh", "mesh"):
        st["leaves"] = _leaf_room(_room(case))
    if do in ("mesh", "lightweight"):
        st["triangles"] = torch.zeros((_triangle_room(case), 3, 3), dtype=torch.float32, device="cuda")
    if do == "convert":
        st["soup"] = _f32(soup)
    elif do == "remesh":
        st["soup"] = _f32(soup).cpu().numpy()  # as read from a file
        st["triangles"] = torch.zeros((_triangle_room(case), 3, 3), dtype=torch.float32)
    elif do == "lightweight":
        st["soup"] = _f32(soup * 25.0 + torch.tensor([0.0, 0.0, 25.0], dtype=torch.float64, device="cuda"))
        st["h"] = h * 25.0
    else:
        st["volume"] = _convert(_f32(soup), h, case.get("band", 3))
    if do == "csg":
        if case["with"] == "sphere":
            st["other"] = bs.VolumeBuilder(voxel_size=h).sphere(0.5, (1.0, 0.0, 0.0))
        else:
            other, _ = _mesh(case, seed + 7919)
            shift = torch.tensor([0.3, 0.0, 0.0], dtype=torch.float64, device="cuda")
            st["other"] = _convert(_f32(other + shift), h, 3)
    return st


def _keep(room, *volumes):
    """The volumes' leaf arrays into the state's buffers.  The volumes are the library's memory: the copies end
    before the volumes do."""
    for out, v in zip(room, volumes):
        for name, t in zip(("origins", "masks", "values"), v.device_arrays(copy=False)):
            out[name][:t.shape[0]].copy_(t)
    torch.cuda.current_stream().synchronize()
    return room


def _keep_triangles(room, triangles):
    if len(triangles):
        room[:len(triangles)].copy_(torch.as_tensor(triangles, device="cuda"))
    torch.cuda.current_stream().synchronize()
    return room


def run(state):
    case, h = state["case"], state["h"]
    do = case["do"]
    if do == "convert":
        return _keep([state["leaves"]], _convert(state["soup"], h, case["band"], case["signs"]))[0]
    if do == "batch":
        return _keep(state["leaves"], *bs.batch_mesh_to_volume(state["soups"], h, case["band"]))
    if do == "remesh":
        method = bs.MeshingMethod.MANIFOLD if case["method"] == "manifold" else bs.MeshingMethod.FEATURE_PRESERVING
        soup = bs.VoxelRemesher().with_voxel_size(h).with_meshing_method(method).remesh(state["soup"])
        state["triangles"][:soup.shape[0]].copy_(torch.from_numpy(soup))
        return state["triangles"]
    if do == "csg":
        # the operations consume their operands: a program that keeps them clones
        return _keep([state["leaves"]], getattr(state["volume"].clone(), case["op"])(state["other"].clone()))[0]
    if do == "offset":
        return _keep([state["leaves"]], state["volume"].clone().offset(case["voxels"] * h))[0]
    if do == "mesh":
        return _keep_triangles(state["triangles"], _mesher(case["method"], h).mesh_device(state["volume"]))
    part = _convert(state["soup"], h, 0)
    build = bs.VolumeBuilder(voxel_size=h)
    lattice = build.iwp((-26.0, -26.0, 0.0), (26.0, 26.0, 50.0), 0.5)
    inner = part.clone().offset(-5.0 * h)
    filling = inner.clone().intersect(lattice)
    clip = build.cuboid((-30.0, -30.0, -2.0), (30.0, -5.0, 50.0))
    result = part.subtract(inner).union(filling).subtract(clip)
    soup = _mesher("feature", h).mesh_device(result)
    return {"volume": _keep([state["leaves"]], result)[0], "soup": _keep_triangles(state["triangles"], soup)}


# ---------------------------------------------------------------- work
def _tris(case):
    return 2 * case["major"] * case["minor"] if case["mesh"] == "torus" else 20 * 4 ** case["level"]


def _area(mesh, span):
    """Surface area in voxel faces."""
    if mesh == "torus":
        return 4 * math.pi ** 2 * TORUS_R * TORUS_r * (span / (2 * (TORUS_R + TORUS_r))) ** 2
    return 4 * math.pi * (span / ISO_EXTENT) ** 2


def _leaves(area, band):
    """Leaves that a shell of `band` voxels on either side of that area meets."""
    return area * (2 * band + 17) / 512


def _ball_leaves(case):
    """Leaves of the sphere of radius 0.5 in a case's grid."""
    ext = 2 * (TORUS_R + TORUS_r) if case["mesh"] == "torus" else ISO_EXTENT
    return _leaves(math.pi * (case["span"] / ext) ** 2, 2)


def _convert_work(tris, area, band, per_voxel):
    # the pair set: every sub-triangle (sides below two voxels) against its box dilated by the band, 82
    # operations a pair; a per-voxel sign evaluates about 290 tree nodes and 10 triangles (16.3 k operations)
    flops = 82.0 * max(tris, 1.7 * area) * (2 * band + 2.9) ** 3
    if per_voxel:
        flops += 16.3e3 * area * (2 * band + 6.8)
    return {"bytes": 36.0 * tris + LEAF_BYTES * _leaves(area, band), "flops": flops}


def work(case):
    do = case["do"]
    if do == "batch":
        total = {"bytes": 0.0, "flops": 0.0}
        rng = random.Random(case["count"] * 1000003 + case["hi"])
        for i in range(case["count"]):
            tris = _log_uniform(rng, case["lo"], case["hi"])
            area = _area("torus" if i % 2 == 0 else "icosphere", case["span"])
            w = _convert_work(tris, area, case["band"], True)
            total = {k: total[k] + w[k] for k in total}
        return total
    tris, area = _tris(case), _area(case["mesh"], case["span"])
    leaves = _leaves(area, case.get("band", 3))
    if do == "convert":
        return _convert_work(tris, area, case["band"], case["signs"] == "voxel")
    if do == "remesh":
        w = _convert_work(tris, area, 0, True)
        return {"bytes": 36.0 * tris + 36.0 * 3.0 * area, "flops": w["flops"]}
    if do == "csg":
        if case["with"] == "mesh":
            return {"bytes": LEAF_BYTES * 3.0 * leaves, "flops": 512.0 * leaves}
        ball = _ball_leaves(case)
        return {"bytes": LEAF_BYTES * 2.0 * (leaves + ball), "flops": 512.0 * ball}
    if do == "offset":
        # the band leaves are read, the extended ones written; one update of about 40 operations a voxel
        out = _leaves(area, 3 + abs(case["voxels"]) / 2)
        return {"bytes": LEAF_BYTES * (leaves + out), "flops": 40.0 * 512.0 * out}
    if do == "mesh":
        return {"bytes": LEAF_BYTES * leaves + 36.0 * 3.0 * area, "flops": 100.0 * 1.5 * area}
    w = _convert_work(tris, area, 0, True)
    return {"bytes": 36.0 * tris + 36.0 * 3.0 * area + LEAF_BYTES * 3.0 * _leaves(area, 2), "flops": w["flops"]}


# ---------------------------------------------------------------- exact
def _sub_triangles(tri, h):
    """The converter's f32 subdivision: a triangle with its longest side over two voxels becomes n * n smaller
    ones, n = floor(side / h), built row by row by adding the two side steps."""
    t = tri.reshape(-1, 3, 3)
    e = [t[:, 1] - t[:, 0], t[:, 2] - t[:, 0], t[:, 2] - t[:, 1]]
    side = torch.stack([(d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1]) + d[:, 2] * d[:, 2] for d in e], 1).amax(1).sqrt()
    n = torch.floor(side / h).to(torch.int64)
    out = [t[n < 2]]
    for ns in torch.unique(n[n >= 2]).tolist():
        p = t[n == ns]
        inv = torch.tensor(1.0, dtype=torch.float32, device=p.device) / ns
        s1, s2 = (p[:, 1] - p[:, 0]) * inv, (p[:, 2] - p[:, 1]) * inv
        a = p[:, 0]
        for i in range(ns):
            b = a + s1
            c = b + s2
            row = [torch.stack([a, b, c], 1)]
            prev, a_s, b_s, c_s = a, a + s2, b + s2, c + s2
            for _ in range(i):
                row += [torch.stack([prev, b_s, a_s], 1), torch.stack([a_s, b_s, c_s], 1)]
                prev, a_s, b_s, c_s = a_s, a_s + s2, b_s + s2, c_s + s2
            out += row
            a = b
    return torch.cat(out)


def _distance2(p, t):
    """Squared distance in float64 from points (n, 3) to triangles (n, 3, 3)."""
    a, b, c = t[:, 0], t[:, 1], t[:, 2]
    best = None
    for s, e in ((a, b), (b, c), (c, a)):
        d, q = e - s, p - s
        k = ((q * d).sum(1) / (d * d).sum(1).clamp_min(1e-300)).clamp(0, 1)
        r = (q - k[:, None] * d).square().sum(1)
        best = r if best is None else torch.minimum(best, r)
    nrm = torch.linalg.cross(b - a, c - a)
    side = torch.stack([(torch.linalg.cross(e - s, p - s) * nrm).sum(1) for s, e in ((a, b), (b, c), (c, a))], 1)
    n2 = nrm.square().sum(1)
    plane = ((p - a) * nrm).sum(1).square() / n2.clamp_min(1e-300)
    return torch.where((side >= 0).all(1) & (n2 > 0), plane, best)


def _winding(p, t):
    """Winding numbers in float64: the solid angles of all triangles, summed."""
    out = torch.zeros(p.shape[0], dtype=torch.float64, device=p.device)
    step = max(1, 40_000_000 // t.shape[0])
    for i in range(0, p.shape[0], step):
        q = p[i:i + step, None]
        a, b, c = (t[None, :, k] - q for k in range(3))
        la, lb, lc = a.norm(dim=2), b.norm(dim=2), c.norm(dim=2)
        num = (a * torch.linalg.cross(b, c)).sum(2)
        den = la * lb * lc + (a * b).sum(2) * lc + (b * c).sum(2) * la + (c * a).sum(2) * lb
        out[i:i + step] = (2.0 * torch.atan2(num, den)).sum(1) / (4 * math.pi)
    return out


def exact(case, seed):
    """A small conversion's values in 64 bits.  The other results follow from a volume that the library itself
    converted (or are soups of it), or take too long."""
    if case["do"] != "convert":
        return None
    tris, area, band = _tris(case), _area(case["mesh"], case["span"]), case["band"]
    if max(tris, 4 * area) * (2 * band + 4) ** 3 > 2e8 or area * (2 * band + 7) * tris > 1e10:
        return None
    state = prepare(case, seed)
    soup = state["soup"]
    h = torch.tensor(state["h"], dtype=torch.float32, device="cuda")
    sub = _sub_triangles(soup, h)
    inv = 1.0 / h
    lo = torch.floor(sub.amin(1) * inv).to(torch.int64) - band
    hi = torch.ceil(sub.amax(1) * inv).to(torch.int64) + band
    flat = (lo == hi).any(1)
    lo[flat] -= 1
    hi[flat] += 1
    # dense indices over whole leaves of the bounding box
    base = torch.div(lo.amin(0), 8, rounding_mode="floor") * 8
    dims = torch.div(hi.amax(0) - base, 8, rounding_mode="floor") * 8 + 8
    nx, ny, nz = dims.tolist()
    d2 = torch.full((nx * ny * nz,), math.inf, dtype=torch.float64, device="cuda")
    ext = hi - lo + 1
    count = ext.prod(1)
    ends = count.cumsum(0)
    h64, chunk, at = h.double(), 4_000_000, 0
    while at < sub.shape[0]:
        limit = (int(ends[at - 1]) if at else 0) + chunk
        nxt = max(at + 1, int(torch.searchsorted(ends, limit)))
        which = torch.repeat_interleave(torch.arange(at, nxt, device="cuda"), count[at:nxt])
        k = torch.arange(which.numel(), device="cuda") - (ends[which] - count[which] - (int(ends[at - 1]) if at else 0))
        ez, ey = ext[which, 2], ext[which, 1]
        v = lo[which] + torch.stack([k // (ey * ez), k // ez % ey, k % ez], 1)
        r = _distance2(v.double() * h64, sub[which].double())
        w = v - base
        d2.scatter_reduce_(0, (w[:, 0] * ny + w[:, 1]) * nz + w[:, 2], r, "amin")
        at = nxt
    active = torch.isfinite(d2)
    i = active.nonzero()[:, 0]
    vox = torch.stack([i // (ny * nz), i // nz % ny, i % nz], 1) + base
    wn = _winding(vox.double() * h64, soup.double())
    value = torch.zeros_like(d2)
    value[i] = torch.where(wn < 0.2, 1.0, -1.0) * d2[i].sqrt()

    def by_leaf(x):
        return x.reshape(nx // 8, 8, ny // 8, 8, nz // 8, 8).permute(0, 2, 4, 1, 3, 5).reshape(-1, 512)
    # leaves that a box meets, in the order of their origins
    met = by_leaf(active).any(1)
    values = by_leaf(value)[met]
    whole = torch.zeros(state["leaves"]["values"].shape, dtype=torch.float64, device="cuda")
    whole[:values.shape[0]] = values
    return {"origins": None, "masks": None, "values": whole}
