"""The work that users of this ray-query engine have it do, as timed cases.

A case is a dict of plain values.  `kind` names the path: a single picking
query, whole frames made on the device, ray batches over one tree, many scenes
in one graph launch, a stream of served requests, and scenes that are loaded,
deformed or moved between traces.  `prepare` makes the inputs on the GPU from
the seed alone and builds what a program keeps (committed scenes, a batch, a
server); `run` is one pass through the public entry points and returns every
hit it computed.
"""
import math

import numpy as np
import torch

import heavyrt_amd as H
from heavyrt_amd import workloads as W

LAYOUTS = {"bvh2": H.LAYOUT_BVH2, "bvh4": H.LAYOUT_BVH4, "bvh4_fp16": H.LAYOUT_BVH4_FP16, "auto": H.LAYOUT_AUTO,
           "auto_fp16": H.LAYOUT_AUTO_FP16, "ploc": H.LAYOUT_PLOC, "ploc_fp16": H.LAYOUT_PLOC_FP16}
FAR = 100.0  # far plane of the ray batches: far outside every scene here
AO_RADIUS = 0.23
EXACT_PAIRS = 1.2e10  # ray-triangle pairs that 64-bit brute force does within seconds

_ctx = None


def context():
    """One context (device and stream) for the whole program, as an application keeps it."""
    global _ctx
    if _ctx is None:
        _ctx = H.Context(0)
    return _ctx


def listed():
    return [
        # a click in a viewport: one synchronous query, all latency
        {"name": "pick_one", "kind": "pick", "mesh": "sphere", "tris": 81920},
        # the eye-ray renderer's frame at its own size, on the default layout
        {"name": "eye_frame_512", "kind": "eye", "mesh": "sphere", "tris": 81920, "width": 512, "height": 512},
        # the ambient-occlusion renderer's frame at its own size: the headline workload
        {"name": "ao_frame_1024", "kind": "ao", "mesh": "hills_boxes", "tris": 1072576, "width": 1024, "height": 1024,
         "spp": 16},
        # offline sampling of a large unstructured scene, FP16 nodes of the clustered tree: the largest batch
        {"name": "scatter_4m", "kind": "nearest", "mesh": "soup", "tris": 4194304, "rays": 4194304,
         "pattern": "scatter", "layout": "ploc_fp16", "test": "mt", "full": False},
        # a path tracer's second bounce with full hit records on the default layout, an odd count
        {"name": "bounce_1m_full", "kind": "nearest", "mesh": "hills_boxes", "tris": 524288, "rays": 1000003,
         "pattern": "bounce", "layout": "bvh2", "test": "mt", "full": True},
        # shadow rays of the same renderer as one stored batch
        {"name": "shadow_2m", "kind": "any", "mesh": "hills_boxes", "tris": 1072576, "rays": 2097152,
         "pattern": "bounce", "layout": "auto_fp16", "test": "mt"},
        # the batched build + trace workload at its own size
        {"name": "batch_256", "kind": "batch", "scenes": 256, "tris_lo": 1000, "tris_hi": 200000, "rays_lo": 4096,
         "rays_hi": 262144, "tune": True},
        # many tiny worlds per simulation step: launch-bound
        {"name": "batch_small", "kind": "batch", "scenes": 37, "tris_lo": 12, "tris_hi": 3000, "rays_lo": 64,
         "rays_hi": 2048, "tune": False},
        # a burst of mixed requests against resident scenes, device buffers
        {"name": "serve_48", "kind": "serve", "scenes": 6, "tris_lo": 50000, "tris_hi": 500000, "requests": 48,
         "rays_lo": 1000, "rays_hi": 1000000},
        # a scene loaded from host arrays and looked at once (a level load, a remeshed simulation)
        {"name": "load_1m", "kind": "load", "mesh": "hills_boxes", "tris": 1072576, "width": 640, "height": 360,
         "layout": "auto_fp16"},
        # a deforming closed mesh: refit, commit, trace, watertight FP32 nodes
        {"name": "deform_300k", "kind": "deform", "mesh": "sphere", "tris": 300000, "width": 512, "height": 512,
         "layout": "bvh4", "test": "wt"},
        # rigid bodies that move each frame: update instances, commit, trace with full records
        {"name": "bodies_2000", "kind": "bodies", "tris": 131072, "bodies": 2000, "moved": 500, "width": 800,
         "height": 600},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["pick", "eye", "ao", "nearest", "nearest", "any", "batch", "serve", "load", "deform", "bodies"])
    mesh = rng.choice(["soup", "hills", "hills_boxes", "sphere"])
    if kind == "pick":
        return {"kind": kind, "mesh": mesh, "tris": _log_int(rng, 12, 1000000)}
    if kind == "eye":
        return {"kind": kind, "mesh": mesh, "tris": _log_int(rng, 1000, 1000000),
                "width": 8 * _log_int(rng, 8, 160), "height": 8 * _log_int(rng, 8, 135)}
    if kind == "ao":
        return {"kind": kind, "mesh": rng.choice(["hills", "hills_boxes"]), "tris": _log_int(rng, 20000, 1072576),
                "width": 8 * _log_int(rng, 16, 128), "height": 8 * _log_int(rng, 16, 128),
                "spp": rng.choice([1, 3, 4, 8, 16])}
    if kind in ("nearest", "any"):
        c = {"kind": kind, "mesh": mesh, "tris": _log_int(rng, 1000, 1000000), "rays": _log_int(rng, 1000, 1000000),
             "pattern": rng.choice(["scatter", "bounce", "camera"]), "layout": rng.choice(sorted(LAYOUTS)),
             "test": rng.choice(["mt", "mt", "mt", "wt"])}
        return dict(c, full=rng.random() < 0.4) if kind == "nearest" else c
    if kind == "batch":
        t, r = _log_int(rng, 12, 2000), _log_int(rng, 64, 8192)
        return {"kind": kind, "scenes": _log_int(rng, 2, 200), "tris_lo": t, "tris_hi": t * _log_int(rng, 2, 40),
                "rays_lo": r, "rays_hi": r * _log_int(rng, 2, 16), "tune": rng.random() < 0.5}
    if kind == "serve":
        return {"kind": kind, "scenes": rng.randint(1, 6), "tris_lo": 20000, "tris_hi": _log_int(rng, 40000, 500000),
                "requests": rng.randint(4, 48), "rays_lo": 1000, "rays_hi": _log_int(rng, 10000, 1000000)}
    if kind == "load":
        return {"kind": kind, "mesh": mesh, "tris": _log_int(rng, 500, 1072576), "width": 320, "height": 8 * rng.randint(8, 45),
                "layout": rng.choice(sorted(LAYOUTS))}
    if kind == "deform":
        return {"kind": kind, "mesh": rng.choice(["sphere", "hills"]), "tris": _log_int(rng, 1000, 500000), "width": 320,
                "height": 8 * rng.randint(8, 45), "layout": rng.choice(sorted(LAYOUTS)), "test": rng.choice(["mt", "wt"])}
    n = _log_int(rng, 2, 3000)
    return {"kind": kind, "tris": _log_int(rng, 2000, 300000), "bodies": n, "moved": rng.randint(1, n), "width": 320,
            "height": 8 * rng.randint(8, 90)}


# ---------------------------------------------------------------------------
# meshes (float64 on the GPU, made from the generator alone)
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) & 0x7FFFFFFFFFFFFFFF)
    return g


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device="cuda", dtype=torch.float64)


def _unit(g, n):
    z = 1.0 - 2.0 * _rand(g, n)
    phi = 2.0 * math.pi * _rand(g, n)
    r = torch.sqrt(torch.clamp(1.0 - z * z, min=0.0))
    return torch.stack([r * torch.cos(phi), r * torch.sin(phi), z], 1)


def _soup(g, n):
    """Random triangles in the unit cube, edge scale LogNormal(-4, 0.5)."""
    c = _rand(g, n, 1, 3)
    e = torch.exp(-4.0 + 0.5 * torch.randn(n, 1, 1, generator=g, device="cuda", dtype=torch.float64))
    v = (c + e * _unit(g, 3 * n).reshape(n, 3, 3)).reshape(-1, 3)
    return v, torch.arange(3 * n, device="cuda").reshape(-1, 3)


def _grid_faces(nx, nz):
    i, j = torch.meshgrid(torch.arange(nx, device="cuda"), torch.arange(nz, device="cuda"), indexing="ij")
    a = (i * (nz + 1) + j).reshape(-1)
    b = a + nz + 1
    return torch.stack([a, a + 1, b, b, a + 1, b + 1], 1).reshape(-1, 3)


def _hills(g, n):
    """A heightfield of about n triangles over [0, 2] x [0, 1], height up to 0.2."""
    nz = max(2, round(math.sqrt(n / 4.0)))
    nx = max(2, round(n / (2.0 * nz)))
    y = torch.zeros(nx + 1, nz + 1, device="cuda", dtype=torch.float64)
    for freq in (4, 8, 16, 32):
        lat = _rand(g, 1, 1, 2 * freq + 1, freq + 1)
        y += (4.0 / freq) * torch.nn.functional.interpolate(lat, size=(nx + 1, nz + 1), mode="bicubic",
                                                            align_corners=True)[0, 0]
    x = torch.linspace(0.0, 2.0, nx + 1, device="cuda", dtype=torch.float64)[:, None].expand_as(y)
    z = torch.linspace(0.0, 1.0, nz + 1, device="cuda", dtype=torch.float64)[None, :].expand_as(y)
    return torch.stack([x, 0.2 * y / 1.875, z], -1).reshape(-1, 3), _grid_faces(nx, nz)


def _rotations(g, n):
    u = _rand(g, 3, n)
    a, b = torch.sqrt(1 - u[0]), torch.sqrt(u[0])
    x, y = a * torch.sin(2 * math.pi * u[1]), a * torch.cos(2 * math.pi * u[1])
    z, w = b * torch.sin(2 * math.pi * u[2]), b * torch.cos(2 * math.pi * u[2])
    return torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w),
                        2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w),
                        2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)], 1).reshape(n, 3, 3)


def _body_frames(g, n):
    """(n, 3, 4) affine frames of boxes of edge 0.01 to 0.05 scattered over the hills."""
    m = torch.empty(n, 3, 4, device="cuda", dtype=torch.float64)
    m[:, :, :3] = _rotations(g, n) * (0.01 + 0.04 * _rand(g, n, 1, 1))
    m[:, :, 3] = _rand(g, n, 3) * torch.tensor([2.0, 0.25, 1.0], device="cuda", dtype=torch.float64)
    return m


def _cube():
    v, f = W.unit_cube()
    return torch.from_numpy(v.astype(np.float64)).cuda(), torch.from_numpy(f.astype(np.int64)).cuda()


def _hills_boxes(g, n):
    """Hills with one rotated box per 512 triangles (2,000 on the million-triangle scene)."""
    k = n // 536
    v, f = _hills(g, n - 12 * k)
    cv, cf = _cube()
    m = _body_frames(g, k)
    bv = torch.einsum("bij,kj->bki", m[:, :, :3], cv) + m[:, None, :, 3]
    bf = cf[None] + 8 * torch.arange(k, device="cuda")[:, None, None]
    return torch.cat([v, bv.reshape(-1, 3)]), torch.cat([f, v.shape[0] + bf.reshape(-1, 3)])


def _sphere(g, n):
    """A closed, bumpy sphere of about n triangles around (0, 1, 0) (a projected cube), and a ground quad."""
    m = max(1, round(math.sqrt(n / 12.0)))
    t = torch.tan(torch.linspace(-math.pi / 4, math.pi / 4, m + 1, device="cuda", dtype=torch.float64))
    a, b = [x.reshape(-1) for x in torch.meshgrid(t, t, indexing="ij")]
    one, grid = torch.ones_like(a), _grid_faces(m, m)
    sides = [(one, a, b), (-one, b, a), (b, one, a), (a, -one, b), (a, b, one), (b, a, -one)]
    p = torch.nn.functional.normalize(torch.cat([torch.stack(s, 1) for s in sides]), dim=1)
    k = 6.28 * _rand(g, 3)
    v = p * (1.0 + 0.1 * torch.sin(4.0 * p + k).prod(1, keepdim=True))
    quad = torch.tensor([[-2, -1.2, -2], [2, -1.2, -2], [2, -1.2, 2], [-2, -1.2, 2]], device="cuda", dtype=torch.float64)
    v = torch.cat([v, quad])
    v[:, 1] += 1.0
    f = torch.cat([grid + s * (m + 1) ** 2 for s in range(6)])
    q = 6 * (m + 1) ** 2
    return v, torch.cat([f, torch.tensor([[q, q + 2, q + 1], [q, q + 3, q + 2]], device="cuda")])


def _mesh(name, g, n):
    return {"soup": _soup, "hills": _hills, "hills_boxes": _hills_boxes, "sphere": _sphere}[name](g, n)


def _host(v, f=None):
    """The float32 / uint32 host arrays a program hands to the engine."""
    vh = v.to(torch.float32).cpu().numpy()
    return vh if f is None else (vh, f.to(torch.int32).cpu().numpy().view(np.uint32))


# ---------------------------------------------------------------------------
# rays ((n, 8) float32 on the GPU)
# ---------------------------------------------------------------------------
def _pack(o, d, tfar):
    r = torch.zeros(d.shape[0], 8, device="cuda", dtype=torch.float32)
    r[:, 0:3] = o
    r[:, 4:7] = d
    r[:, 7] = tfar
    return r


def _view(g, v):
    """Eye point and target of a camera that looks at the mesh from outside, moved a little by the seed."""
    lo, hi = v.min(0).values, v.max(0).values
    c, ext = 0.5 * (lo + hi), float((hi - lo).max())
    j = _rand(g, 3) - 0.5
    eye = c + torch.tensor([0.2, 0.5, 1.0], device="cuda", dtype=torch.float64) * ext + 0.15 * ext * j
    return eye, c


def _camera_rays(g, v, width, height):
    eye, c = _view(g, v)
    fwd = torch.nn.functional.normalize(c - eye, dim=0)
    right = torch.nn.functional.normalize(torch.linalg.cross(fwd, torch.tensor([0.0, 1.0, 0.0], device="cuda", dtype=torch.float64)), dim=0)
    up = torch.linalg.cross(right, fwd)
    th = math.tan(math.radians(22.5))
    k = torch.arange(width * height, device="cuda")
    sx = (2.0 * ((k % width) + 0.5) / width - 1.0) * th * width / height
    sy = (1.0 - 2.0 * (torch.div(k, width, rounding_mode="floor") + 0.5) / height) * th
    d = torch.nn.functional.normalize(fwd[None] + sx[:, None] * right[None] + sy[:, None] * up[None], dim=1)
    return _pack(eye[None].expand_as(d), d, FAR)


def _bounce_rays(g, v, f, n, tfar):
    """From points on the surface, cosine-weighted about the upper side of the normal; neighbours stay neighbours, as pixels do."""
    t = torch.sort((_rand(g, n) * f.shape[0]).long()).values
    a, b, c = v[f[t, 0]], v[f[t, 1]], v[f[t, 2]]
    w = _rand(g, 2, n)
    s = torch.sqrt(w[0])
    p = (1 - s)[:, None] * a + (s * (1 - w[1]))[:, None] * b + (s * w[1])[:, None] * c
    m = torch.linalg.cross(b - a, c - a)
    m = m / torch.clamp(m.norm(dim=1, keepdim=True), min=1e-30)
    m = torch.where(m[:, 1:2] < 0, -m, m)
    d = torch.nn.functional.normalize(m + 0.999 * _unit(g, n), dim=1)
    return _pack(p + 1e-4 * m, d, tfar)


def _rays(pattern, g, v, f, n, tfar=FAR):
    if pattern == "camera":
        w = max(1, round(math.sqrt(n * 4.0 / 3.0)))
        return _camera_rays(g, v, w, -(-n // w))[:n].contiguous()
    if pattern == "bounce":
        return _bounce_rays(g, v, f, n, tfar)
    lo, hi = v.min(0).values, v.max(0).values
    return _pack(lo + (hi - lo) * _rand(g, n, 3), _unit(g, n), tfar)


def _camera_matrices(g, v, width, height):
    eye, c = _view(g, v)
    return W.eye_camera(width, height, eye=tuple(eye.tolist()), target=tuple(c.tolist()))


# ---------------------------------------------------------------------------
# what a program holds
# ---------------------------------------------------------------------------
def _committed(v, f, layout, test="mt"):
    s = H.Scene(context())
    s.add_instance(s.add_triangles(*_host(v, f)))
    s.set_triangle_test(H.TRI_WATERTIGHT if test == "wt" else H.TRI_MT)
    s.commit(layout=LAYOUTS[layout])
    return s


class _DeviceArray:
    """A device buffer the engine owns, for torch.as_tensor."""

    def __init__(self, ptr, shape, typestr):
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": typestr, "version": 2}


def _spread(lo, hi, n):
    """n sizes over the logarithm of [lo, hi], the same for every seed, in no particular order."""
    k = max(1, int(0.618 * n))
    while math.gcd(k, n) != 1:
        k += 1
    return [max(1, int(round(lo * (hi / lo) ** ((i * k % n + 0.5) / n)))) for i in range(n)]


def _compact(n):
    return torch.zeros(n, 2, device="cuda", dtype=torch.int32)


def _hits(buf):
    """Compact records as distances and triangle ids, full ones as distances, ids and barycentrics."""
    if buf.shape[1] == 2:
        return {"t": buf[:, 0].view(torch.float32), "prim": buf[:, 1]}
    return {"t": buf[:, 0].view(torch.float32), "ids": buf[:, 1:4], "uv": buf[:, 4:6].view(torch.float32)}


def prepare(case, seed):
    c, g = case, _gen(seed)
    ctx = context()
    kind = c["kind"]
    st = {"kind": kind}
    if kind == "batch":
        nt = _spread(c["tris_lo"], c["tris_hi"], c["scenes"])
        nr = _spread(c["rays_hi"], c["rays_lo"], c["scenes"])
        b = H.Batch(ctx, [3 * n for n in nt], nt, nr)
        verts = torch.as_tensor(_DeviceArray(b.d_verts, (3 * sum(nt), 4), "<f4"), device="cuda")
        idx = torch.as_tensor(_DeviceArray(b.d_idx, (sum(nt), 3), "<i4"), device="cuda")
        rays = torch.as_tensor(_DeviceArray(b.d_rays, (sum(nr), 8), "<f4"), device="cuda")
        verts[:, :3] = _soup(g, sum(nt))[0]
        verts[:, 3] = 1.0
        rays[:] = _pack(_rand(g, sum(nr), 3), _unit(g, sum(nr)), FAR)
        at = 0
        for n in nt:
            idx[at:at + n] = torch.arange(3 * n, device="cuda", dtype=torch.int32).reshape(-1, 3)
            at += n
        torch.cuda.synchronize()
        if c["tune"]:
            b.autotune(1)
        hits = torch.as_tensor(_DeviceArray(b.d_hits, (sum(nr), 2), "<i4"), device="cuda")
        out = _hits(hits)
        for x in out.values():
            x.owner = b  # the hits are the batch's own memory: whoever holds them holds the batch
        return dict(st, batch=b, out=out)
    if kind == "serve":
        sv = H.Server(ctx, 1 << 30, 3)
        scenes, pools = [], []
        for k, n in enumerate(_spread(c["tris_lo"], c["tris_hi"], c["scenes"])):
            v, f = _mesh("soup" if k % 2 == 0 else "hills", g, n)
            s = _committed(v, f, "auto_fp16")
            scenes.append((sv.add_scene(s), s))
            pools.append((v, f))
        sizes = _spread(c["rays_lo"], c["rays_hi"], c["requests"])
        near = torch.zeros(sum(sizes[0::2]), 2, device="cuda", dtype=torch.int32)
        occ = torch.zeros(sum(sizes[1::2]), device="cuda", dtype=torch.uint8)
        reqs, at = [], [0, 0]
        for i, n in enumerate(sizes):
            any_hit, (v, f) = i % 2, pools[(i // 2) % len(pools)]
            r = _rays("bounce" if any_hit else "camera", g, v, f, n, AO_RADIUS)
            reqs.append((scenes[(i // 2) % len(pools)][0], r, (occ if any_hit else near)[at[any_hit]:at[any_hit] + n], bool(any_hit)))
            at[any_hit] += n
        torch.cuda.synchronize()
        return dict(st, server=sv, reqs=reqs, out={"near": _hits(near), "any": occ}, hold=scenes)
    if kind == "bodies":
        v, f = _hills(g, c["tris"])
        cv, cf = _cube()
        s = H.Scene(ctx)
        ground, box = s.add_triangles(*_host(v, f)), s.add_triangles(*_host(cv, cf))
        s.add_instance(ground)

        def columns(m):  # (n, 3, 4) -> 16 column-major floats each
            full = torch.zeros(m.shape[0], 4, 4, device="cuda", dtype=torch.float64)
            full[:, :3] = m
            full[:, 3, 3] = 1.0
            return full.transpose(1, 2).reshape(-1, 16).to(torch.float32).cpu().numpy()

        for m in columns(_body_frames(g, c["bodies"])):
            s.add_instance(box, m)
        moved = [(1 + i, m) for i, m in enumerate(columns(_body_frames(g, c["moved"])))]
        s.commit()
        rays = _camera_rays(g, v, c["width"], c["height"])
        hits = torch.zeros(rays.shape[0], 8, device="cuda", dtype=torch.int32)
        torch.cuda.synchronize()
        return dict(st, scene=s, moved=moved, rays=rays, hits=hits, out=_hits(hits))
    v, f = _mesh(c["mesh"], g, c["tris"])
    if kind == "load":
        rays = _camera_rays(g, v, c["width"], c["height"])
        hits = _compact(rays.shape[0])
        torch.cuda.synchronize()
        return dict(st, scene=H.Scene(ctx), mesh=_host(v, f), layout=LAYOUTS[c["layout"]], rays=rays, hits=hits, out=_hits(hits))
    if kind == "deform":
        s = _committed(v, f, c["layout"], c["test"])
        k = _rand(g, 4)
        moved = v + 0.05 * torch.sin(5.0 * v[:, [1, 2, 0]] + 6.28 * k[:3])
        rays = _camera_rays(g, v, c["width"], c["height"])
        hits = _compact(rays.shape[0])
        torch.cuda.synchronize()
        return dict(st, scene=s, verts=_host(moved), layout=LAYOUTS[c["layout"]], rays=rays, hits=hits, out=_hits(hits))
    if kind == "pick":
        r = _rays("camera", g, v, f, 1)[0].cpu().numpy()
        return dict(st, scene=_committed(v, f, "bvh2"), ray=(r[:4].copy(), r[4:].copy()))
    if kind in ("eye", "ao"):
        cam = _camera_matrices(g, v, c["width"], c["height"])
        image = torch.zeros(c["height"], c["width"], device="cuda", dtype=torch.int32)
        torch.cuda.synchronize()
        s = _committed(v, f, "bvh2" if kind == "eye" else "auto_fp16")
        return dict(st, scene=s, cam=cam, size=(c["width"], c["height"]), spp=c.get("spp", 0), image=image, seed=seed)
    rays = _rays(c["pattern"], g, v, f, c["rays"], AO_RADIUS if kind == "any" else FAR)
    s = _committed(v, f, c["layout"], c["test"])
    if kind == "any":
        out = torch.zeros(c["rays"], device="cuda", dtype=torch.uint8)
        torch.cuda.synchronize()
        return dict(st, scene=s, rays=rays, hits=out)
    hits = torch.zeros(c["rays"], 8, device="cuda", dtype=torch.int32) if c["full"] else _compact(c["rays"])
    torch.cuda.synchronize()
    return dict(st, scene=s, rays=rays, hits=hits, fmt=H.HIT_FULL if c["full"] else H.HIT_COMPACT, out=_hits(hits))


def run(st):
    kind = st["kind"]
    if kind == "pick":
        t, prim, inst, geom, u, v = st["scene"].query_nearest_one(*st["ray"])
        return {"t": t, "ids": [prim, inst, geom], "uv": [u, v]}
    if kind == "eye":
        st["scene"].eye_render(*st["cam"], *st["size"], W.EYE_PALETTE, st["image"])
        return st["image"]
    if kind == "ao":
        st["scene"].rtao_render(*st["cam"], *st["size"], st["spp"], AO_RADIUS, st["seed"], st["image"])
        return st["image"]
    if kind == "nearest":
        st["scene"].trace_nearest(st["rays"], st["rays"].shape[0], st["hits"], st["fmt"])
        return st["out"]
    if kind == "any":
        st["scene"].trace_any(st["rays"], st["rays"].shape[0], st["hits"])
        return st["hits"]
    if kind == "batch":
        st["batch"].run()
        return st["out"]
    if kind == "serve":
        sv = st["server"]
        ids = [sv.submit(*r) for r in st["reqs"]]
        for i in ids:
            sv.wait(i)
        return st["out"]
    s = st["scene"]
    if kind == "load":
        s.clear_geom()
        s.add_instance(s.add_triangles(*st["mesh"]))
        s.commit(layout=st["layout"])
    elif kind == "deform":
        s.update_triangles(0, st["verts"])
        s.commit(layout=st["layout"])
    else:
        for i, m in st["moved"]:
            s.update_instance(i, m)
        s.commit()
    s.trace_nearest(st["rays"], st["rays"].shape[0], st["hits"], H.HIT_FULL if kind == "bodies" else H.HIT_COMPACT)
    return st["out"]


def work(case):
    """Rays and geometry read once, answers written once; per ray one descent of a binary tree (two box tests of
    18 operations a level) and one triangle test of 40; per built triangle its record and node written once."""
    c, kind = case, case["kind"]

    def trace(rays, tris, out, ray_bytes=32):
        touched = min(tris, rays * max(1.0, math.log2(tris + 1)))  # a small batch does not reach every node
        return (ray_bytes + out) * rays + 112.0 * touched, rays * (36.0 * math.log2(tris + 1) + 40.0)

    if kind == "pick":
        b, fl = trace(1, c["tris"], 32)
    elif kind == "eye":
        b, fl = trace(c["width"] * c["height"], c["tris"], 4, 0)
    elif kind == "ao":
        n = c["width"] * c["height"]
        b, fl = trace(n, c["tris"], 4, 0)
        fl += trace(n * c["spp"], c["tris"], 0, 0)[1]
    elif kind in ("nearest", "any"):
        b, fl = trace(c["rays"], c["tris"], 1 if kind == "any" else 32 if c["full"] else 8)
    elif kind in ("batch", "serve"):
        n, serve = c["scenes"], kind == "serve"
        t = sum(_spread(c["tris_lo"], c["tris_hi"], n))
        r = sum(_spread(c["rays_lo"], c["rays_hi"], c["requests"] if serve else n))
        b, fl = trace(r, t / n, 5 if serve else 8)
        b += 0 if serve else (48.0 + 12.0 + 112.0) * t
    else:
        n = c["width"] * c["height"]
        b, fl = trace(n, c["tris"], 32 if kind == "bodies" else 8)
        if kind == "bodies":
            b += (64.0 + 80.0 + 64.0) * c["bodies"]  # a matrix in, an instance record and a node out
        else:
            b += ((12.0 if kind == "deform" else 24.0) + 112.0) * c["tris"]
    return {"bytes": float(b), "flops": float(fl)}


# ---------------------------------------------------------------------------
# the nearest hits in 64 bits, by brute force
# ---------------------------------------------------------------------------
def _brute(v, f, rays):
    """(t, u, v) of the nearest hit of each ray: every triangle against every ray, in float64; t = tFar on a miss."""
    p = v.to(torch.float32).double()
    a, e1, e2 = p[f[:, 0]], p[f[:, 1]] - p[f[:, 0]], p[f[:, 2]] - p[f[:, 0]]
    r = rays.double()
    t = r[:, 7].clone()
    uv = torch.zeros(r.shape[0], 2, device="cuda", dtype=torch.float64)
    rows = max(1, int(4e7 // a.shape[0]))
    for k in range(0, r.shape[0], rows):
        for m in range(0, a.shape[0], 1 << 22):
            A, E1, E2 = a[None, m:m + (1 << 22)], e1[None, m:m + (1 << 22)], e2[None, m:m + (1 << 22)]
            o, d = r[k:k + rows, None, 0:3], r[k:k + rows, None, 4:7]
            pv = torch.linalg.cross(d.expand(-1, A.shape[1], -1), E2.expand(d.shape[0], -1, -1))
            s = o - A
            q = torch.linalg.cross(s, E1.expand_as(s))
            inv = 1.0 / (E1 * pv).sum(-1)
            b1 = (s * pv).sum(-1) * inv
            b2 = (q * d).sum(-1) * inv
            tt = (E2 * q).sum(-1) * inv
            ok = (b1 >= -1e-6) & (b2 >= -1e-6) & (b1 + b2 <= 1.0 + 1e-6) & (tt > r[k:k + rows, None, 3])
            tt = torch.where(ok, tt, math.inf)
            best, at = tt.min(1)
            now = best < t[k:k + rows]
            t[k:k + rows] = torch.where(now, best, t[k:k + rows])
            bc = torch.stack([b2.gather(1, at[:, None])[:, 0], b1.gather(1, at[:, None])[:, 0]], 1)
            uv[k:k + rows] = torch.where(now[:, None], bc, uv[k:k + rows])
    return t, uv


def exact(case, seed):
    c, g, kind = case, _gen(seed), case["kind"]
    if kind not in ("pick", "nearest", "load", "deform"):
        return None  # images, occlusion bytes, and scenes too many for brute force
    rays_n = 1 if kind == "pick" else c["rays"] if kind == "nearest" else c["width"] * c["height"]
    if rays_n * c["tris"] > EXACT_PAIRS:
        return None
    v, f = _mesh(c["mesh"], g, c["tris"])
    if kind == "deform":
        k = _rand(g, 4)
        moved = v + 0.05 * torch.sin(5.0 * v[:, [1, 2, 0]] + 6.28 * k[:3])
        return {"t": _brute(moved, f, _camera_rays(g, v, c["width"], c["height"]))[0], "prim": None}
    if kind == "load":
        return {"t": _brute(v, f, _camera_rays(g, v, c["width"], c["height"]))[0], "prim": None}
    if kind == "pick":
        t, uv = _brute(v, f, _rays("camera", g, v, f, 1))
        return {"t": float(t[0]), "ids": [None, None, None], "uv": [float(uv[0, 0]), float(uv[0, 1])]}
    t, uv = _brute(v, f, _rays(c["pattern"], g, v, f, c["rays"]))
    return {"t": t, "ids": None, "uv": uv} if c["full"] else {"t": t, "prim": None}
