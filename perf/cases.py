"""The workloads this framework's speed is measured on.

Each case is one call (or one short chain of calls) of the public interface on
inputs a user's program would hold: device tensors for the ``*_device`` entry
points, numpy arrays for the host ones.  ``listed()`` spans the range from a
1,000-query call on a small mesh to 16.8M queries on a million triangles;
``draw()`` gives further cases of the same kinds and ranges.
"""
import math

import numpy as np
import torch

import fcpw_amd as fcpw
from fcpw_amd import synth
from fcpw_amd.batch import BatchedScenes
from fcpw_amd.torch_ops import closest_point_distance

INF = float("inf")

# Fields: kind = the entry point; mesh = torus | sphere (radial noise) | star
# (2D polygon); prims = about how many triangles or segments; n = queries;
# near = the share of queries within `radius` of the surface, the others being
# uniform in `box` times the mesh's bounding box; bound = the search radius
# (0 = unbounded); scale = size of the mesh (unit meshes, or a scan in
# millimetres).


def listed():
    return [
        # nearest points of a bulk batch on a large mesh, half of it near the
        # surface: signed-distance grids, point-cloud registration
        dict(name="closest_torus_1m_16m", kind="closest", mesh="torus", prims=1048576, n=16777216, near=0.5,
             radius=0.05, box=1.2, bound=0.0, normals=False, scale=1.0),
        # a few queries a call, as in an interactive tool or a physics step:
        # latency and launches count
        dict(name="closest_sphere_20k_1k", kind="closest", mesh="sphere", prims=20480, n=1000, near=0.5,
             radius=0.05, box=1.5, bound=0.0, normals=False, scale=1.0),
        # one registration step: a scan of ragged size, bounded search radius,
        # normals wanted
        dict(name="closest_torus_131k_100k", kind="closest", mesh="torus", prims=131072, n=100003, near=0.9,
             radius=0.05, box=1.2, bound=0.06, normals=True, scale=1.0),
        # a planar distance field around a fine outline
        dict(name="closest_star_262k_8m", kind="closest", mesh="star", prims=262144, n=8388608, near=0.0,
             radius=0.05, box=1.25, bound=0.0, normals=False, scale=1.0),
        # bulk ray casting, closest hit
        dict(name="rays_torus_1m_4m", kind="rays", mesh="torus", prims=1048576, n=4194304, occlusion=False,
             bound=0.0, box=1.0, scale=1.0),
        # a frame's shadow rays: any hit within a bounded distance
        dict(name="occlusion_torus_131k_65k", kind="rays", mesh="torus", prims=131072, n=65537, occlusion=True,
             bound=1.5, box=1.0, scale=1.0),
        # Monte Carlo sampling of the surface inside spheres
        dict(name="spheres_sphere_82k_1m", kind="spheres", mesh="sphere", prims=81920, n=1000003, near=0.5,
             radius=0.2, box=1.0, bound=0.1, scale=1.0),
        # silhouette distances for boundary-value solvers
        dict(name="silhouettes_torus_131k_262k", kind="silhouettes", mesh="torus", prims=131072, n=262144, near=0.5,
             radius=0.05, box=1.2, bound=0.0, scale=1.0),
        # a scene of placed copies of one object
        dict(name="instances_256_1m", kind="instances", mesh="sphere", prims=20480, n=1048576, count=256),
        # many meshes of uneven size served by one launch
        dict(name="batch_48_meshes", kind="batch", mesh="torus", count=48, prims=65536, n=131072, near=0.5,
             radius=0.05, box=1.2),
        # one step of fitting a mesh to points: new vertices, refit, distances,
        # gradients of points and vertices
        dict(name="adjoint_sphere_200k_4m", kind="adjoint", mesh="sphere", prims=200000, n=4194304, near=1.0,
             radius=0.1, box=1.0, scale=1.0),
        # the reference's own call on host arrays, lists filled and read back
        dict(name="host_sphere_20k_1m", kind="host", mesh="sphere", prims=20480, n=1048576, near=0.0,
             radius=0.05, box=1.5, bound=0.0, normals=False, scale=1.0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["closest", "closest", "closest", "rays", "spheres", "silhouettes", "instances", "batch",
                       "adjoint", "host"])
    near = rng.choice([0.0, 0.5, 0.9, 1.0])
    radius = rng.choice([0.02, 0.05, 0.1])
    scale = rng.choice([1.0, 1.0, 40.0])
    if kind == "closest":
        mesh = rng.choice(["torus", "torus", "sphere", "star"])
        return dict(kind=kind, mesh=mesh, prims=_log(rng, 1000, 262144 if mesh == "sphere" else 1048576),
                    n=_log(rng, 1000, 8000000), near=0.0 if mesh == "star" else near, radius=radius,
                    box=rng.choice([1.0, 1.2, 1.5]), bound=rng.choice([0.0, 0.0, 0.06]),
                    normals=rng.random() < 0.5, scale=scale)
    if kind == "rays":
        return dict(kind=kind, mesh=rng.choice(["torus", "sphere", "star"]), prims=_log(rng, 1000, 262144),
                    n=_log(rng, 1000, 8000000), occlusion=rng.random() < 0.5, bound=rng.choice([0.0, 1.5]),
                    box=rng.choice([1.0, 1.5]), scale=scale)
    if kind == "spheres":
        return dict(kind=kind, mesh=rng.choice(["torus", "sphere", "star"]), prims=_log(rng, 1000, 262144),
                    n=_log(rng, 1000, 8000000), near=0.0, radius=radius, box=1.0, bound=rng.choice([0.05, 0.1]),
                    scale=scale)
    if kind == "silhouettes":
        return dict(kind=kind, mesh=rng.choice(["torus", "star"]), prims=_log(rng, 1000, 131072),
                    n=_log(rng, 1000, 300000), near=0.0, radius=radius, box=1.2, bound=0.0, scale=1.0)
    if kind == "instances":
        return dict(kind=kind, mesh="sphere", prims=_log(rng, 1000, 40000), n=_log(rng, 1000, 1500000),
                    count=_log(rng, 2, 300))
    if kind == "batch":
        return dict(kind=kind, mesh="torus", count=_log(rng, 2, 64), prims=_log(rng, 4000, 100000),
                    n=_log(rng, 4000, 200000), near=0.5, radius=radius, box=1.2)
    if kind == "adjoint":
        return dict(kind=kind, mesh=rng.choice(["torus", "sphere", "star"]), prims=_log(rng, 1000, 200000),
                    n=_log(rng, 1000, 4000000), near=0.0, radius=radius, box=1.2, scale=1.0)
    return dict(kind=kind, mesh=rng.choice(["torus", "sphere", "star"]), prims=_log(rng, 1000, 131072),
                n=_log(rng, 1000, 2000000), near=0.0, radius=radius, box=1.5, bound=rng.choice([0.0, 0.06]),
                normals=rng.random() < 0.5, scale=scale)


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------
def _dim(case):
    return 2 if case["mesh"] == "star" else 3


def _mesh(kind, prims, seed, scale=1.0):
    """vertices (float32) and indices (int32) of about `prims` primitives"""
    rng = synth.Rng(1000003 * (seed + 1) + prims)
    if kind == "torus":
        m = max(3, int(round(math.sqrt(prims / 4.0))))
        v, f = synth.torus_mesh(2 * m, m, jitter=0.25 / m, stream_seed=1000003 * (seed + 1) + prims)
    elif kind == "sphere":
        v, f = synth.geodesic_sphere(max(1, int(round(math.sqrt(prims / 20.0)))))
        v = synth.radial_noise(v, 0.01, rng)
    else:
        v, f = synth.star_polygon(max(3, prims), rng)
    return synth.f32(v * scale), f.astype(np.int32)


def _scene(V, F, silhouettes=False, transforms=None):
    dim = V.shape[1]
    s = fcpw.Scene3D() if dim == 3 else fcpw.Scene2D()
    s.set_object_count(1)
    s.set_object_vertices(V, 0)
    (s.set_object_triangles if dim == 3 else s.set_object_line_segments)(F, 0)
    if transforms is not None:
        s.set_object_instance_transforms(transforms, 0)
    if silhouettes:
        s.compute_silhouettes()
    s.build(fcpw.AggregateType.Bvh_SurfaceArea, False)
    g = fcpw.GPUScene3D("") if dim == 3 else fcpw.GPUScene2D("")
    g.transfer_to_gpu(s)
    return s, g


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(1000 + seed)
    return g


def _points(case, V, F, n, gen):
    """(n, dim) query points on the device: uniform ones first, then the near ones"""
    dim = V.shape[1]
    near = int(n * case.get("near", 0.0))
    lo, hi = torch.from_numpy(V.min(0)).cuda(), torch.from_numpy(V.max(0)).cuda()
    u = torch.rand((n - near, dim), generator=gen, device="cuda") * 2.0 - 1.0
    q = 0.5 * (lo + hi) + u * (0.5 * case.get("box", 1.0)) * (hi - lo)
    if near == 0:
        return q.contiguous()
    Vd, Fd = torch.from_numpy(V).cuda(), torch.from_numpy(F).cuda().long()
    t = Fd[torch.randint(0, len(F), (near,), generator=gen, device="cuda")]
    w = torch.rand((near, dim), generator=gen, device="cuda") + 1e-6
    w = w / w.sum(1, keepdim=True)
    p = sum(w[:, k:k + 1] * Vd[t[:, k]] for k in range(dim))
    d = torch.randn((near, dim), generator=gen, device="cuda")
    d = d / d.norm(dim=1, keepdim=True).clamp_min(1e-12)
    r = torch.rand((near, 1), generator=gen, device="cuda") * case["radius"] * case.get("scale", 1.0)
    return torch.cat([q, p + r * d]).contiguous()


def _spheres(q, bound):
    s = torch.zeros((len(q), 4), dtype=torch.float32, device=q.device)
    s[:, :q.shape[1]] = q
    s[:, 3] = bound * bound if bound > 0.0 else INF
    return s


def _transforms(count, seed):
    """rotations, uniform scales in [0.3, 1] and centres in a cube that keeps
    the density of 256 copies in [-8, 8]^3"""
    rng = synth.Rng(7000 + seed)
    half = 8.0 * (count / 256.0) ** (1.0 / 3.0)
    out = []
    for _ in range(count):
        ax, a = rng.sphere(1, 3)[0], rng.uniform(1, 0.0, 2.0 * np.pi)[0]
        K = np.array([[0, -ax[2], ax[1]], [ax[2], 0, -ax[0]], [-ax[1], ax[0], 0]])
        M = np.eye(4)
        M[:3, :3] = rng.uniform(1, 0.3, 1.0)[0] * (np.eye(3) + np.sin(a) * K + (1.0 - np.cos(a)) * K @ K)
        M[:3, 3] = rng.uniform(3, -half, half)
        out.append(M)
    return np.asarray(out, np.float32), half + 1.0


def _batch_sizes(case):
    """(primitives, queries) per mesh, log-uniform over a factor of 64 below the case's largest"""
    rng = synth.Rng(9000 + case["count"])
    lo = math.log(1.0 / 64.0)
    a = np.exp(rng.uniform(case["count"], lo, 0.0))
    b = np.exp(rng.uniform(case["count"], lo, 0.0))
    return [(max(64, int(case["prims"] * x)), max(16, int(case["n"] * y))) for x, y in zip(a, b)]


def prepare(case, seed):
    kind, st = case["kind"], {"case": case}
    gen = _gen(seed)
    if kind == "batch":
        scenes, keep, parts = [], [], []
        sizes = _batch_sizes(case)
        for k, (prims, n) in enumerate(sizes):
            V, F = _mesh(case["mesh"], prims, 100 * seed + k)
            s, g = _scene(V, F)
            keep.append(s)
            scenes.append(g)
            parts.append(_points(case, V, F, n, gen))
        q = torch.cat(parts)
        b = BatchedScenes(scenes)
        b.set_queries([n for _, n in sizes])
        st.update(batch=b, keep=keep, spheres=_spheres(q, 0.0), out=torch.empty((len(q), 10), device="cuda"))
        return st
    if kind == "instances":
        V, F = _mesh(case["mesh"], case["prims"], seed)
        T, half = _transforms(case["count"], seed)
        st["scene"], st["gpu"] = _scene(V, F, transforms=T)
        q = (torch.rand((case["n"], 3), generator=gen, device="cuda") * 2.0 - 1.0) * half
        st.update(spheres=_spheres(q, 0.0), out=torch.empty((case["n"], 10), device="cuda"),
                  obj=torch.empty(case["n"], dtype=torch.int32, device="cuda"))
        return st
    dim, n, scale = _dim(case), case["n"], case["scale"]
    V, F = _mesh(case["mesh"], case["prims"], seed, scale)
    st["V"], st["F"] = V, F
    st["scene"], st["gpu"] = _scene(V, F, silhouettes=kind == "silhouettes")
    bound = case.get("bound", 0.0) * scale
    if kind == "rays":
        q = _points(case, V, F, n, gen)
        d = torch.randn((n, dim), generator=gen, device="cuda")
        d = d / d.norm(dim=1, keepdim=True).clamp_min(1e-12)
        rays = torch.zeros((n, 10), device="cuda")
        rays[:, :dim] = q
        rays[:, 3:3 + dim] = d
        rays[:, 6:9] = 1.0 / rays[:, 3:6]
        rays[:, 9] = bound if bound > 0.0 else INF
        st.update(rays=rays, out=torch.empty((n, 10), device="cuda"))
        return st
    q = _points(case, V, F, n, gen)
    if kind == "adjoint":
        moved = torch.from_numpy(V).cuda()
        moved = moved * (1.0 + 0.002 * torch.randn((len(V), 1), generator=gen, device="cuda"))
        st.update(x=q.requires_grad_(True), V=moved.requires_grad_(True),
                  gd=torch.randn(n, generator=gen, device="cuda") / n)
        return st
    if kind == "host":
        st.update(points=q.cpu().numpy(), r2=np.full(n, bound * bound if bound > 0.0 else INF, np.float32),
                  hits=fcpw.GPUInteractionList())
        return st
    st.update(spheres=_spheres(q, bound), out=torch.empty((n, 10), device="cuda"))
    if kind == "spheres":
        st["rnd"] = torch.rand((n, 3), generator=gen, device="cuda")
    elif kind == "silhouettes":
        st["flip"] = torch.zeros(n, dtype=torch.int32, device="cuda")
    return st


# --------------------------------------------------------------------------
# one pass
# --------------------------------------------------------------------------
def _record(out):
    """the fields of the GPUInteraction records, as views"""
    return {"p": out[:, 0:3], "n": out[:, 3:6], "uv": out[:, 6:8], "d": out[:, 8],
            "index": out.view(torch.int32)[:, 9]}


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "closest":
        st["gpu"].find_closest_points_device(st["spheres"], st["out"], record_normals=case["normals"])
    elif kind == "rays":
        st["gpu"].intersect_device(st["rays"], st["out"], check_for_occlusion=case["occlusion"])
    elif kind == "spheres":
        st["gpu"].intersect_spheres_device(st["spheres"], st["rnd"], st["out"])
    elif kind == "silhouettes":
        st["gpu"].find_closest_silhouette_points_device(st["spheres"], st["flip"], st["out"])
    elif kind == "instances":
        st["gpu"].find_closest_points_device(st["spheres"], st["out"], object_index=st["obj"])
        return dict(_record(st["out"]), object=st["obj"])
    elif kind == "batch":
        st["batch"].find_closest_points_device(st["spheres"], st["out"])
    elif kind == "adjoint":
        d, p, prim = closest_point_distance(st["gpu"], st["x"], st["V"])
        gx, gV = torch.autograd.grad(d, (st["x"], st["V"]), st["gd"])
        return {"d": d, "p": p, "index": prim, "gx": gx, "gV": gV}
    else:
        hits = st["hits"]
        st["gpu"].find_closest_points(st["points"], st["r2"], hits, case["normals"])
        return {"p": hits.get_positions(), "n": hits.get_normals(), "uv": hits.get_uvs(), "d": hits.get_distances(),
                "index": hits.get_indices()}
    return _record(st["out"])


# --------------------------------------------------------------------------
# what a pass cannot do without, and how far results may differ
# --------------------------------------------------------------------------
def work(case):
    """Bytes: queries, records and geometry once.  Operations: one root-to-leaf
    descent (two boxes a level) and four primitive tests a query."""
    kind, prims, n = case["kind"], case["prims"], case["n"]
    if kind == "batch":
        share = (1.0 - 1.0 / 64.0) / math.log(64.0)  # mean of the log-uniform sizes
        n, prims = int(case["count"] * n * share), int(case["count"] * prims * share)
        depth = math.log2(max(2.0, case["prims"] * share))
    else:
        depth = math.log2(max(2, prims)) + (math.log2(max(2, case["count"])) if kind == "instances" else 0.0)
    dim = _dim(case)
    per = {"rays": 40 + 40, "spheres": 16 + 12 + 40, "silhouettes": 16 + 4 + 40, "instances": 16 + 40 + 4,
           "adjoint": 4 * dim + 4 + 4 * dim + 4 + 4 + 4 * dim}.get(kind, 16 + 40)
    box, prim = (44.0, 60.0) if dim == 3 else (28.0, 20.0)
    if kind == "spheres":
        prim = 0.5 * prim
    return {"bytes": float(n) * per + float(prims) * (12.0 * dim / 2.0 + 4.0 * dim),
            "flops": float(n) * (box * max(1.0, depth - 2.0) + 4.0 * prim)}


def tolerance(case):
    """Queries promise the records of the reference traversal bit for bit, ties
    included; gradients of vertices are sums of atomics in any order."""
    if case["kind"] == "adjoint":
        return {"rel": 1e-5, "max": 1e-3, "differ": 0.0}
    return "exact"


# --------------------------------------------------------------------------
# the same in 64 bits, by brute force
# --------------------------------------------------------------------------
def _dot(a, b):
    return (a * b).sum(-1)


def _segment_d2(q, a, b):
    u = b - a
    t = (_dot(q - a, u) / _dot(u, u).clamp_min(1e-300)).clamp(0.0, 1.0)
    r = q - a - t[..., None] * u
    return _dot(r, r)


def _nearest64(q, V, F):
    """distances (float64) of the points to the mesh: the plane's foot where it
    falls inside the triangle, otherwise the nearest edge"""
    best = torch.full((len(q),), INF, dtype=torch.float64, device="cuda")
    chunk = max(1, min(len(F), (1 << 25) // max(1, min(len(q), 8192))))
    for i in range(0, len(q), 8192):
        x = q[i:i + 8192, None, :]
        for j in range(0, len(F), chunk):
            c = [V[F[j:j + chunk, k]][None] for k in range(F.shape[1])]
            d2 = _segment_d2(x, c[0], c[1])
            if F.shape[1] == 3:
                d2 = torch.minimum(d2, _segment_d2(x, c[1], c[2]))
                d2 = torch.minimum(d2, _segment_d2(x, c[2], c[0]))
                e0, e1 = c[1] - c[0], c[2] - c[0]
                m = torch.linalg.cross(e0, e1)
                mm = _dot(m, m).clamp_min(1e-300)
                w = x - c[0]
                s = _dot(torch.linalg.cross(w.expand(-1, c[0].shape[1], -1), e1.expand(w.shape[0], -1, -1)), m) / mm
                t = _dot(torch.linalg.cross(e0.expand(w.shape[0], -1, -1), w.expand(-1, c[0].shape[1], -1)), m) / mm
                inside = (s >= 0.0) & (t >= 0.0) & (s + t <= 1.0)
                h = _dot(w, m)
                d2 = torch.where(inside, torch.minimum(d2, h * h / mm), d2)
            best[i:i + 8192] = torch.minimum(best[i:i + 8192], d2.min(1).values)
    return best.sqrt()


def exact(case, seed):
    """Distances in 64 bits where the brute force takes seconds; points, uv and
    index are decided by ties and have no such value."""
    if case["kind"] not in ("closest", "host") or case["bound"] > 0.0 or float(case["n"]) * case["prims"] > 2.5e9:
        return None
    V, F = _mesh(case["mesh"], case["prims"], seed, case["scale"])
    q = _points(case, V, F, case["n"], _gen(seed)).double()
    d = _nearest64(q, torch.from_numpy(V).cuda().double(), torch.from_numpy(F).cuda().long())
    return {"p": None, "n": None, "uv": None, "d": d if case["kind"] == "closest" else d.cpu().numpy(), "index": None}
