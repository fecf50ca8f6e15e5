"""The tight bounds (disks) of small subtrees leave every record as it was:
closest points bit for bit against the oracle's reference-order traversal where
a bound could go wrong -- thin plates in every tilt, slivers, subtrees at the
size limit of the disks, meshes away from the origin and at extreme scales,
queries far outside the scene, vertex updates with and without a refit, both
record orders, batches."""
import numpy as np
import pytest

import oracle
from fcpw_amd import synth
from tests import meshes
from tests.test_gpu_parity import as_records, assert_bit_equal, make_scene

pytestmark = pytest.mark.gpu
fcpw = pytest.importorskip("fcpw_amd")

DISK_MAX_PRIMS = 1024  # device.hpp


def plate(n_side, tilt, seed):
    """a flat square grid of triangles, tilted about two axes"""
    u = np.linspace(-1.0, 1.0, n_side + 1)
    X, Y = np.meshgrid(u, u, indexing="ij")
    v = np.stack([X, Y, np.zeros_like(X)], -1).reshape(-1, 3)
    a, b = tilt
    Rx = np.array([[1, 0, 0], [0, np.cos(a), -np.sin(a)], [0, np.sin(a), np.cos(a)]])
    Ry = np.array([[np.cos(b), 0, np.sin(b)], [0, 1, 0], [-np.sin(b), 0, np.cos(b)]])
    i, j = np.meshgrid(np.arange(n_side), np.arange(n_side), indexing="ij")
    k = (i * (n_side + 1) + j).ravel()
    f = np.concatenate([np.stack([k, k + n_side + 1, k + n_side + 2], -1), np.stack([k, k + n_side + 2, k + 1], -1)])
    return synth.f32(v @ (Rx @ Ry).T), f.astype(np.int32)


def slivers(seed):
    """a sphere whose triangles are squeezed to heights from 1e-1 to 1e-6 of their length"""
    v, f = synth.geodesic_sphere(12)
    t = v[f].reshape(-1, 3, 3).copy()
    rng = synth.Rng(seed)
    s = 10.0 ** rng.uniform(len(t), -6.0, -1.0)
    m = 0.5 * (t[:, 0] + t[:, 1])
    t[:, 2] = m + (t[:, 2] - m) * s[:, None]
    return synth.f32(t.reshape(-1, 3)), np.arange(3 * len(t), dtype=np.int32).reshape(-1, 3)


CASES = {
    "plate_axis": lambda: plate(40, (0.0, 0.0), 1),
    "plate_tilted": lambda: plate(40, (0.7, 0.4), 2),
    "plate_at_limit": lambda: plate(32, (0.3, 1.1), 3),          # 2048 triangles: subtrees of 1024
    "plate_past_limit": lambda: plate(33, (0.3, 1.1), 3),
    "sphere": lambda: meshes.small_icosphere(4),
    "smooth_sphere": lambda: tuple(a(x) for a, x in zip((synth.f32, lambda i: i.astype(np.int32)),
                                                        synth.geodesic_sphere(40))),
    "slivers": lambda: slivers(5),
    "degenerate": meshes.degenerate_soup,
    "soup": lambda: meshes.triangle_soup(2000),
    "one_record": lambda: meshes.triangle_soup(5, seed=3),
    "one_leaf": lambda: meshes.triangle_soup(3, seed=4),
    "star2d": lambda: meshes.small_star(5000),
    "walker2d": lambda: meshes.load_obj("walker.obj", 2),
}


def queries(V, n, seed):
    """inside the box, near vertices (from 1e-7 to 1e-1 of the box) and far outside it"""
    rng = synth.Rng(seed)
    lo, hi = V.min(0).astype(np.float64), V.max(0).astype(np.float64)
    dim, ext = V.shape[1], float((hi - lo).max())
    a = synth.uniform_in_box(n, lo, hi, 1.5, rng)
    v = V[rng.integers(n, len(V))].astype(np.float64)
    b = v + rng.sphere(n, dim) * (ext * 10.0 ** rng.uniform(n, -7.0, -1.0))[:, None]
    c = 0.5 * (lo + hi) + rng.sphere(n // 4, dim) * (ext * 10.0 ** rng.uniform(n // 4, 0.0, 5.0))[:, None]
    return synth.f32(np.concatenate([a, b, c]))


def check(g, V, F, q, r2=None, bvh=None):
    r2 = np.full(len(q), np.inf, np.float32) if r2 is None else r2
    hits = fcpw.GPUInteractionList()
    g.find_closest_points(q, r2, hits, record_normals=True)
    ref = (bvh or oracle.Bvh(V, F)).closest_points_gpuorder(q, r2, record_normal=True)
    assert_bit_equal(as_records(hits), ref)


@pytest.mark.parametrize("place", ["unit", "away", "large", "tiny", "huge"])
@pytest.mark.parametrize("name", sorted(CASES))
def test_records_equal_the_oracle(gpu, name, place):
    V, F = CASES[name]()
    with np.errstate(over="ignore"):
        V = {"unit": V, "away": V + np.float32(300.0), "large": V * np.float32(700.0),
             "tiny": V * np.float32(1e-12), "huge": V * np.float32(1e18)}[place].astype(np.float32)
    _, g = make_scene(V, F)
    q = queries(V, 6000, 11)
    check(g, V, F, q)
    ext = float((V.max(0) - V.min(0)).max())
    r2 = ((0.05 * ext * synth.Rng(12).uniform(len(q))) ** 2).astype(np.float32)
    check(g, V, F, q, r2)


@pytest.mark.parametrize("layout", [0, 1])
def test_updates_refits_and_layouts(gpu, layout):
    """after a vertex update without a refit the boxes are the old ones and the
    disks hold for nothing; the refit brings both back"""
    import torch
    V, F = meshes.small_torus(64, 32)
    scene, g = make_scene(V, F)
    g.set_option("layout", layout)
    q = queries(V, 6000, 21)
    check(g, V, F, q)
    b = oracle.Bvh(V, F)
    rng = synth.Rng(22)
    for k in range(3):
        V = (V + rng.uniform(V.size, -0.02, 0.02).reshape(V.shape)).astype(np.float32)
        st = torch.cuda.current_stream().cuda_stream
        dv = torch.from_numpy(V).cuda()
        g._update_positions_device(dv.data_ptr(), len(V), st)
        b.update_vertices(V)
        check(g, V, F, q, bvh=b)  # stale boxes, new triangles
        g._refit_device(st)
        b.refit()
        check(g, V, F, q, bvh=b)


def test_batch_members_use_their_own_disks(gpu):
    import torch
    from fcpw_amd.batch import BatchedScenes
    names = ["plate_tilted", "sphere", "one_leaf", "slivers"]
    data = [CASES[n]() for n in names]
    gs = [make_scene(V, F) for V, F in data]
    qs = [queries(V, 3000, 31 + k) for k, (V, _) in enumerate(data)]
    batch = BatchedScenes([g for _, g in gs])
    batch.set_queries([len(q) for q in qs])
    q = torch.from_numpy(np.concatenate(qs)).cuda()
    sph = torch.cat([q, torch.full((len(q), 1), float("inf"), device="cuda")], 1).contiguous()
    out = torch.empty((len(q), 10), device="cuda")
    batch.find_closest_points_device(sph, out)
    rec = out.cpu().numpy().view(fcpw.INTERACTION_DTYPE).reshape(-1)
    at = 0
    for (V, F), qk in zip(data, qs):
        ref = oracle.Bvh(V, F).closest_points_gpuorder(qk, np.full(len(qk), np.inf, np.float32))
        assert_bit_equal(rec[at:at + len(qk)], ref)
        at += len(qk)


def torn(V, k):
    """one half moved far away: the boxes it leaves behind shrink the reference's
    r^2 for queries near them, so that the other half is out of reach"""
    V2 = V.copy()
    V2[(V[:, 0] < 0.0) == (k == 0), -1] += np.float32(10.0)
    return V2


@pytest.mark.parametrize("mesh", ["torus", "star2d"])
def test_stale_boxes_stay_without_disks(gpu, mesh):
    """boxes that do not hold their primitives shrink the reference's r^2 too, so
    no subtree may be dropped: after a vertex update, also when the records are
    reordered before the refit, and for a tree uploaded with boxes from before one"""
    import torch
    V, F = meshes.small_torus(64, 32) if mesh == "torus" else meshes.small_star(5000)
    _, g = make_scene(V, F)
    q = queries(V, 6000, 41)
    b = oracle.Bvh(V, F)
    for k, layout in enumerate((1, 0)):
        V2 = torn(V, k)
        st = torch.cuda.current_stream().cuda_stream
        dv = torch.from_numpy(V2).cuda()
        g._update_positions_device(dv.data_ptr(), len(V2), st)
        torch.cuda.synchronize()
        b.update_vertices(V2)
        g.set_option("layout", layout)
        check(g, V2, F, q, bvh=b)
        g._refit_device(st)
        b.refit()
        check(g, V2, F, q, bvh=b)


def test_disks_off_where_few_slots_keep_one(gpu):
    """a soup's patches are no plates: the walk goes without disks, after a refit
    that makes a smooth surface of it with them, and back; the records stay"""
    import torch
    V, F = meshes.small_torus(64, 32)
    V = V[F].reshape(-1, 3).copy()  # triangles of their own
    F = np.arange(len(V), dtype=np.int32).reshape(-1, 3)
    soup = synth.f32(synth.Rng(71).uniform(V.size, -1.0, 1.0).reshape(V.shape))
    _, g = make_scene(soup, F)
    b = oracle.Bvh(soup, F)
    q = queries(V, 6000, 72)
    check(g, soup, F, q, bvh=b)
    st = torch.cuda.current_stream().cuda_stream
    for W in (V, soup, V):
        dv = torch.from_numpy(W).cuda()
        g._update_positions_device(dv.data_ptr(), len(W), st)
        g._refit_device(st)
        torch.cuda.synchronize()
        b.update_vertices(W)
        b.refit()
        check(g, W, F, q, bvh=b)


@pytest.mark.parametrize("n", [4, 5, 9, 17, 64, 65, 257, 1023, 1024, 1025, 1040])
@pytest.mark.parametrize("mesh", ["torus", "star2d"])
def test_trees_around_the_one_block_size(gpu, mesh, n):
    """trees of at most DISK_MAX_PRIMS primitives get their ranges, disks and
    refits from one block: uploaded, reordered and refitted, against the oracle"""
    import torch
    V, F = meshes.small_torus(65, 8) if mesh == "torus" else meshes.small_star(1040)
    F = np.ascontiguousarray(F[:n])
    assert len(F) == n
    _, g = make_scene(V, F)
    b = oracle.Bvh(V, F)
    q = queries(V[np.unique(F)], 3000, 81)
    check(g, V, F, q, bvh=b)
    for k in range(3):
        V = (V + synth.Rng(82 + k).uniform(V.size, -0.02, 0.02).reshape(V.shape)).astype(np.float32)
        st = torch.cuda.current_stream().cuda_stream
        dv = torch.from_numpy(V).cuda()
        g._update_positions_device(dv.data_ptr(), len(V), st)
        b.update_vertices(V)
        if k:
            g.set_option("layout", k % 2)
        check(g, V, F, q, bvh=b)
        g._refit_device(st)
        b.refit()
        check(g, V, F, q, bvh=b)
    # the boxes themselves: the counting variant expands what the reference does
    g.set_option("stats", 1)
    check(g, V, F, q, bvh=b)
    _, ni, npr, _ = b.closest_points_gpuorder(q, counters=True)
    assert (g.info("stat_internal_nodes"), g.info("stat_prim_tests")) == (int(ni.sum()), int(npr.sum()))
    g.set_option("stats", 0)
