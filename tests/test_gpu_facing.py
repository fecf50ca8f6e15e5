"""Facing entries of the silhouette queries: the cooperative kernel, which drops
subtrees and records by them, against the per-lane kernel, which does not know
them.  Bit for bit, where the bound could go wrong: queries close to faces,
edges and vertices and far outside, precisions from none to large, open meshes,
slivers, meshes away from the origin and scaled, both record orders, after a
refit."""
import numpy as np
import pytest

from fcpw_amd import synth
from tests import meshes
from tests.test_gpu_disks import CASES, queries
from tests.test_gpu_silhouettes import gpu_scene, records
from tests.test_oracle_silhouettes import product_scene

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
fcpw = pytest.importorskip("fcpw_amd")

MESHES = {
    "torus": lambda: meshes.small_torus(64, 32),
    "torus_past_limit": lambda: meshes.small_torus(96, 48),  # subtrees above 1,024 triangles
    "sphere": CASES["smooth_sphere"],
    "slivers": CASES["slivers"],
    "open_plate": CASES["plate_tilted"],
    "star2d": CASES["star2d"],
    "walker2d": CASES["walker2d"],
}


def both_kernels(g, q, r2, flip, prec, r2min=0.0):
    out = []
    for coop in (1, 0):
        g.set_option("coop", coop)
        hits = fcpw.GPUInteractionList()
        g.find_closest_silhouette_points(q, r2, flip, hits, r2min, prec)
        out.append(records(hits).copy())
    g.set_option("coop", 1)
    return out


@pytest.mark.parametrize("place", ["unit", "away", "large", "tiny"])
@pytest.mark.parametrize("name", sorted(MESHES))
def test_facing_entries_change_no_record(gpu, name, place):
    V, F = MESHES[name]()
    scale = {"unit": 1.0, "away": 1.0, "large": 300.0, "tiny": 1e-3}[place]
    V = (V * np.float32(scale) + np.float32(50.0 if place == "away" else 0.0)).astype(np.float32)
    s = product_scene(V, F)
    g = gpu_scene(s, V.shape[1])
    q = queries(V, 6000, 17)
    flip = (np.arange(len(q)) % 2).astype(np.int32)
    ext = float((V.max(0) - V.min(0)).max())
    inf = np.full(len(q), np.inf, np.float32)
    near = np.full(len(q), (0.2 * ext) ** 2, np.float32)
    for prec, r2, r2min in ((1e-3, inf, 0.0), (0.0, inf, 0.0), (0.2, inf, 0.0), (1e-3, near, 0.0),
                            (1e-3, inf, (0.05 * ext) ** 2)):
        a, b = both_kernels(g, q, r2, flip, prec, r2min)
        assert a.tobytes() == b.tobytes(), (prec, r2min, int((a != b).sum()))


@pytest.mark.parametrize("layout", [0, 1])
def test_facing_entries_follow_the_boxes(gpu, layout):
    """they are about the box centres: rebuilt with a refit, as are records in another order"""
    V, F = MESHES["torus"]()
    g = gpu_scene(product_scene(V, F), 3)
    q = queries(V, 6000, 23)
    flip, inf = np.zeros(len(q), np.int32), np.full(len(q), np.inf, np.float32)
    g.set_option("layout", layout)
    st = torch.cuda.current_stream().cuda_stream
    moved = (V + synth.Rng(5).uniform(V.size, -0.05, 0.05).reshape(V.shape)).astype(np.float32)
    for k in range(3):
        a, b = both_kernels(g, q, inf, flip, 1e-3)
        assert a.tobytes() == b.tobytes(), (layout, k)
        if k == 0:
            g._update_positions_device(torch.from_numpy(moved).cuda().data_ptr(), len(moved), st)
        elif k == 1:
            g._refit_device(st)
