"""The cooperative kernels with 64 queries in every wave (batches of at least
eight waves a CU), where leaf passes take several groups of 64: the same records
as the one-query-per-lane kernels, bit for bit, for the knobs they read."""
import numpy as np
import pytest

from fcpw_amd import synth
from tests import meshes, scenes
from tests.test_gpu_disks import CASES, queries
from tests.test_gpu_instances import setup
from tests.test_gpu_parity import as_records, make_scene
from tests.test_gpu_silhouettes import gpu_scene, records
from tests.test_oracle_silhouettes import product_scene

pytestmark = pytest.mark.gpu
fcpw = pytest.importorskip("fcpw_amd")


def full(g):
    """a batch of full waves, the last one ragged"""
    return 512 * g.info("n_cus") + 77


def noisy_sphere(amplitude):
    v, f = synth.geodesic_sphere(12)
    return synth.f32(synth.radial_noise(v, amplitude, synth.Rng(9))), f.astype(np.int32)


# with facing entries and prepass, with the prepass alone, with neither; in 2D with the entries alone
SILHOUETTES = {
    "torus": (lambda: meshes.small_torus(64, 32), 8),
    "noisy": (lambda: noisy_sphere(0.05), 8),
    "spiky": (lambda: noisy_sphere(0.6), 4),
    "soup": (CASES["soup"], 4),
    "open_plate": (CASES["plate_tilted"], 8),
    "star2d": (CASES["star2d"], 8),
    "star2d_past_the_line": (lambda: meshes.small_star((1 << 15) + 1), 8),  # no facing entries
}


@pytest.mark.parametrize("name", sorted(SILHOUETTES))
def test_silhouettes(gpu, name):
    make, entries = SILHOUETTES[name]
    V, F = make()
    g = gpu_scene(product_scene(V, F), V.shape[1])
    n = full(g)
    q = queries(V, n, 71)[:n]
    flip = (np.arange(n) % 2).astype(np.int32)
    r2 = np.full(n, np.inf, np.float32)
    r2[1::3] = np.float32((0.3 * float((V.max(0) - V.min(0)).max())) ** 2)

    def run(**opts):
        for key, value in opts.items():
            g.set_option(key, value)
        hits = fcpw.GPUInteractionList()
        g.find_closest_silhouette_points(q, r2, flip, hits)
        return records(hits).tobytes()

    ref = run(coop=0)
    for hold in (3, 1, 64):
        assert run(coop=1, sil_hold_min=hold) == ref, hold
        assert g.info("launch_wave_queries") == 64 and g.info("launch_hold_min") == hold
        assert g.info("launch_stack") == entries
    for k in (8, 12):
        assert run(sil_stack=k, sil_hold_min=3) == ref, k


@pytest.mark.parametrize("mesh", ["torus", "star2d"])
@pytest.mark.parametrize("occlusion", [False, True])
def test_rays(gpu, mesh, occlusion):
    V, F = meshes.small_torus(48, 24) if mesh == "torus" else meshes.small_star(3000)
    _, g = make_scene(V, F)
    n = full(g)
    o, d = meshes.rays_from(V, n, seed=72)
    tmax = np.full(n, np.inf, np.float32)
    tmax[::7] = 0.3

    def run(**opts):
        for key, value in opts.items():
            g.set_option(key, value)
        hits = fcpw.GPUInteractionList()
        g.intersect(o, d, tmax, hits, check_for_occlusion=occlusion)
        return as_records(hits).tobytes()

    ref = run(ray_coop=0)
    for hold in (1, 8, 64):
        assert run(ray_coop=1, ray_hold_min=hold) == ref, hold
        assert g.info("launch_wave_queries") == 64 and g.info("launch_hold_min") == hold


@pytest.mark.parametrize("mesh", ["torus", "soup", "star2d"])
def test_closest_points(gpu, mesh):
    V, F = meshes.small_torus(64, 32) if mesh == "torus" else CASES[mesh]()
    _, g = make_scene(V, F)
    n = full(g)
    q = queries(V, n, 73)[:n]
    r2 = np.full(n, np.inf, np.float32)
    r2[1::3] = np.float32((0.05 * float((V.max(0) - V.min(0)).max())) ** 2)

    def run(**opts):
        for key, value in opts.items():
            g.set_option(key, value)
        hits = fcpw.GPUInteractionList()
        g.find_closest_points(q, r2, hits, record_normals=True)
        return as_records(hits).tobytes()

    ref = run(coop=0)
    for hold in (1, 8, 64):
        for k in (6, 12):
            assert run(coop=1, hold_min=hold, stack=k) == ref, (hold, k)
            assert g.info("launch_wave_queries") == 64 and g.info("launch_hold_min") == hold


@pytest.mark.parametrize("name", scenes.NAMES + ["crowd3d"])
def test_instances(gpu, name):
    objs, tr, s, g, bv, I = setup(name)
    n = full(g)
    q = scenes.queries(objs, tr, n, seed=74)
    r2 = np.full(n, np.inf, np.float32)
    r2[1::3] = np.float32(0.04)

    def run(**opts):
        for key, value in opts.items():
            g.set_option(key, value)
        hits = fcpw.GPUInteractionList()
        obj = np.full(n, -7, np.int32)
        g.find_closest_points(q, r2, hits, record_normals=True, object_indices=obj)
        return records(hits).tobytes() + obj.tobytes()

    try:
        ref = run(coop=0)
        for hold in (1, 8, 64):
            assert run(coop=1, hold_min=hold) == ref, hold
    finally:
        run(coop=1, hold_min=1)
