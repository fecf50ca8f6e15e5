"""Batch sizes around the lines of the launch rules: the ordering grid's cells
(by the batch size, from 4,096 queries on) and the queries per wave (halved
while a batch makes fewer than eight waves per CU).  Records bit for bit against
the oracle's reference-order traversal, which neither rule may change."""
import numpy as np
import pytest

import oracle
from tests import meshes
from tests.test_gpu_disks import check, queries
from tests.test_gpu_parity import as_records, assert_bit_equal, make_scene

pytestmark = pytest.mark.gpu
fcpw = pytest.importorskip("fcpw_amd")

SIZES = (1, 3, 2047, 2048, 4095, 4096, 4097, 8191, 16385, 65535, 131073)


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("mesh", ["torus", "star2d"])
def test_batch_sizes(gpu, mesh, n):
    V, F = meshes.small_torus(48, 24) if mesh == "torus" else meshes.small_star(3000)
    _, g = make_scene(V, F)
    q = queries(V, max(n, 16), 7)[:n]
    b = oracle.Bvh(V, F)
    check(g, V, F, q, bvh=b)
    rng = np.random.default_rng(n)
    dim = V.shape[1]
    d = rng.standard_normal((n, dim))
    d = (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)
    for occlusion in (False, True):
        tmax = np.full(n, 0.7 if occlusion else np.inf, np.float32)
        hits = fcpw.GPUInteractionList()
        g.intersect(q, d, tmax, hits, check_for_occlusion=occlusion)
        assert_bit_equal(as_records(hits), b.intersect_gpuorder(q, d, tmax, occlusion))


def cast(g, n):
    hits = fcpw.GPUInteractionList()
    o = np.zeros((n, 3), np.float32)
    d = np.tile(np.array([[0.6, 0.8, 0.0]], np.float32), (n, 1))
    g.intersect(o, d, np.full(n, np.inf, np.float32), hits)


def test_a_chosen_leaf_pass_threshold_is_kept(gpu):
    """the size rule stands in for the default of ray_hold_min only"""
    _, g = make_scene(*meshes.small_torus(48, 24))
    full = 512 * g.info("n_cus")
    for value, part_filled in ((8, 1), (64, 64), (2, 2), (8, 1)):
        g.set_option("ray_hold_min", value)
        assert g.get_option("ray_hold_min") == value
        cast(g, 1000)
        assert g.info("launch_wave_queries") < 64 and g.info("launch_hold_min") == part_filled
        cast(g, full)
        assert g.info("launch_wave_queries") == 64 and g.info("launch_hold_min") == value
