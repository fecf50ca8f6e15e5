"""Batch sizes around the lines of the launch rules: the ordering grid's cells
(by the batch size, from 4,096 queries on) and the queries per wave (halved
while a batch makes fewer than eight waves per CU).  Records bit for bit against
the oracle's reference-order traversal, which neither rule may change."""
import numpy as np
import pytest

import oracle
from tests import meshes, scenes
from tests.test_gpu_disks import check, queries
from tests.test_gpu_instances import setup
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


def test_a_default_written_back_is_the_size_rule_again(gpu):
    """reading an option and setting it to what was read changes nothing"""
    _, g = make_scene(*meshes.small_torus(48, 24))
    n_small, n_full = 1000, 2048 * g.info("n_cus")
    q = queries(meshes.small_torus(48, 24)[0], n_full, 3)[:n_full]

    def entries(n):
        g.find_closest_points(q[:n], np.full(n, np.inf, np.float32), fcpw.GPUInteractionList())
        return g.info("launch_stack")

    default = g.get_option("stack")
    assert default == 6
    for _ in range(2):
        assert (entries(n_small), entries(n_full)) == (12, 6)
        g.set_option("stack", 8)
        assert (entries(n_small), entries(n_full)) == (8, 8)
        g.set_option("stack", default)


def test_a_default_block_written_back_is_the_size_rule_again(gpu):
    objs, tr, s, g, bv, I = setup("crowd3d")
    q = scenes.queries(objs, tr, 5000, seed=3)

    def block():
        g.find_closest_points(q, np.full(len(q), np.inf, np.float32), fcpw.GPUInteractionList())
        return g.info("launch_block")

    default = g.get_option("inst_seed")
    assert default == 1024
    for _ in range(2):
        assert block() == 0
        g.set_option("inst_seed", 512)
        assert block() == 512
        g.set_option("inst_seed", default)
