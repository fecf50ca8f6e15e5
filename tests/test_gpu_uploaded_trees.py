"""Trees a caller uploads through the C ABI, which need not be those of a build:
boxes from before a vertex update, leaves whose primitives lie in another
order than the leaves do.  The records are the oracle's bit for bit, whose
traversal knows neither."""
import ctypes
import os

import numpy as np
import pytest

import oracle
from fcpw_amd import synth
from tests import meshes
from tests.test_gpu_disks import queries, torn
from tests.test_gpu_parity import assert_bit_equal
from tests.test_gpu_silhouettes import MAX_ULP_FLIPS

pytestmark = pytest.mark.gpu
fcpw = pytest.importorskip("fcpw_amd")

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fcpw_amd", "lib", "libfcpw_hip.so")
VP, I64 = ctypes.c_void_p, ctypes.c_int64
MESHES = {"torus": lambda: meshes.small_torus(64, 32), "star2d": lambda: meshes.small_star(5000)}


class Tree:
    """the arrays fcpw_hip_upload_bvh takes"""

    def __init__(self, b, F):
        self.pmin, self.pmax, self.nrefs, self.offset = (np.ascontiguousarray(a) for a in b.nodes())
        self.index = np.ascontiguousarray(b.prim_order(), np.int32)
        self.prims = np.ascontiguousarray(F[self.index], np.int32)


class Context:
    def __init__(self, dim):
        L = self.lib = ctypes.CDLL(LIB)
        L.fcpw_hip_create.argtypes = [ctypes.c_int, ctypes.POINTER(VP)]
        L.fcpw_hip_last_error.restype = ctypes.c_char_p
        L.fcpw_hip_last_error.argtypes = [VP]
        L.fcpw_hip_destroy.argtypes = [VP]
        L.fcpw_hip_upload_bvh.argtypes = [VP, ctypes.c_int, ctypes.c_int] + [VP] * 4 + [ctypes.c_int, VP, VP,
                                                                                       ctypes.c_int, VP]
        L.fcpw_hip_refit.argtypes = [VP, VP]
        L.fcpw_hip_set_option.argtypes = [VP, ctypes.c_char_p, ctypes.c_int]
        L.fcpw_hip_update_positions.argtypes = [VP, VP, ctypes.c_int]
        L.fcpw_hip_closest_points.argtypes = [VP, VP, I64, ctypes.c_int, VP]
        L.fcpw_hip_upload_silhouettes.argtypes = [VP, ctypes.c_int, VP, VP, VP, ctypes.c_int, VP]
        L.fcpw_hip_closest_silhouette_points.argtypes = [VP, VP, VP, I64, ctypes.c_float, ctypes.c_float, VP]
        self.dim, self.h = dim, VP()
        self.ok(L.fcpw_hip_create(0, ctypes.byref(self.h)))

    def __enter__(self):
        return self

    def __exit__(self, *unused):
        self.lib.fcpw_hip_destroy(self.h)

    def ok(self, st):
        assert st == 0, self.lib.fcpw_hip_last_error(self.h)

    def upload(self, t, V):
        V = np.ascontiguousarray(V, np.float32)
        self.ok(self.lib.fcpw_hip_upload_bvh(
            self.h, self.dim, len(t.nrefs), t.pmin.ctypes.data, t.pmax.ctypes.data, t.nrefs.ctypes.data,
            t.offset.ctypes.data, len(t.prims), t.prims.ctypes.data, t.index.ctypes.data, len(V), V.ctypes.data))

    def update(self, V):
        V = np.ascontiguousarray(V, np.float32)
        self.ok(self.lib.fcpw_hip_update_positions(self.h, V.ctypes.data, len(V)))

    def refit(self):
        self.ok(self.lib.fcpw_hip_refit(self.h, None))

    def option(self, key, value):
        self.ok(self.lib.fcpw_hip_set_option(self.h, key.encode(), value))

    def closest(self, q):
        s = np.full((len(q), 4), np.inf, np.float32)
        s[:, :3] = 0.0
        s[:, :self.dim] = q
        out = np.zeros(len(q), fcpw.INTERACTION_DTYPE)
        self.ok(self.lib.fcpw_hip_closest_points(self.h, s.ctypes.data, len(q), 1, out.ctypes.data))
        return out

    def check(self, b, q):
        ref = b.closest_points_gpuorder(q, record_normal=True)
        assert_bit_equal(self.closest(q), ref)


@pytest.mark.parametrize("mesh", sorted(MESHES))
def test_boxes_from_before_a_vertex_update(gpu, mesh):
    """they shrink the reference's r^2 although they hold nothing, so no subtree may be dropped"""
    V, F = MESHES[mesh]()
    b = oracle.Bvh(V, F)
    t = Tree(b, F)
    V2 = torn(V, 0)
    q = queries(V, 6000, 46)
    b.update_vertices(V2)
    with Context(V.shape[1]) as c:
        c.upload(t, V2)
        c.check(b, q)
        c.refit()
        b.refit()
        c.check(b, q)


def test_nodes_without_a_parent(gpu):
    """Arrays in which many nodes no other names all have the same second child:
    they pass the upload's checks, queries never reach them, and the slots of the
    ranges' lists would outnumber those of a tree."""
    V, F = meshes.small_torus(64, 32)  # 4,096 triangles, as the root's second child
    b = oracle.Bvh(V, F)
    t = Tree(b, F)
    E = np.array([[3.0, 0.0, 0.0], [3.0, 0.1, 0.0], [3.0, 0.0, 0.1]], np.float32)  # the first: one triangle
    extra = 5000
    pad = 2 + 2 * extra  # the root, its first child, pairs of an unnamed node and its leaf
    at = np.arange(extra) * 2 + 2
    nrefs, offset = np.zeros(pad, np.int32), np.zeros(pad, np.int32)
    nrefs[1], offset[0] = 1, pad
    nrefs[at + 1], offset[at] = 1, pad - at
    t.nrefs, t.offset = np.concatenate([nrefs, t.nrefs]), np.concatenate([offset, t.offset + (t.nrefs > 0)])
    t.offset = t.offset.astype(np.int32)
    t.pmin = np.concatenate([np.full((pad, 3), -4.0, np.float32), t.pmin])
    t.pmax = np.concatenate([np.full((pad, 3), 4.0, np.float32), t.pmax])
    t.pmin[1], t.pmax[1] = E.min(0), E.max(0)
    t.prims = np.concatenate([np.arange(3, dtype=np.int32)[None] + len(V), t.prims])
    t.index = np.concatenate([np.array([len(F)], np.int32), t.index])
    W = np.concatenate([V, E])
    q = queries(W, 3000, 51)
    ref = np.minimum(b.closest_points_gpuorder(q)["d"],
                     oracle.Bvh(E, np.array([[0, 1, 2]], np.int32)).closest_points_gpuorder(q)["d"])
    with Context(3) as c:
        c.upload(t, W)
        for refitted in (False, True):
            rec = c.closest(q)
            np.testing.assert_array_equal(rec["d"], ref)
            assert (rec["index"] == len(F)).any() and (rec["index"] < len(F)).any()
            c.option("coop", 0)
            assert c.closest(q).tobytes() == rec.tobytes()
            c.option("coop", 1)
            c.refit()


def leaves_reversed(t):
    """the same tree, its leaves' primitives laid out from the last leaf to the first"""
    n = len(t.prims)
    old = np.empty(n, np.int64)
    for i in np.nonzero(t.nrefs > 0)[0]:
        a, k = int(t.offset[i]), int(t.nrefs[i])
        new = n - a - k
        old[new:new + k] = np.arange(a, a + k)
        t.offset[i] = new
    t.prims, t.index = np.ascontiguousarray(t.prims[old]), np.ascontiguousarray(t.index[old])
    return t


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("mesh", sorted(MESHES))
def test_leaves_out_of_order(gpu, mesh, layout):
    """such a tree has no ranges: boxes alone, refitted by climbing from the leaves"""
    V, F = MESHES[mesh]()
    b = oracle.Bvh(V, F)
    q = queries(V, 6000, 61)
    with Context(V.shape[1]) as c:
        c.option("layout", layout)
        c.upload(leaves_reversed(Tree(b, F)), V)
        c.check(b, q)
        for k in range(2):
            V = (V + synth.Rng(62 + k).uniform(V.size, -0.02, 0.02).reshape(V.shape)).astype(np.float32)
            c.update(V)
            c.refit()
            b.update_vertices(V)
            b.refit()
            c.check(b, q)


@pytest.mark.parametrize("mesh", sorted(MESHES))
def test_silhouettes_with_leaves_out_of_order(gpu, mesh):
    """such a tree has no facing entries: the cooperative kernel against the
    per-lane one bit for bit, and the oracle's traversal, which may round a cone
    test the other way in MAX_ULP_FLIPS queries"""
    V, F = MESHES[mesh]()
    b = oracle.Bvh(V, F)
    b.build_silhouettes()
    cones, count, offset, rec = b.silhouettes()
    if V.shape[1] == 2:  # fcpw_hip_vertex has one point
        rec = np.ascontiguousarray(rec[["pa", "n0", "n1", "index", "has_one_adjacent_face"]].astype(
            [("pa", "<f4", (3,)), ("n0", "<f4", (3,)), ("n1", "<f4", (3,)), ("index", "<u4"), ("one", "<u4")]))
    q = queries(V, 4000, 63)
    s = np.full((len(q), 4), np.finfo(np.float32).max, np.float32)
    s[:, :3] = 0.0
    s[:, :V.shape[1]] = q
    flip = (np.arange(len(q)) % 2).astype(np.uint32)
    with Context(V.shape[1]) as c:
        c.upload(leaves_reversed(Tree(b, F)), V)
        c.ok(c.lib.fcpw_hip_upload_silhouettes(c.h, len(count), cones.ctypes.data, count.ctypes.data,
                                               offset.ctypes.data, len(rec), rec.ctypes.data))
        out = []
        for coop in (1, 0):
            c.option("coop", coop)
            o = np.zeros(len(q), fcpw.INTERACTION_DTYPE)
            c.ok(c.lib.fcpw_hip_closest_silhouette_points(c.h, s.ctypes.data, flip.ctypes.data, len(q), 0.0, 1e-3,
                                                          o.ctypes.data))
            out.append(o)
        assert out[0].tobytes() == out[1].tobytes()
        ref = b.closest_silhouettes(q, flip=flip)
        same = (out[0]["index"].view(np.int32) == ref["index"]) & (out[0]["d"] == ref["d"])
        assert (~same).sum() <= MAX_ULP_FLIPS


@pytest.mark.parametrize("shared", [False, True])
def test_silhouettes_out_of_leaf_order(gpu, shared):
    """a caller's records in another order than the leaves (they are laid out in
    leaf order), and leaves that share records (no facing entries): the oracle's
    silhouettes, before and after a refit"""
    V, F = MESHES["torus"]()
    b = oracle.Bvh(V, F)
    b.build_silhouettes()
    cones, count, offset, rec = b.silhouettes()
    if shared:  # one leaf also lists the record that follows its own
        leaf = np.nonzero(count)[0]
        count[leaf[np.argmin(offset[leaf])]] += 1
    else:
        order = np.random.default_rng(5).permutation(np.nonzero(count)[0])
        new, at = np.empty_like(rec), 0
        for i in order:
            new[at:at + count[i]] = rec[offset[i]:offset[i] + count[i]]
            offset[i], at = at, at + count[i]
        rec = new
    q = queries(V, 4000, 64)
    s = np.full((len(q), 4), np.finfo(np.float32).max, np.float32)
    s[:, :3] = q
    flip = np.zeros(len(q), np.uint32)
    with Context(3) as c:
        c.upload(Tree(b, F), V)
        c.ok(c.lib.fcpw_hip_upload_silhouettes(c.h, len(count), cones.ctypes.data, count.ctypes.data,
                                               offset.ctypes.data, len(rec), rec.ctypes.data))
        for refitted in (False, True):
            out = []
            for coop in (1, 0):
                c.option("coop", coop)
                o = np.zeros(len(q), fcpw.INTERACTION_DTYPE)
                c.ok(c.lib.fcpw_hip_closest_silhouette_points(c.h, s.ctypes.data, flip.ctypes.data, len(q), 0.0,
                                                              1e-3, o.ctypes.data))
                out.append(o)
            assert out[0].tobytes() == out[1].tobytes()
            if not refitted:
                ref = b.closest_silhouettes(q, flip=flip)
                same = (out[0]["index"].view(np.int32) == ref["index"]) & (out[0]["d"] == ref["d"])
                assert (~same).sum() <= MAX_ULP_FLIPS
            c.refit()
