"""Chunk kernels of the optimizer at the sizes where their paths change."""
import ctypes

import numpy as np
import pytest

from test_bittner_gpu import replay_check
from test_features_numbering_gpu import chain
from test_mlp_gpu import features_ref

pytestmark = pytest.mark.gpu


# One chunk of K patches per step on 3,840 triangles, K on either side of what
# the conflict rounds hold per thread (1,024) and in LDS (1,638).
@pytest.mark.parametrize("percent", [0.3, 13.0, 14.0, 21.0, 22.0, 35.0, 49.0])
def test_conflict_rounds_equal_replay(bvh, orc, percent):
    v, f = bvh.scene_heightfield(48, 40, 51, 0.2)
    print(f"K={int(percent / 100 * (2 * len(f) - 1))}", flush=True)
    replay_check(bvh, orc, v, f, 2, 1, percent, search=1)


# Chunks with one, two and three rounds over the whole GPU (767 and 768 patches, 4,095 and 4,096), and one
# that leaves more undecided patches than the workgroup's table holds.
@pytest.mark.parametrize("grid,percent", [((48, 40), 9.993), ((48, 40), 10.008), ((128, 64), 12.499), ((128, 64), 12.503),
                                          ((256, 128), 20.0)])
def test_round_counts_equal_replay(bvh, orc, grid, percent):
    v, f = bvh.scene_heightfield(*grid, 53, 0.2)
    print(f"K={int(np.float32(percent) / np.float32(100.0) * np.float32(2 * len(f) - 1))}", flush=True)
    replay_check(bvh, orc, v, f, 1, 1, percent, search=1)


# Refits from lists of leaves: one walk, a workgroup's edge (256), more than the
# meeting places of one launch (a quarter of the leaves), all leaves, all of
# them twice over and some inner nodes among them.
@pytest.mark.parametrize("count", [1, 2, 63, 255, 256, 257, 2000, 2001, "all", "twice"])
def test_refit_from_leaf_lists(bvh, orc, count):
    v, f = bvh.scene_spheres_soup(8, 4000, 61)
    mesh = bvh.DeviceMesh(v, f)
    tree = bvh.lbvh_build(mesh)
    opt = bvh.Bittner13GPU(maxNumStepps=1, numChunks=4, batchPercent=0.5)
    opt.run(tree, len(f))
    nodes = tree.download()
    rng = np.random.default_rng(5)
    leaves = np.nonzero(nodes["isLeafFlag"] != 0)[0].astype(np.uint32)
    inner = np.nonzero(nodes["isLeafFlag"] == 0)[0].astype(np.uint32)
    moved = leaves if count in ("all", "twice") else np.sort(rng.choice(leaves, count, replace=False))
    starts = moved
    if count == "twice":
        starts = rng.permutation(np.concatenate([moved, moved, rng.choice(inner, 500)]))
    print(f"{len(starts)} starts over {len(leaves)} leaves", flush=True)
    v2 = v + rng.uniform(-0.05, 0.05, v.shape).astype(np.float32)
    L = bvh.lib()
    mem, raw = opt.mem, mesh.raw
    d_moved = bvh.DeviceBuffer(moved.nbytes).upload(moved)
    d_starts = bvh.DeviceBuffer(starts.nbytes).upload(starts)
    assert L.runMemcpy(raw.vert, v2.ctypes.data_as(ctypes.c_void_p), v2.nbytes, 1)
    L.refitDynamicTris(ctypes.byref(tree.ptr), raw, d_moved.ptr, len(moved), 64)
    assert L.bvht_fixTreeFrom(ctypes.byref(mem), ctypes.byref(tree.ptr), d_starts.ptr, len(starts))
    L.doCudaDevSync()
    assert bvh.last_error() == ""
    want = orc.fix_tree1(orc.refit_leaf_tris(nodes, v2, f, moved))
    assert tree.download().tobytes() == want.tobytes()
    assert opt.stats()["unresolved"] == 0
    # the words are clear again: the next refit from one leaf changes nothing
    assert L.bvht_fixTreeFrom(ctypes.byref(mem), ctypes.byref(tree.ptr), d_starts.ptr, 1)
    L.doCudaDevSync()
    assert tree.download().tobytes() == want.tobytes()


# Trees of one path: the nodes above an insertion point fit its stored path (127), or one workgroup
# checks every patch of the chunk.
@pytest.mark.parametrize("leaves", [40, 126, 127, 128, 129, 130, 700])
def test_deep_trees_equal_replay(bvh, orc, leaves):
    nodes = chain(bvh, leaves)
    steps, chunks, percent = 3, 2, 12.0
    rc, _, _, _, trees = orc.bittner_gpuref(nodes, percent, chunks, steps, search=1, chunk_trees=True)
    assert rc == 0
    tree = bvh.DeviceBVH.from_host(nodes)
    opt = bvh.Bittner13GPU(maxNumStepps=steps, numChunks=chunks, batchPercent=percent)
    opt.setup(tree, leaves)
    cfg, L = opt.cfg(opt.chunk), bvh.lib()
    for s in range(steps):
        L.bn13_selectNodes(ctypes.byref(opt.mem), ctypes.byref(tree.ptr), cfg)
        for c in range(chunks):
            L.bn13_rmAndReinsChunk(ctypes.byref(opt.mem), ctypes.byref(tree.ptr), cfg, c)
            assert tree.download().tobytes() == trees[s * chunks + c].tobytes(), (s, c)
    st = opt.stats()
    assert bvh.last_error() == "" and st["applied"] > 0 and st["unresolved"] == 0 and st["runaway"] == 0


# Node and leaf lists whose lengths lie at the edges of a wave (64 items) and of a block (4,096).
@pytest.mark.parametrize("n", [2, 31, 32, 33, 2047, 2048, 2049, 4096, 4097, 10000])
def test_ordered_selections(bvh, orc, n):
    v, f = bvh.scene_soup(n, n)
    mesh = bvh.DeviceMesh(v, f)
    tree = bvh.lbvh_build(mesh)
    nodes = tree.download()
    opt = bvh.Bittner13GPU(maxNumStepps=1, numChunks=1, batchPercent=75.0)
    opt.setup(tree, n)
    ids = bvh.DeviceBuffer(4 * n)
    num = ctypes.c_uint32()
    leaves = np.nonzero(nodes["isLeafFlag"] != 0)[0]
    for begin in (0, 1, n // 2, n - 1, n):
        bvh.lib().selectDynamicLeafNodes(ctypes.byref(opt.mem), ctypes.byref(tree.ptr), ids.ptr, ctypes.byref(num), begin)
        assert bvh.last_error() == ""
        want = leaves[nodes["left"][leaves] >= begin]
        assert num.value == len(want) and np.array_equal(ids.download(np.uint32, num.value), want)
    ref = features_ref(nodes)  # by inner node id
    assert np.allclose(opt.features(tree), ref, rtol=1e-5, atol=1e-6)
