"""Refits from lists of more than a quarter of the leaves: in order and mixed, on the builder's numbering
and on any, over wide and deep trees, with leaves named more than once and inner nodes among them."""
import ctypes

import numpy as np
import pytest

from test_features_numbering_gpu import chain, renumbered

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [3, 4, 255, 1024, 1025, 20000])
@pytest.mark.parametrize("shape", ["built", "built renumbered", "chain", "chain renumbered"])
@pytest.mark.parametrize("lists", ["half", "all in order", "all mixed", "three times"])
def test_long_lists(bvh, orc, shape, n, lists):
    if shape.startswith("chain"):
        n = min(n, 1500)
        nodes = chain(bvh, n)
    else:
        v, f = bvh.scene_soup(n, n)
        nodes = bvh.lbvh_build(bvh.DeviceMesh(v, f)).download()
    root = 0
    if "renumbered" in shape:
        nodes, root = renumbered(nodes, n)
    rng = np.random.default_rng(n)
    leaves = np.nonzero(nodes["isLeafFlag"] != 0)[0].astype(np.uint32)
    inner = np.nonzero(nodes["isLeafFlag"] == 0)[0].astype(np.uint32)
    starts = {"half": rng.permutation(leaves)[:(n + 1) // 2], "all in order": leaves, "all mixed": rng.permutation(leaves),
              "three times": rng.permutation(np.concatenate([leaves, leaves, leaves, inner[::3]]))}[lists]
    moved = np.unique(starts)
    moved = moved[nodes["isLeafFlag"][moved] != 0]
    tree = bvh.DeviceBVH.from_host(nodes, root)
    opt = bvh.Bittner13GPU(numChunks=1)
    opt.mem = bvh.lib().allocateMemory(ctypes.byref(tree.ptr), 1, n)
    assert opt.mem.result
    L = bvh.lib()
    L.initData(ctypes.byref(opt.mem), ctypes.byref(tree.ptr), 128)
    print(f"{shape} n={n} {lists}: {len(starts)} starts", flush=True)
    d = bvh.DeviceBuffer(starts.nbytes).upload(starts)
    for _ in range(2):  # the second finds the words as the first did
        lo = rng.random((len(moved), 3), np.float32)
        nodes["bbox"][moved] = np.concatenate([lo, lo + rng.random((len(moved), 3), np.float32)], 1)
        assert L.runMemcpy(tree.ptr.nodes, bvh._ptr(nodes), nodes.nbytes, 1)
        assert L.bvht_fixTreeFrom(ctypes.byref(opt.mem), ctypes.byref(tree.ptr), d.ptr, len(starts))
        want = orc.fix_tree1(nodes)
        assert tree.download().tobytes() == want.tobytes()
        assert bvh.last_error() == "" and opt.stats()["unresolved"] == 0
        nodes = want
