"""Chunks over trees whose insertion points lie deeper than a patch's stored path: a built tree below a
path of nodes with a leaf each.  Trees and counters after every chunk equal the oracle's replay."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def grafted(bvh, n, c):
    """Inner nodes 0 .. c - 1 on a path (the root is 0), a built tree of n triangles below it, c leaves last."""
    v, f = bvh.scene_soup(n + c, n)
    sub = bvh.lbvh_build(bvh.DeviceMesh(v, f[:n])).download()
    inner = sub["isLeafFlag"] == 0
    sub["parent"] += c
    sub["left"][inner] += c
    sub["right"][inner] += c
    nodes = np.zeros(2 * (n + c) - 1, bvh.NODE_DTYPE)
    nodes[c:c + len(sub)] = sub
    first = c + len(sub)
    tri = v[f[n:]].astype(np.float32)
    leaf, path = nodes[first:], nodes[:c]
    leaf["bbox"] = np.concatenate([tri.min(1), tri.max(1)], 1)
    leaf["isLeafFlag"], leaf["left"], leaf["right"], leaf["isLeft"] = 1, n + np.arange(c), 1, 1
    leaf["parent"] = np.arange(c)
    path["left"], path["right"] = first + np.arange(c), 1 + np.arange(c)
    path["parent"] = np.maximum(np.arange(c) - 1, 0)
    nodes["parent"][c], nodes["isLeft"][c] = c - 1, 0
    for i in range(c - 1, -1, -1):
        a, b = leaf["bbox"][i], nodes["bbox"][i + 1]
        path["bbox"][i] = np.concatenate([np.minimum(a[:3], b[:3]), np.maximum(a[3:], b[3:])])
    d = nodes["bbox"][:, 3:] - nodes["bbox"][:, :3]
    nodes["surfaceArea"] = 2 * (d[:, 0] * d[:, 1] + d[:, 0] * d[:, 2] + d[:, 1] * d[:, 2])
    return nodes


# 127 nodes of a path are stored where a chunk has at most a 32nd of the nodes (the first line), none where
# it has more; the last of each: more patches than a workgroup has
@pytest.mark.parametrize("n,c,percent,chunks", [(2000, c, 10.0, 4) for c in (100, 113, 114, 115, 116, 117, 600)] +
                                               [(30000, 200, 12.0, 4)] +
                                               [(2000, c, 10.0, 2) for c in (100, 128, 600)] +
                                               [(4000, 150, 9.0, 1), (30000, 200, 20.0, 2)])
def test_deep_paths_equal_replay(bvh, orc, n, c, percent, chunks):
    nodes = grafted(bvh, n, c)
    rc, _, _, st, trees = orc.bittner_gpuref(nodes, percent, chunks, 2, search=1, chunk_trees=True)
    assert rc == 0
    tree = bvh.DeviceBVH.from_host(nodes)
    opt = bvh.Bittner13GPU(maxNumStepps=2, numChunks=chunks, batchPercent=percent)
    opt.setup(tree, n + c)
    print(f"K={opt.chunk}", flush=True)
    cfg, L = opt.cfg(opt.chunk), bvh.lib()
    for s in range(2):
        L.bn13_selectNodes(ctypes.byref(opt.mem), ctypes.byref(tree.ptr), cfg)
        for k in range(chunks):
            L.bn13_rmAndReinsChunk(ctypes.byref(opt.mem), ctypes.byref(tree.ptr), cfg, k)
            assert tree.download().tobytes() == trees[s * chunks + k].tobytes(), (s, k)
    got = opt.stats()
    assert bvh.last_error() == "" and got["applied"] > 0 and got["unresolved"] == 0
    assert got["contained"] == int(st[2]) and got["contained"] > 0


def test_memory_of_a_large_chunk(bvh):
    """A patch of a chunk with half of the nodes takes no stored path: its record, entries, slots and starts
    are 528 bytes."""
    L = bvh.lib()
    with open("/proc/self/maps") as maps:  # the HIP runtime that the library uses
        hip = ctypes.CDLL(next(l.split()[-1] for l in maps if "libamdhip64" in l))

    def free():
        got, total = ctypes.c_size_t(), ctypes.c_size_t()
        L.doCudaDevSync()
        assert hip.hipMemGetInfo(ctypes.byref(got), ctypes.byref(total)) == 0
        return got.value

    n = 500000
    v, f = bvh.scene_soup(n, 3)
    tree = bvh.lbvh_build(bvh.DeviceMesh(v, f))
    used = []
    for K in (1, n - 1):
        before = free()
        mem = L.allocateMemory(ctypes.byref(tree.ptr), K, n)
        assert mem.result
        used.append(before - free())
        L.freeMemory(ctypes.byref(mem))
    print(f"{used[0]} bytes with 1 patch, {(used[1] - used[0]) / n:.1f} more per patch", flush=True)
    assert used[1] - used[0] < 528 * n + (64 << 20)  # allocations are rounded up
