"""Node features on trees whose numbering and shape are not the builder's: the
bottom-up sums and the depths may rely on neither."""
import ctypes

import numpy as np
import pytest

from test_mlp_gpu import features_ref

pytestmark = pytest.mark.gpu


def built(bvh, n):
    v, f = bvh.scene_soup(n, 70 + n)
    mesh = bvh.DeviceMesh(v, f)
    return bvh.lbvh_build(mesh).download()


def chain(bvh, n):
    """n leaves on one path: inner node i has leaf i on the left and inner node i + 1 (the last: a
    leaf) on the right."""
    rng = np.random.default_rng(n)
    nodes = np.zeros(2 * n - 1, bvh.NODE_DTYPE)
    lo = rng.random((n, 3), np.float32)
    nodes["bbox"][n - 1:] = np.concatenate([lo, lo + rng.random((n, 3), np.float32) + np.float32(0.01)], 1)
    nodes["isLeafFlag"][n - 1:], nodes["left"][n - 1:], nodes["right"][n - 1:] = 1, np.arange(n), 1
    for i in range(n - 2, -1, -1):
        l, r = n - 1 + i, (i + 1 if i + 1 < n - 1 else 2 * n - 2)
        a, b = nodes["bbox"][l], nodes["bbox"][r]
        nodes["bbox"][i] = np.concatenate([np.minimum(a[:3], b[:3]), np.maximum(a[3:], b[3:])])
        nodes["left"][i], nodes["right"][i] = l, r
        nodes["parent"][l] = nodes["parent"][r] = i
        nodes["isLeft"][l] = 1
    d = nodes["bbox"][:, 3:] - nodes["bbox"][:, :3]
    nodes["surfaceArea"] = 2 * (d[:, 0] * d[:, 1] + d[:, 0] * d[:, 2] + d[:, 1] * d[:, 2])
    return nodes


def renumbered(nodes, seed):
    """(nodes under a random numbering, root)"""
    n = len(nodes)
    new = np.random.default_rng(seed).permutation(n).astype(np.uint32)
    out = np.empty_like(nodes)
    out[new] = nodes
    out["parent"] = new[out["parent"]]
    inner = out["isLeafFlag"] == 0
    out["left"][inner] = new[out["left"][inner]]
    out["right"][inner] = new[out["right"][inner]]
    return out, int(new[0])


# A tile of the first pass holds 1,024 leaves; depths saturate at 255.
@pytest.mark.parametrize("shape,n", [("built", 2), ("built", 3), ("built", 1023), ("built", 1024), ("built", 1025),
                                     ("built", 5000), ("chain", 2), ("chain", 257), ("chain", 258), ("chain", 1500)])
@pytest.mark.parametrize("renumber", [False, True])
def test_features_on_any_numbering(bvh, shape, n, renumber):
    nodes = built(bvh, n) if shape == "built" else chain(bvh, n)
    root = 0
    if renumber:
        nodes, root = renumbered(nodes, n)
    print(f"{shape} n={n} root={root}", flush=True)
    tree = bvh.DeviceBVH.from_host(nodes, root)
    opt = bvh.Bittner13GPU(numChunks=1)
    opt.mem = bvh.lib().allocateMemory(ctypes.byref(tree.ptr), 1, n)
    assert opt.mem.result
    bvh.lib().initData(ctypes.byref(opt.mem), ctypes.byref(tree.ptr), 128)
    assert bvh.last_error() == ""
    for _ in range(2):  # the second evaluation keeps the sums
        got = opt.features(tree)
        ref = features_ref(nodes, root)
        ref[:, 7] = np.minimum(ref[:, 7], 255 / 64)
        # sums of up to n areas and a log2 of them, in 32 bits against 64
        assert np.allclose(got, ref, rtol=1e-4, atol=1e-5), np.abs(got - ref).max(axis=0)
