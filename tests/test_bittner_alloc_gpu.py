"""A first use of the learned priority's or altSort's memory that fails at any of its allocations can be
made again."""
import ctypes

import numpy as np
import pytest

from test_mlp_gpu import features_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fail", [1, 2, 3, 4])
def test_features_after_a_failed_allocation(bvh, fail):
    v, f = bvh.scene_soup(3000, 2)
    tree = bvh.lbvh_build(bvh.DeviceMesh(v, f))
    opt = bvh.Bittner13GPU(numChunks=1)
    opt.setup(tree, len(f))
    out = bvh.DeviceBuffer(48 * opt.mem.numInnerNodes)
    args = ctypes.byref(opt.mem), ctypes.byref(tree.ptr), out.ptr
    bvh.lib().bvht_setAllocFailAfter(fail)
    assert not bvh.lib().bvht_bn13_features(*args)
    assert "injected allocation failure" in bvh.last_error()
    bvh.lib().bvht_clearError()
    assert bvh.lib().bvht_bn13_features(*args)
    got = out.download(np.float32, 12 * opt.mem.numInnerNodes).reshape(-1, 12)
    assert np.allclose(got, features_ref(tree.download()), rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("fail", [1, 2])
def test_alt_sort_after_a_failed_allocation(bvh, fail):
    v, f = bvh.scene_soup(3000, 2)
    mesh, trees = bvh.DeviceMesh(v, f), []
    for first in (fail, 0):
        tree = bvh.lbvh_build(mesh)
        opt = bvh.Bittner13GPU(numChunks=2, batchPercent=5.0, altSort=True)
        opt.setup(tree, len(f))
        if first:
            bvh.lib().bvht_setAllocFailAfter(first)
            bvh.lib().bn13_selectNodes(ctypes.byref(opt.mem), ctypes.byref(tree.ptr), opt.cfg(opt.chunk))
            assert "injected allocation failure" in bvh.last_error()
            bvh.lib().bvht_clearError()
        opt.step(tree)
        trees.append(tree.download().tobytes())
    assert trees[0] == trees[1]
