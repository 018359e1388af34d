"""The sort status is the last sort's: errors that an earlier one left in the scratch are gone after any
full build, in one workgroup (up to 8,192 triangles) and past it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [30, 63])
@pytest.mark.parametrize("n", [1, 3000, 8192, 8193])
def test_status_after_an_earlier_error(bvh, bits, n):
    v, f = bvh.scene_soup(n, 11)
    b = bvh.LBVHBuilder(bvh.DeviceMesh(v, f), bits)
    tree = b.allocate_bvh()
    ones = np.full(b.mem.sortScratchBytes // 4, 0xFFFFFFFF, np.uint32)
    assert bvh.lib().runMemcpy(b.mem.sortScratch, bvh._ptr(ones), ones.nbytes, 1)
    assert b.sort_status() != 0
    b.build(tree)
    assert b.sort_status() == 0
    first = tree.download()
    b.build_staged(tree)
    assert b.sort_status() == 0 and tree.download().tobytes() == first.tobytes()
