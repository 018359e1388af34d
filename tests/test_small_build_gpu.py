"""Builds on either side of what one workgroup sorts: multiples of 1,024 triangles
per workgroup up to 8,192, and one more."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def scene(bvh, kind, n):
    if kind == "soup":
        return bvh.scene_soup(n, 90 + n)
    if kind == "equal":  # every key equal: the order is the index order
        v, f = bvh.scene_soup(1, 3)
        return v, np.repeat(f, n, axis=0)
    v, f = bvh.scene_soup(n, 7)  # a stray vertex outside the triangles' box
    return np.concatenate([v, [[9.0, -4.0, 6.0]]]).astype(np.float32), f


@pytest.mark.parametrize("bits", [30, 63])
@pytest.mark.parametrize("kind,n", [("soup", n) for n in (1, 2, 3, 63, 64, 65, 1023, 1024, 1025, 2049, 3073, 4097, 5121,
                                                          6145, 7169, 8191, 8192, 8193)] +
                         [("equal", 3000), ("stray", 2500)])
def test_small_builds(bvh, orc, kind, n, bits):
    v, f = scene(bvh, kind, n)
    print(f"{kind} n={n} bits={bits}", flush=True)
    keys, order, expect, _ = orc.lbvh(v, f, bits)
    b = bvh.LBVHBuilder(bvh.DeviceMesh(v, f), bits)
    tree = b.allocate_bvh()
    for _ in range(2):
        b.build(tree)
        assert b.sort_status() == 0
        assert np.array_equal(b.sorted_faces(), order)
        assert tree.download().tobytes() == expect.tobytes()
    # the key-based topology needs the sorted keys
    karras = bvh.LBVHBuilder(bvh.DeviceMesh(v, f), bits, topology=1)
    t1 = karras.allocate_bvh()
    karras.build(t1)
    assert np.array_equal(karras.sorted_faces(), order)
    if n > 1:
        assert np.array_equal(karras.sorted_keys(), keys)
