"""The onesweep at the key counts where its tile size changes (on a 256-CU device:
128 tiles of 512 and 1,024 keys, 256 of 2,048 to 12,288) and one key more, against
numpy's stable order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EDGES = [512, 128 * 512, 128 * 1024, 256 * 2048, 256 * 4096, 256 * 8192, 256 * 12288]


@pytest.mark.parametrize("more", [0, 1])
@pytest.mark.parametrize("n", EDGES)
@pytest.mark.parametrize("bits", [30, 63])
def test_tile_edges(bvh, bits, n, more):
    n += more
    rng = np.random.default_rng(n + bits)
    # a third of the keys from a few values: equal keys keep their order across tiles
    keys = rng.integers(0, 1 << bits, n, dtype=np.uint64)
    keys[rng.random(n) < 0.33] &= np.uint64(((1 << bits) - 1) & ~((1 << (bits - 3)) - 1))
    keys = keys.astype(np.uint64 if bits == 63 else np.uint32)
    print(f"n={n} bits={bits}", flush=True)
    idx, sk = bvh.sort_key_index_pairs(keys, bits, 8)
    ref = np.argsort(keys, kind="stable").astype(np.uint32)
    assert np.array_equal(idx, ref)
    assert np.array_equal(sk, keys[ref])


# the full build (packed 63-bit keys) past one tile size and the next
@pytest.mark.parametrize("n", [8193, 65537, 131073, 524289])
@pytest.mark.parametrize("bits", [30, 63])
def test_builds_at_tile_edges(bvh, orc, n, bits):
    v, f = bvh.scene_soup(n, 100 + n)
    _, order, expect, _ = orc.lbvh(v, f, bits)
    b = bvh.LBVHBuilder(bvh.DeviceMesh(v, f), bits)
    tree = b.allocate_bvh()
    for _ in range(2):
        b.build(tree)
        assert b.sort_status() == 0
        assert np.array_equal(b.sorted_faces(), order)
        assert tree.download().tobytes() == expect.tobytes()
