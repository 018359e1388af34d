"""One-round sort passes wait for no workgroup that may not have started: a tile whose counts do not come
is counted by the workgroup that needs them.  Every tile counted that way (0 looks), and all that are
late (1 look), at every tile size."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def default_polls(bvh):
    yield
    bvh.lib().bvht_setSortPolls(-1)


# the last size is a partial tile behind whole ones for every tile of 512 to 17,408 keys (128 and 256 tiles
# at most); 63-bit keys above 8,192 take the digits of both words
@pytest.mark.parametrize("polls", [0, 1])
@pytest.mark.parametrize("bits", [30, 63])
@pytest.mark.parametrize("n", [513, 65536, 65537, 130000, 262145, 600000, 1100000, 2100000, 3150000, 4300000])
def test_missing_counts_are_made(bvh, bits, n, polls):
    rng = np.random.default_rng(n + bits)
    print(f"n={n} bits={bits} polls={polls}", flush=True)
    # equal digits over whole tiles (a count of 17,408) and random ones
    keys = rng.integers(0, 1 << bits, n, np.uint64)
    keys[n // 3:2 * n // 3] &= np.uint64((1 << bits) - 1 - 0xFF00)
    keys = keys if bits == 63 else keys.astype(np.uint32)
    bvh.lib().bvht_setSortPolls(polls)
    vals, out = bvh.sort_key_index_pairs(keys, bits)
    order = np.argsort(keys, kind="stable")
    assert np.array_equal(vals, order.astype(np.uint32)) and np.array_equal(out, keys[order])


# whole builds: identity values, packed 63-bit keys without values, and the error word
@pytest.mark.parametrize("bits", [30, 63])
@pytest.mark.parametrize("n", [9000, 300001, 2000003])
def test_builds(bvh, bits, n):
    v, f = bvh.scene_soup(n, 5)
    b = bvh.LBVHBuilder(bvh.DeviceMesh(v, f), bits)
    want, got = b.allocate_bvh(), b.allocate_bvh()
    b.build(want)
    for polls in (0, 1):
        bvh.lib().bvht_setSortPolls(polls)
        b.build(got)
        assert got.download().tobytes() == want.download().tobytes()
        assert b.sort_status() == 0
