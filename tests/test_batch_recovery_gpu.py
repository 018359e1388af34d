"""A batched build that stops half way leaves the sort's counts, statuses and boxes of the kernels that
ran: the next build, eager, replayed from an older graph or recorded into a new one, clears them first."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# The launches of an eager build with 8-bit digits and every mesh in one tile: vertex boxes, keys, keys'
# repair, four sort passes, tree; with 10-bit digits the histograms' scan and three passes.
@pytest.mark.parametrize("bits,stop", [(8, s) for s in (1, 2, 3, 5, 7, 8)] + [(10, s) for s in (2, 4, 6, 8)])
@pytest.mark.parametrize("then", ["eager", "replay", "new graph"])
def test_build_after_one_that_stopped(bvh, orc, bits, stop, then):
    counts = [1, 63, 1000, 900, 7]
    rng = np.random.default_rng(stop)
    vc = [n + 2 for n in counts]
    v = rng.random((sum(vc), 3), np.float32)
    f = np.concatenate([np.arange(n, dtype=np.uint32)[:, None] + np.uint32([0, 1, 2]) for n in counts])
    want, fo, vo = [], 0, 0
    for n, nv in zip(counts, vc):
        want.append(orc.lbvh(v[vo:vo + nv], f[fo:fo + n])[2].tobytes())
        fo, vo = fo + n, vo + nv
    want = b"".join(want)
    L = bvh.lib()
    b = bvh.BatchBuilder(v, f, counts, vc, radix_bits=bits)
    for _ in range(2):
        b.build(use_graph=then == "replay")
    L.bvht_setLaunchFailAfter(stop)
    with pytest.raises(bvh.BVHTestError, match="injected launch failure"):
        b.build(use_graph=False)
    L.bvht_clearError()
    for _ in range(3):
        b.nb.upload(np.zeros(b.mem.totalNodes, bvh.NODE_DTYPE))
        b.build(use_graph=then != "eager")
        assert b.nodes().tobytes() == want
        assert b.status() == 0
