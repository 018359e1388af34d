"""Every sort tile size and both key chunk sizes of the batched build, meshes at the tiles' edges: each
segment is byte for byte the oracle's tree of its mesh, eager and replayed."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# keys per thread of the tile size that the counts select: 1, 1 (meshes below a tile), 2, 4, 7, 11
@pytest.mark.parametrize("counts", [
    [1023, 1024, 1025, 1, 16384, 5],
    [500, 1024, 3] * 120,
    [2047, 2048, 2049, 16385, 40000],
    [4095, 4096, 4097, 65537, 250000, 230001],
    [7167, 7168, 7169, 600000, 590000],
    [11263, 11264, 11265, 180225, 1000000, 900000]], ids=["1", "1small", "2", "4", "7", "11"])
def test_segments_at_tile_edges(bvh, orc, counts):
    rng = np.random.default_rng(len(counts) + counts[0])
    vc = [n + 2 for n in counts]
    v = rng.integers(0, 200, (sum(vc), 3)).astype(np.float32) / np.float32(64)  # many equal keys
    f = np.concatenate([np.arange(n, dtype=np.uint32)[:, None] + np.uint32([0, 1, 2]) for n in counts])
    b = bvh.BatchBuilder(v, f, counts, vc)
    for graph in (False, True, True):
        b.nb.upload(np.zeros(b.mem.totalNodes, bvh.NODE_DTYPE))
        b.build(use_graph=graph)
        nodes = b.nodes()
        assert b.status() == 0
        fo = vo = no = 0
        for n, nv in zip(counts, vc):
            if not graph:
                expect = orc.lbvh(v[vo:vo + nv], f[fo:fo + n])[2].tobytes()
                assert nodes[no:no + 2 * n - 1].tobytes() == expect, n
            fo, vo, no = fo + n, vo + nv, no + 2 * n - 1
        first = nodes if not graph else first
        assert nodes.tobytes() == first.tobytes()


def test_every_build_leaves_the_state_clear(bvh, orc):
    """One batch, every digit width and tile size in turn, eager and replayed: no build finds another's
    counts, statuses or boxes, and the error word stays 0."""
    counts = [1, 63, 1025, 4096, 30000, 7]
    rng = np.random.default_rng(4)
    vc = [n + 2 for n in counts]
    v = rng.random((sum(vc), 3), np.float32)
    f = np.concatenate([np.arange(n, dtype=np.uint32)[:, None] + np.uint32([0, 1, 2]) for n in counts])
    b = bvh.BatchBuilder(v, f, counts, vc)
    want, fo, vo = [], 0, 0
    for n, nv in zip(counts, vc):
        want.append(orc.lbvh(v[vo:vo + nv], f[fo:fo + n])[2].tobytes())
        fo, vo = fo + n, vo + nv
    want = b"".join(want)
    for bits, tile, graph in [(8, 10, False), (10, 10, False), (8, 8, True), (8, 8, True), (10, 11, True), (8, 9, False),
                              (10, 9, False), (8, 10, True)]:
        b.mem.radixBits, b.mem.tileLog2 = bits, tile
        b.nb.upload(np.zeros(b.mem.totalNodes, bvh.NODE_DTYPE))
        b.build(use_graph=graph)
        assert b.nodes().tobytes() == want, (bits, tile, graph)
        assert b.status() == 0
