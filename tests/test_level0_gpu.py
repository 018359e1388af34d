"""Boxes inside a wave and inner nodes of partly filled tiles: every remainder of a wave, of a tile and of
two tiles, per tile size, byte for byte the oracle's tree."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile", [8, 9, 10, 11])
def test_partial_waves_and_tiles(bvh, orc, tile):
    rng = np.random.default_rng(tile)
    T = 1 << tile
    counts = list(range(1, 70)) + [127, 128, 129, T - 65, T - 1, T, T + 1, T + 33, 2 * T - 1, 2 * T + 1, 5 * T + 7]
    fs, vs = [], []
    for n in counts:  # coordinates with many ties, zeros of both signs included
        v = rng.choice(np.float32([-1.5, -0.0, 0.0, 0.25, 1.0, 3.0]), (3 * n, 3)).astype(np.float32)
        v += rng.choice(np.float32([0.0, 0.125]), (3 * n, 3))
        vs.append(v)
        fs.append(np.arange(3 * n, dtype=np.uint32).reshape(n, 3))
    for v, f in zip(vs[60:], fs[60:]):
        mesh = bvh.DeviceMesh(v, f)
        b = bvh.LBVHBuilder(mesh, 30, tile_log2=tile)
        tree = b.allocate_bvh()
        b.build(tree)
        assert tree.download().tobytes() == orc.lbvh(v, f)[2].tobytes(), len(f)
    b = bvh.BatchBuilder(np.concatenate(vs), np.concatenate(fs), counts, [3 * n for n in counts], tile_log2=tile)
    b.build()
    nodes, at = b.nodes(), 0
    for v, f in zip(vs, fs):
        assert nodes[at:at + 2 * len(f) - 1].tobytes() == orc.lbvh(v, f)[2].tobytes(), len(f)
        at += 2 * len(f) - 1
