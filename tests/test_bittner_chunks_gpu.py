"""Chunk kernels of the optimizer at the sizes where their paths change."""
import pytest

from test_bittner_gpu import replay_check

pytestmark = pytest.mark.gpu


# One chunk of K patches per step on 3,840 triangles, K on either side of what
# the conflict rounds hold per thread (1,024) and in LDS (1,638).
@pytest.mark.parametrize("percent", [0.3, 13.0, 14.0, 21.0, 22.0, 35.0, 49.0])
def test_conflict_rounds_equal_replay(bvh, orc, percent):
    v, f = bvh.scene_heightfield(48, 40, 51, 0.2)
    print(f"K={int(percent / 100 * (2 * len(f) - 1))}", flush=True)
    replay_check(bvh, orc, v, f, 2, 1, percent, search=1)
