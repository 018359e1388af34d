"""Walks at the edges of the packed records and of the pending stack: every hit, distance and inner-node
count equals the oracle's byte for byte."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def make_rays(bvh, pos, d):
    r = np.zeros(len(pos), bvh.RAY_DTYPE)
    r["pos"], r["dir"] = pos, d
    with np.errstate(divide="ignore"):
        r["invDir"] = np.float32(1.0) / r["dir"]
    r["sign"] = r["invDir"] < 0
    return r


def check(bvh, orc, nodes, root, v, f, rays):
    mesh, tree = bvh.DeviceMesh(v, f), bvh.DeviceBVH.from_host(nodes, root)
    pix, hits = bvh.trace_rays(tree, mesh, rays, root=root)
    opix, ohits = orc.trace(rays, nodes, root, v, f)
    assert hits.tobytes() == ohits.tobytes() and pix.tobytes() == opix.tobytes()
    skip = np.where(np.arange(len(rays)) % 3 == 0, hits["triId"], 0xFFFFFFFF).astype(np.uint32)
    pix, second = bvh.trace_rays(tree, mesh, rays, mode=1, tmin=0.5, skip=skip, root=root)
    opix, ohits = orc.trace(rays, nodes, root, v, f, mode=1, tmin=0.5, skip=skip)
    assert second.tobytes() == ohits.tobytes() and pix.tobytes() == opix.tobytes()
    return hits


# A ray from above meets the deepest leaf first and leaves one child pending on every level:
# 24 of them fit the stack, one more starts the ray over.
@pytest.mark.parametrize("n", [1, 2, 24, 25, 26, 27, 64, 66, 120])
def test_deep_trees(bvh, orc, n):
    rng = np.random.default_rng(n)
    z = (np.arange(n) / n).astype(np.float32)
    c = rng.random((n, 1, 2), np.float32) * np.float32(0.4) + np.float32(0.3)
    xy = c + (rng.random((n, 3, 2), np.float32) - np.float32(0.5)) * np.float32(0.9)
    v = np.concatenate([xy, np.broadcast_to(z[:, None, None], (n, 3, 1))], 2).reshape(-1, 3).astype(np.float32)
    f = np.arange(3 * n, dtype=np.uint32).reshape(n, 3)
    nodes = np.zeros(2 * n - 1, bvh.NODE_DTYPE)
    leaf = nodes[n - 1:]
    leaf["bbox"] = np.concatenate([v.reshape(n, 3, 3).min(1) - np.float32(1e-3), v.reshape(n, 3, 3).max(1) + np.float32(1e-3)], 1)
    leaf["isLeafFlag"], leaf["left"], leaf["right"] = 1, np.arange(n), 1
    for i in range(n - 2, -1, -1):
        l, r = n - 1 + i, (i + 1 if i + 1 < n - 1 else 2 * n - 2)
        a, b = nodes["bbox"][l], nodes["bbox"][r]
        nodes["bbox"][i] = np.concatenate([np.minimum(a[:3], b[:3]), np.maximum(a[3:], b[3:])])
        nodes["left"][i], nodes["right"][i] = l, r
        nodes["parent"][l] = nodes["parent"][r] = i
        nodes["isLeft"][l] = 1
    pos = np.concatenate([rng.random((500, 2)), np.full((500, 1), 2.0)], 1).astype(np.float32)
    d = np.concatenate([(rng.random((500, 2)) - 0.5) * 0.1, np.full((500, 1), -1.0)], 1).astype(np.float32)
    hits = check(bvh, orc, nodes, 0, v, f, make_rays(bvh, pos, d))
    assert n < 24 or (hits["triId"] != 0xFFFFFFFF).sum() > 100


# Leaves of up to `most` triangles (the builder's have one); rays along the axes from points on
# the boxes' planes (0 * inf in the slab test).
@pytest.mark.parametrize("most", [1, 2, 5, 40])
def test_leaves_of_several_triangles(bvh, orc, most):
    v, f = bvh.scene_heightfield(33, 17, 3, 0.2)
    _, order, _, _ = orc.lbvh(v, f)
    f = np.ascontiguousarray(f[order])  # faces in leaf order
    _, order, nodes, _ = orc.lbvh(v, f)
    assert np.array_equal(order, np.arange(len(f)))
    count, first = np.ones(len(nodes), np.uint32), nodes["left"].copy()
    visit, stack = [], [0]
    while stack:
        x = stack.pop()
        visit.append(x)
        if nodes["isLeafFlag"][x] == 0:
            stack += [int(nodes["left"][x]), int(nodes["right"][x])]
    for x in reversed(visit):
        if nodes["isLeafFlag"][x] == 0:
            count[x] = count[nodes["left"][x]] + count[nodes["right"][x]]
            first[x] = min(first[nodes["left"][x]], first[nodes["right"][x]])
    small = (nodes["isLeafFlag"] == 0) & (count <= most)
    nodes["isLeafFlag"][small], nodes["left"][small], nodes["right"][small] = 1, first[small], count[small]
    rng = np.random.default_rng(most)
    on = v[rng.integers(0, len(v), 600)]
    lo, hi = v.min(0), v.max(0)
    pos = rng.random((1200, 3), np.float32) * (hi - lo) * np.float32(1.5) + lo
    pos[:600] = on
    d = (rng.random((1200, 3)) - 0.5).astype(np.float32)
    d[:400] = np.eye(3, dtype=np.float32)[rng.integers(0, 3, 400)] * rng.choice([-1, 1], (400, 1)).astype(np.float32)
    pos[:600] -= d[:600] * np.float32(0.5)
    check(bvh, orc, nodes, 0, v, f, make_rays(bvh, pos, d))


# Whole waves of rays with the same signs, in every octant, and a wave with one ray that differs.
@pytest.mark.parametrize("octant", range(8))
def test_waves_of_one_octant(bvh, orc, octant):
    v, f = bvh.scene_spheres_soup(16, 2000, 77)
    nodes = orc.lbvh(v, f)[2]
    rng = np.random.default_rng(octant)
    sign = np.float32([-1 if octant >> k & 1 else 1 for k in range(3)])
    lo, hi = v.min(0), v.max(0)
    d = (rng.random((640, 3), np.float32) + np.float32(0.05)) * sign
    d[192:256] *= np.float32([0, 1, 1])  # along a plane: zeros of one sign, infinite inverses
    pos = (lo + hi) / 2 - d * np.float32(2) + (rng.random((640, 3), np.float32) - np.float32(0.5)) * (hi - lo)
    rays = make_rays(bvh, pos.astype(np.float32), d)
    rays[100]["dir"] *= -1
    rays[100]["invDir"] *= -1
    rays["sign"] = rays["invDir"] < 0
    hits = check(bvh, orc, nodes, 0, v, f, rays)
    assert (hits["triId"] != 0xFFFFFFFF).any()


# The last launch whose walks load ahead (2,560 waves on 256 CUs) and the first whose do not, as image and as rays.
@pytest.mark.parametrize("w,h", [(512, 320), (512, 321), (640, 400)])
def test_walks_ahead_and_plain(bvh, orc, w, h):
    v, f = bvh.scene_spheres_soup(16, 2000, 77)
    mesh = bvh.DeviceMesh(v, f)
    tree = bvh.lbvh_build(mesh)
    cam = ((0.5, 0.5, 2.0), (0.5, 0.5, 0.5), (0, 1, 0), 45.0)
    rays = bvh.generate_rays(w, h, *cam)
    opix, ohits = orc.trace(rays, tree.download(), 0, v, f)
    pix, hits = bvh.trace_rays(tree, mesh, rays)
    assert hits.tobytes() == ohits.tobytes() and pix.tobytes() == opix.tobytes()
    assert bvh.trace_image(tree, mesh, w, h, *cam).tobytes() == opix.tobytes()


# Bundles: 12,288 waves on 256 CUs and more.
@pytest.mark.parametrize("w,h", [(1024, 768), (1024, 776)])
def test_bundles_ahead_and_plain(bvh, orc, w, h):
    v, f = bvh.scene_heightfield(64, 32, 5, 0.2)
    mesh = bvh.DeviceMesh(v, f)
    tree = bvh.lbvh_build(mesh)
    cam = ((0.5, 1.0, 1.25), (0.5, 0.1, 0.25), (0, 1, 0), 45.0)
    opix, _ = orc.trace_bundle(bvh.generate_rays(w, h, *cam), w, h, tree.download(), 0, v, f)
    assert bvh.trace_image(tree, mesh, w, h, *cam, bundle=True).tobytes() == opix.tobytes()
