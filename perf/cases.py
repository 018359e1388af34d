"""Performance cases of the BVH pipeline: what a program that builds, optimises,
refits and traces bounding volume hierarchies with this package asks of it.

  build      LBVH build of one mesh already on the device (the LBVH command)
  batch      one segmented build of many meshes, replayed from its graph
  image      camera rays + traced image (the CUDATracer command)
  frame      camera rays, primary hits + image, one diffuse bounce, its hits
  optimise   LBVH build, then steps of the Bittner13 optimizer (the LBVH and
             bittner13GPU commands), heuristic or learned removal priority
  refit      a frame of a scene whose last triangles move: their leaf boxes and
             the paths above them

`listed` gives the named cases, `draw` others of the same ranges.  Meshes are
seeded synthetic scenes of this repository's kinds: heightfields, icosphere
clusters with triangle soup, and batches of both.  Every buffer that a case
returns is the program's own device memory, handed to the package by pointer.
"""
import ctypes
import math
import os
import random

import numpy as np
import torch

import bvhtest_amd as bt

HERE = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
FLT_EPSILON = 1.1920928955078125e-07
CAM = {"pos": (0.5, 0.5, 2.0), "look_at": (0.5, 0.5, 0.5)}  # in front of the unit cube
CAM_FIELD = {"pos": (0.5, 1.0, 1.25), "look_at": (0.5, 0.1, 0.25)}  # above a heightfield
LIGHT = (2.0, 2.0, 2.0)


def listed():
    return [
        # one small object, rebuilt each frame: launches and latency count
        {"name": "build_4k", "kind": "build", "scene": "field", "gx": 64, "gz": 32, "bits": 30},
        # the 65,536-triangle heightfield, reference keys
        {"name": "build_65k", "kind": "build", "scene": "field", "gx": 256, "gz": 128, "bits": 30},
        # an ordinary production mesh, an odd count, long keys
        {"name": "build_1m", "kind": "build", "scene": "clusters", "tris": 1003207, "bits": 63},
        # the benchmark scene's size
        {"name": "build_4m", "kind": "build", "scene": "clusters", "tris": 4236960, "bits": 63},
        # the objects of one scene, rebuilt together
        {"name": "batch_64", "kind": "batch", "meshes": 64, "min": 100, "max": 60000, "sizes": 5},
        # an asset library: 512 meshes of 1,000 to 500,000 triangles
        {"name": "batch_512", "kind": "batch", "meshes": 512, "min": 1000, "max": 500000, "sizes": 1},
        # the image command on the 65,536-triangle heightfield
        {"name": "image_65k", "kind": "image", "scene": "field", "gx": 256, "gz": 128, "w": 1024, "h": 1024,
         "bundle": False},
        # one full-HD frame with a diffuse bounce on the benchmark scene's size
        {"name": "frame_4m", "kind": "frame", "scene": "clusters", "tris": 4236960, "w": 1920, "h": 1080},
        # a small tree: 10% of the nodes per step in 8 chunks
        {"name": "optimise_65k", "kind": "optimise", "scene": "field", "gx": 256, "gz": 128, "bits": 30,
         "percent": 10.0, "chunks": 8, "steps": 3, "learned": False},
        # the optimizer's defaults: 1% of the nodes per step in 32 chunks
        {"name": "optimise_1m", "kind": "optimise", "scene": "clusters", "tris": 1003207, "bits": 63,
         "percent": 1.0, "chunks": 32, "steps": 3, "learned": False},
        # the same with the learned removal priority on the benchmark scene's size
        {"name": "learned_4m", "kind": "optimise", "scene": "clusters", "tris": 4236960, "bits": 63,
         "percent": 1.0, "chunks": 32, "steps": 2, "learned": True},
        # an animated part of a large static scene
        {"name": "refit_1m", "kind": "refit", "tris": 1003207, "moving": 100000},
    ]


def log_int(rng, lo, hi):
    """An integer between lo and hi, spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def scene_fields(rng, lo, hi):
    """A heightfield or a cluster scene of lo to hi triangles."""
    n = log_int(rng, lo, hi)
    if rng.random() < 0.35:
        gx = max(2, int(math.sqrt(n * rng.uniform(0.3, 1.5))))
        return {"scene": "field", "gx": gx, "gz": max(1, n // (2 * gx))}
    return {"scene": "clusters", "tris": n}


def draw(rng):
    kind = rng.choice(["build", "build", "batch", "image", "frame", "optimise", "refit"])
    c = {"kind": kind}
    if kind == "build":
        c.update(scene_fields(rng, 1000, 16900000), bits=rng.choice([30, 63]))
    elif kind == "batch":
        lo = log_int(rng, 50, 2000)
        c.update(meshes=log_int(rng, 8, 512), min=lo, max=lo * log_int(rng, 4, 200), sizes=rng.randrange(1 << 20))
    elif kind == "image":
        c.update(scene_fields(rng, 2000, 2000000), w=log_int(rng, 160, 1920), h=log_int(rng, 120, 1080),
                 bundle=rng.random() < 0.3)
    elif kind == "frame":
        c.update(scene="clusters", tris=log_int(rng, 20000, 4236960), w=log_int(rng, 320, 1920), h=log_int(rng, 240, 1080))
    elif kind == "optimise":
        learned = rng.random() < 0.4
        chunks = rng.choice([8, 16, 32])
        c.update(scene_fields(rng, 30000, 4236960), bits=rng.choice([30, 63]), percent=rng.choice([1.0, 2.0, 5.0]),
                 chunks=chunks, steps=rng.choice([1, 2]), learned=learned)
    else:
        n = log_int(rng, 20000, 4236960)
        c.update(tris=n, moving=log_int(rng, max(100, n // 500), n // 4))
    return c


# ---------------------------------------------------------------------------
# scenes
# ---------------------------------------------------------------------------

_SPHERES = {}


def unit_sphere(level):
    """Icosphere of 20 * 4^level triangles, wound outwards: (vertices f64, faces)."""
    if level not in _SPHERES:
        t = (1.0 + math.sqrt(5.0)) / 2.0
        v = np.array([[-1, t, 0], [1, t, 0], [-1, -t, 0], [1, -t, 0], [0, -1, t], [0, 1, t],
                      [0, -1, -t], [0, 1, -t], [t, 0, -1], [t, 0, 1], [-t, 0, -1], [-t, 0, 1]], np.float64)
        f = np.array([[0, 11, 5], [0, 5, 1], [0, 1, 7], [0, 7, 10], [0, 10, 11], [1, 5, 9], [5, 11, 4], [11, 10, 2],
                      [10, 7, 6], [7, 1, 8], [3, 9, 4], [3, 4, 2], [3, 2, 6], [3, 6, 8], [3, 8, 9], [4, 9, 5],
                      [2, 4, 11], [6, 2, 10], [8, 6, 7], [9, 8, 1]], np.int64)
        v /= np.linalg.norm(v, axis=1, keepdims=True)
        for _ in range(level):
            edges = np.sort(np.concatenate([f[:, [0, 1]], f[:, [1, 2]], f[:, [2, 0]]]), axis=1)
            u, inv = np.unique(edges, axis=0, return_inverse=True)
            mid = v[u[:, 0]] + v[u[:, 1]]
            mid /= np.linalg.norm(mid, axis=1, keepdims=True)
            a, b, c = (len(v) + inv.reshape(3, -1))
            f = np.concatenate([np.stack([f[:, 0], a, c], 1), np.stack([f[:, 1], b, a], 1),
                                np.stack([f[:, 2], c, b], 1), np.stack([a, b, c], 1)])
            v = np.concatenate([v, mid])
        _SPHERES[level] = (v, f)
    return _SPHERES[level]


def rand(g, *shape):
    return torch.rand(*shape, generator=g, dtype=torch.float64, device="cuda")


def soup(g, n, size=0.01):
    """n separate triangles with centres in the unit cube."""
    v = (rand(g, n, 1, 3) + (rand(g, n, 3, 3) * 2 - 1) * size).reshape(-1, 3)
    return v.float(), torch.arange(3 * n, dtype=torch.int32, device="cuda").reshape(-1, 3)


def field(g, gx, gz, amplitude=0.2):
    """Heightfield of gx x gz cells, two triangles each, from four octaves of smooth noise."""
    h = torch.zeros(gz + 1, gx + 1, dtype=torch.float64, device="cuda")
    for o in range(4):
        k = 4 << o
        lattice = rand(g, 1, 1, k + 1, k + 1)
        h += torch.nn.functional.interpolate(lattice, size=(gz + 1, gx + 1), mode="bilinear", align_corners=True)[0, 0] / (1 << o)
    x = torch.arange(gx + 1, dtype=torch.float64, device="cuda") / gx
    z = torch.arange(gz + 1, dtype=torch.float64, device="cuda") / gx
    v = torch.stack([x.expand(gz + 1, -1), h * (amplitude / 1.875), z[:, None].expand(-1, gx + 1)], 2)
    j, i = torch.meshgrid(torch.arange(gz, device="cuda"), torch.arange(gx, device="cuda"), indexing="ij")
    a = j * (gx + 1) + i
    f = torch.stack([a, a + gx + 1, a + 1, a + 1, a + gx + 1, a + gx + 2], 2)
    return v.reshape(-1, 3).float(), f.reshape(-1, 3).int()


def cluster_counts(n):
    """(spheres of each level 2..5, soup triangles) of a cluster scene of n triangles: about 88%
    of them on spheres, 60 / 25 / 12 / 3 of 100 spheres at the four levels."""
    mean = 0.60 * 320 + 0.25 * 1280 + 0.12 * 5120 + 0.03 * 20480
    spheres = int(0.88 * n / mean)
    levels = [int(spheres * w) for w in (0.60, 0.25, 0.12, 0.03)]
    return levels, n - sum(c * 20 * 4 ** (2 + i) for i, c in enumerate(levels))


def clusters(g, n):
    levels, loose = cluster_counts(n)
    vs, fs, base = [], [], 0
    for i, c in enumerate(levels):
        if c == 0:
            continue
        uv, uf = unit_sphere(2 + i)
        r = torch.exp(math.log(1e-3) + math.log(50.0) * rand(g, c, 1, 1))
        v = rand(g, c, 1, 3) + r * torch.from_numpy(uv).cuda()
        start = base + torch.arange(c, device="cuda") * len(uv)
        f = start[:, None, None] + torch.from_numpy(uf).cuda()
        vs.append(v.reshape(-1, 3).float())
        fs.append(f.reshape(-1, 3).int())
        base += c * len(uv)
    v, f = soup(g, loose)
    vs.append(v)
    fs.append(f + base)
    return torch.cat(vs), torch.cat(fs)


def generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 2654435761 % (1 << 62) + 1)


def mesh_of(case, seed):
    g = generator(seed)
    return field(g, case["gx"], case["gz"]) if case.get("scene") == "field" else clusters(g, case["tris"])


def counts_of(case):
    """(triangles, vertices) of a case's mesh."""
    if case.get("scene") == "field":
        return 2 * case["gx"] * case["gz"], (case["gx"] + 1) * (case["gz"] + 1)
    levels, loose = cluster_counts(case["tris"])
    return case["tris"], 3 * loose + sum(c * (10 * 4 ** (2 + i) + 2) for i, c in enumerate(levels))


def batch_sizes(case):
    """(kind, triangles-defining numbers) of every mesh of a batch, the same for every seed."""
    r = random.Random(case["sizes"])
    out = []
    for i in range(case["meshes"]):
        n = log_int(r, case["min"], case["max"])
        if i % 3 == 0:
            gx = max(2, int(math.sqrt(n / 2)))
            out.append({"scene": "field", "gx": gx, "gz": max(1, n // (2 * gx))})
        else:
            out.append({"scene": "clusters" if i % 3 == 1 else "soup", "tris": n})
    return out


def batch_counts(case):
    nf, nv = [], []
    for m in batch_sizes(case):
        f, v = (m["tris"], 3 * m["tris"]) if m["scene"] == "soup" else counts_of(m)
        nf.append(f)
        nv.append(v)
    return nf, nv


def batch_meshes(case, seed):
    g = generator(seed)
    return [soup(g, m["tris"]) if m["scene"] == "soup" else
            field(g, m["gx"], m["gz"]) if m["scene"] == "field" else clusters(g, m["tris"]) for m in batch_sizes(case)]


# ---------------------------------------------------------------------------
# the program's device objects
# ---------------------------------------------------------------------------

class Mesh:
    """A mesh in the program's own tensors."""

    def __init__(self, vert, faces):
        self.vert, self.faces = vert.contiguous(), faces.contiguous()
        self.num_faces, self.num_vert = len(faces), len(vert)
        self.raw = bt.MeshRaw(self.vert.data_ptr(), None, self.faces.data_ptr(), self.num_vert, 0, self.num_faces)


class Tree:
    """A tree of 2n - 1 nodes (48 bytes each) and its header, in the program's own tensors."""

    def __init__(self, num_faces):
        self.num_nodes = 2 * num_faces - 1
        self.nodes = torch.zeros(self.num_nodes, 12, dtype=torch.int32, device="cuda")
        self.header = torch.tensor([self.nodes.data_ptr(), self.num_nodes, self.num_nodes, 0], dtype=torch.int64,
                                   device="cuda")
        self.ptr = bt.CUDAMemoryBVHPointer(self.header.data_ptr(), self.nodes.data_ptr(), self.num_nodes)


def node_outputs(nodes):
    """A node array's boxes and areas as numbers, its links and flags as whole numbers."""
    f = nodes.view(torch.float32)
    return {"boxes": f[:, :6], "area": f[:, 11], "links": nodes[:, 6:11]}


def dev(t):
    return ctypes.c_void_p(t.data_ptr())


def done():
    """Raises what a call recorded as an error."""
    if bt.last_error():
        raise RuntimeError(bt.last_error())


def prepare(case, seed):
    lib = bt.lib()
    lib.bvht_setStream(torch.cuda.current_stream().cuda_stream)
    s = {"case": case, "lib": lib}
    kind = case["kind"]
    if kind == "batch":
        meshes = batch_meshes(case, seed)
        s["vert"] = torch.cat([v for v, _ in meshes])
        s["faces"] = torch.cat([f for _, f in meshes])
        nf = np.array([len(f) for _, f in meshes], np.uint32)
        nv = np.array([len(v) for v, _ in meshes], np.uint32)
        u32p = ctypes.POINTER(ctypes.c_uint32)
        s["mem"] = BatchMemory(lib.bvht_LBVH_allocateBatch(len(nf), nf.ctypes.data_as(u32p), nv.ctypes.data_as(u32p), 10))
        s["nodes"] = torch.zeros(s["mem"].raw.totalNodes, 12, dtype=torch.int32, device="cuda")
        return s
    if kind == "refit":
        return prepare_refit(case, seed, s)
    s["mesh"] = Mesh(*mesh_of(case, seed))
    s["builder"] = bt.LBVHBuilder(s["mesh"], case.get("bits", 63))
    s["tree"] = Tree(s["mesh"].num_faces)
    if kind in ("image", "frame"):
        s["builder"].build(s["tree"])
        torch.cuda.synchronize()
        s["builder"].free()
        n = case["w"] * case["h"]

        def words(k):
            return torch.zeros(n, k, dtype=torch.int32, device="cuda")

        s.update(rays=words(12), img=words(1), hits=words(2))
        if kind == "frame":
            s.update(brays=words(12), skip=words(1), bhits=words(2))
        cam = CAM_FIELD if case["scene"] == "field" else CAM
        s["cam"] = (case["w"], case["h"], bt.vec3(cam["pos"]), bt.vec3(cam["look_at"]), bt.vec3((0.0, 1.0, 0.0)), 45.0)
    if kind == "optimise":
        s["builder"].build(s["tree"])
        s["opt"] = bt.Bittner13GPU(numChunks=case["chunks"], batchPercent=case["percent"],
                                   priority=1 if case["learned"] else 0)
        s["opt"].setup(s["tree"], s["mesh"].num_faces)
        if case["learned"]:
            s["model"] = bt.PriorityModel.load(os.path.join(HERE, "bvhtest_amd", "data", "priority_mlp.npy"))
            s["opt"].set_model(s["model"])
    done()
    return s


class BatchMemory:
    """The batch's working memory, released with the object."""

    def __init__(self, raw):
        if not raw.lRes:
            raise RuntimeError(bt.last_error())
        self.raw = raw

    def __del__(self):
        bt.lib().bvht_LBVH_freeBatch(ctypes.byref(self.raw))


def moving_mesh(case, seed):
    """(vertices, faces, vertices after the move): a cluster scene whose last `moving` triangles are
    loose ones that move."""
    g = generator(seed)
    v, f = clusters(g, case["tris"] - case["moving"])
    dv, df = soup(g, case["moving"])
    shift = torch.sin(dv.double() * 7.0 + rand(g, 3) * 6.0) * 0.02
    return torch.cat([v, dv]), torch.cat([f, df + len(v)]), torch.cat([v, (dv + shift).float()])


def prepare_refit(case, seed, s):
    v, f, moved = moving_mesh(case, seed)
    s["mesh"] = Mesh(v, f)
    s["tree"] = Tree(len(f))
    b = bt.LBVHBuilder(s["mesh"], 30)
    b.build(s["tree"])
    torch.cuda.synchronize()
    b.free()
    s["opt"] = bt.Bittner13GPU(numChunks=1)
    s["opt"].setup(s["tree"], len(f))
    s["leaves"] = torch.zeros(len(f), dtype=torch.int32, device="cuda")
    num = ctypes.c_uint32()
    s["lib"].selectDynamicLeafNodes(ctypes.byref(s["opt"].mem), ctypes.byref(s["tree"].ptr), dev(s["leaves"]),
                                    ctypes.byref(num), len(f) - case["moving"])
    done()
    s["num"] = num.value
    s["mesh"].vert.copy_(moved)
    return s


def run(s):
    case, lib = s["case"], s["lib"]
    kind = case["kind"]
    if kind == "build":
        s["builder"].build(s["tree"])
        return node_outputs(s["tree"].nodes)
    if kind == "batch":
        if not lib.bvht_LBVH_buildBatch(ctypes.byref(s["mem"].raw), dev(s["vert"]), dev(s["faces"]), dev(s["nodes"]), True):
            raise RuntimeError(bt.last_error())
        return node_outputs(s["nodes"])
    tree, mesh = s["tree"], s["mesh"]
    if kind == "image":
        lib.generateRays(dev(s["rays"]), *s["cam"])
        lib.tracerImage(dev(s["rays"]), dev(s["img"]), dev(tree.nodes), 0, mesh.raw, bt.vec3(LIGHT), case["w"], case["h"],
                        case["bundle"])
        done()
        return {"image": s["img"], "rays": s["rays"].view(torch.float32)[:, :9]}
    if kind == "frame":
        n = case["w"] * case["h"]
        light = bt.vec3(LIGHT)
        lib.generateRays(dev(s["rays"]), *s["cam"])
        lib.bvht_traceRays(dev(s["rays"]), n, dev(tree.nodes), 0, mesh.raw, light, 0, 0.0, None, dev(s["hits"]), dev(s["img"]))
        lib.bvht_makeBounceRays(dev(s["rays"]), dev(s["hits"]), n, mesh.raw, 1, dev(s["brays"]), dev(s["skip"]))
        lib.bvht_traceRays(dev(s["brays"]), n, dev(tree.nodes), 0, mesh.raw, light, 1, 0.0, dev(s["skip"]), dev(s["bhits"]), None)
        done()
        out = {"image": s["img"], "rays": s["brays"].view(torch.float32)[:, :9]}
        for k in ("hits", "bhits"):
            out[k] = {"triangle": s[k][:, 0], "t": s[k].view(torch.float32)[:, 1]}
        return out
    if kind == "optimise":
        opt = s["opt"]
        s["builder"].build(tree)
        lib.initData(ctypes.byref(opt.mem), ctypes.byref(tree.ptr), 128)
        for _ in range(case["steps"]):
            opt.step(tree)
        return {"tree": node_outputs(tree.nodes), "sah": bt.calc_sah(tree, 1.2, 1.0)}
    lib.refitDynamicTris(ctypes.byref(tree.ptr), mesh.raw, dev(s["leaves"]), s["num"], 64)
    if not lib.bvht_fixTreeFrom(ctypes.byref(s["opt"].mem), ctypes.byref(tree.ptr), dev(s["leaves"]), s["num"]):
        raise RuntimeError(bt.last_error())
    return node_outputs(tree.nodes)


# ---------------------------------------------------------------------------
# work and exact values
# ---------------------------------------------------------------------------

def work(case):
    """Mesh and nodes once each for a build; for a trace the tree, the mesh, the rays and the
    results once, and two box tests (24 operations each) at every level of a balanced tree for each
    ray; for an optimizer step one read of the nodes and of each chosen patch's ten nodes (read and written);
    for a refit the moving triangles and two nodes read and written for each of their leaves."""
    kind = case["kind"]
    if kind == "batch":
        nf, nv = batch_counts(case)
        return {"bytes": 12 * sum(nf) + 12 * sum(nv) + 48 * (2 * sum(nf) - len(nf)), "flops": 60 * sum(nf)}
    if kind == "refit":
        return {"bytes": case["moving"] * (4 + 12 + 36 + 2 * 2 * 48), "flops": 40 * case["moving"]}
    n, nv = counts_of(case)
    mesh, nodes = 12 * n + 12 * nv, 48 * (2 * n - 1)
    if kind == "build":
        return {"bytes": mesh + nodes, "flops": 60 * n}
    if kind in ("image", "frame"):
        rays = case["w"] * case["h"]
        tests = 2 * 24 * math.log2(2 * n)
        if kind == "image":
            return {"bytes": mesh + nodes + (48 + 4) * rays, "flops": tests * rays}
        return {"bytes": mesh + nodes + (48 + 8 + 4 + 48 + 4 + 8) * rays, "flops": 2 * tests * rays}
    patches = int(case["percent"] / 100.0 * 2 * n)
    return {"bytes": mesh + nodes + case["steps"] * (nodes + patches * 10 * 2 * 48),
            "flops": 60 * n + case["steps"] * (20 * n + (9856 * n if case["learned"] else 0))}


def spread(x, bits):
    """Bit b of x to bit 3b."""
    out = np.zeros(x.shape, np.uint64)
    for b in range(bits):
        out |= ((x >> np.uint64(b)) & np.uint64(1)) << np.uint64(3 * b)
    return out


def sorted_faces(v, f, bits):
    """The order of the triangles by their Morton code: the codes' arithmetic is in 32 bits by
    definition, so the order is the same whole numbers everywhere."""
    p = v[f]
    eps, three = np.float32(FLT_EPSILON), np.float32(3.0)
    lo = np.minimum(np.float32(0.0), p.min((0, 1)) - eps)
    hi = np.maximum(np.float32(0.0), p.max((0, 1)) + eps)
    c = ((p[:, 0] + p[:, 1]) + p[:, 2]) / three
    off = np.float32(0.0) - lo
    scale = np.float32(1.0) / (hi + off)
    q = 10 if bits == 30 else 21
    cells = np.clip(((c + off) * scale) * np.float32(1 << q), np.float32(0.0), np.float32((1 << q) - 1)).astype(np.uint64)
    x, y, z = (spread(cells[:, k], q) for k in range(3))
    return np.argsort((x << np.uint64(2)) | (y << np.uint64(1)) | z, kind="stable")


def area_of(b):
    d = b[:, 3:] - b[:, :3]
    return 2.0 * (d[:, 0] * d[:, 1] + d[:, 0] * d[:, 2] + d[:, 1] * d[:, 2])


def exact_tree(v, f, bits, moved=None):
    """Boxes and areas in 64 bits of the nodes of the index topology: leaf p at n - 1 + p; the inner
    node at an odd index p ends the aligned block that ends there, at an even one starts the block that
    starts there, and 0 is the root.  `moved`: the vertices of a later refit, which keeps the leaves' areas."""
    order = sorted_faces(v, f, bits)

    def leaves(vert):
        p = vert[f[order]].astype(np.float64)
        return np.concatenate([p.min(1) - FLT_EPSILON, p.max(1) + FLT_EPSILON], 1)

    n = len(f)
    boxes = np.empty((2 * n - 1, 6))
    leaf = leaves(v if moved is None else moved)
    boxes[n - 1:] = leaf
    idx = np.arange(n - 1, dtype=np.int64)
    edge = np.where(idx & 1, idx + 1, idx)
    level, cur = 0, leaf
    while len(cur) > 1:
        if len(cur) & 1:
            cur = np.concatenate([cur, [[np.inf] * 3 + [-np.inf] * 3]])
        cur = np.concatenate([np.minimum(cur[0::2, :3], cur[1::2, :3]), np.maximum(cur[0::2, 3:], cur[1::2, 3:])], 1)
        level += 1
        at = idx[(edge & ((2 << level) - 1)) == (1 << level)]
        boxes[at] = cur[at >> level]
    boxes[0] = cur[0]
    area = area_of(boxes)
    if moved is not None:
        area[n - 1:] = area_of(leaves(v))
    return {"boxes": boxes, "area": area, "links": None}


def exact_rays(case):
    """Camera rays in 64 bits: position, direction, inverse direction."""
    cam = CAM_FIELD if case["scene"] == "field" else CAM
    pos, look = np.array(cam["pos"], np.float32).astype(np.float64), np.array(cam["look_at"], np.float32).astype(np.float64)
    f = (look - pos) / np.linalg.norm(look - pos)
    r = np.cross(f, [0.0, 1.0, 0.0])
    r /= np.linalg.norm(r)
    u = np.cross(r, f)
    scale, ratio = math.tan(math.radians(22.5)), case["w"] / case["h"]
    x = (2 * (np.arange(case["w"]) + 0.5) / case["w"] - 1) * scale * ratio
    y = (1 - 2 * (np.arange(case["h"]) + 0.5) / case["h"]) * scale
    d = x[None, :, None] * r + y[:, None, None] * u + f
    d /= np.linalg.norm(d, axis=2, keepdims=True)
    d = d.reshape(-1, 3)
    with np.errstate(divide="ignore"):
        return np.concatenate([np.broadcast_to(pos, d.shape), d, 1.0 / d], 1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "build":
        if counts_of(case)[0] > 5000000:  # the sort and the tree take too long on one CPU core
            return None
        v, f = mesh_of(case, seed)
        return exact_tree(v.cpu().numpy(), f.cpu().numpy(), case["bits"])
    if kind == "refit":
        v, f, moved = moving_mesh(case, seed)
        return exact_tree(v.cpu().numpy(), f.cpu().numpy(), 30, moved.cpu().numpy())
    if kind == "batch":
        if sum(batch_counts(case)[0]) > 4000000:
            return None
        trees = [exact_tree(v.cpu().numpy(), f.cpu().numpy(), 30) for v, f in batch_meshes(case, seed)]
        return {"boxes": np.concatenate([t["boxes"] for t in trees]), "area": np.concatenate([t["area"] for t in trees]),
                "links": None}
    if kind == "image":
        return {"image": None, "rays": exact_rays(case)}
    # traced distances and optimised trees follow from discrete choices made in 32 bits
    return None
