"""The work that users of this framework have it do each frame, as cases that can be timed.

Every case goes through the C ABI (include/cadr_hip.h) or the Python driver over it, on scenes that stay
in device memory, as a renderer's loop does: the descriptors, tiles, workspaces and plans are made once,
then each pass is the frame's calls on the default stream.  Matrices, spheres, mesh tables and handle
tables are made with torch from the seed alone.  The kinds:

  view       one camera over resident world spheres (cadrCullView)
  flat       a scene without a hierarchy whose world matrices a simulation wrote: world spheres, then
             one camera (cadrComputeWorldSpheres + cadrCullView)
  frame      a transform tree and one camera: the inner levels, then the leaf level fused with the cull
             (cadrPropagateTransformsBatch + cadrPropagateCullView)
  levels     a transform tree, level by level, then a few cameras (shadow cascades, cube faces, stereo):
             cadrPropagateTransforms per level, the last with world spheres, + cadrCullBatch
  views      many cameras over one resident scene (cadrCullBatch, one job)
  scenes     many transform trees of uneven size, depth and camera count in one frame: one propagation
             launch per inner depth, then cadrPropagateCullBatch over all scenes
  served     what one batch of a view server holds: scenes of uneven size, a few cameras each, in one
             cadrCullBatch
  gather     the reference's own pass: handles of every drawable resolved into commands and pointers,
             after the records edited since the last frame were sent (cadrScatterDrawables +
             cadrProcessDrawables)
  instances  the facade's cull frame: instanced MatrixLists written by a transform plan, then gather,
             mesh table, cull items, cull of one camera and the draw contract
"""
from __future__ import annotations

import ctypes
import math
import random

import numpy as np
import torch

from cadr_amd import _native as N
from cadr_amd import cull, scenes

DEV = "cuda"
INF = float("inf")

# ---------------------------------------------------------------------------------------------- cases


def listed():
    return [
        # the smallest scene of the repository's workloads, one camera, one StateSet: latency
        {"name": "view_100k", "kind": "view", "drawables": 100_000, "statesets": 1, "meshes": 64, "lods": 1,
         "block": 256, "items": 4},
        # the headline scene's drawables and StateSets with their spheres resident (a still scene, a moving camera)
        {"name": "view_10m", "kind": "view", "drawables": 10_000_000, "statesets": 64, "meshes": 64, "lods": 3,
         "block": 1024, "items": 8},
        # a flat scene of odd size, few StateSets, the driver's default shape
        {"name": "flat_1m", "kind": "flat", "drawables": 1_234_567, "statesets": 7, "meshes": 64, "lods": 2,
         "block": 256, "items": 4},
        # the headline workload: 1000 x 100 x 100 nodes, 10M drawables, one camera, the shape the autotuner picks
        {"name": "frame_10m", "kind": "frame", "drawables": 10_000_000, "depth": 3, "roots": 1000, "statesets": 64,
         "meshes": 64, "lods": 3, "block": 512, "items": 4},
        # a small deep tree, odd sizes, the driver's default shape: a frame of launches
        {"name": "frame_40k", "kind": "frame", "drawables": 40_961, "depth": 4, "roots": 33, "statesets": 12,
         "meshes": 48, "lods": 4, "block": 256, "items": 4},
        # a middle-sized tree and six cameras, levels propagated one by one
        {"name": "levels_2m", "kind": "levels", "drawables": 2_000_000, "depth": 3, "roots": 500, "statesets": 64,
         "meshes": 64, "lods": 3, "views": 6, "block": 256, "items": 4},
        # many cameras over one scene, as the 256-view workload has them, at a quarter of its drawables (its
        # 51 GB of commands would not fit the card three times)
        {"name": "views_256", "kind": "views", "drawables": 2_500_000, "statesets": 64, "meshes": 64, "lods": 3,
         "views": 256, "block": 256, "items": 8},
        # a few dozen cameras, odd counts, a mesh table too large for one small copy of it
        {"name": "views_37", "kind": "views", "drawables": 333_337, "statesets": 9, "meshes": 150, "lods": 4,
         "views": 37, "block": 256, "items": 8},
        # the uneven multi-scene workload: 64 trees, log-uniform sizes, 1-32 cameras each
        {"name": "scenes_64", "kind": "scenes", "scenes": 64, "smallest": 10_000, "largest": 2_000_000,
         "max_views": 32, "statesets": 64, "meshes": 64, "layout": 3, "block": 256, "items": 8},
        # a server's batch at a moderate load: 24 scenes, one or two cameras each, the server's default shape
        {"name": "served_24", "kind": "served", "scenes": 24, "smallest": 10_000, "largest": 4_000_000,
         "max_views": 2, "statesets": 64, "meshes": 64, "layout": 4, "block": 256, "items": 4},
        # the reference's pass at full size, handle level 3, one drawable in a thousand edited
        {"name": "gather_10m", "kind": "gather", "drawables": 10_000_000, "statesets": 1, "level": 3,
         "geometries": 64},
        # the facade's frame: 5M instances in 4096 MatrixLists over a 50k-node inner level
        {"name": "instances_5m", "kind": "instances", "drawables": 4096, "instances": 5_000_000, "nodes": 50_000,
         "statesets": 64, "meshes": 64, "lods": 3, "block": 1024, "items": 8},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(["view", "view", "flat", "frame", "frame", "levels", "views", "scenes", "served", "gather",
                       "instances"])
    K = rng.choice([1, 2, 5, 13, 64, 64, 200])
    # a view of more drawables takes larger tiles, as the autotuner finds
    shapes1 = lambda n: rng.choice([(256, 4), (512, 4), (1024, 8)] if n > 400_000 else [(256, 4), (256, 2), (512, 4)])  # noqa: E731
    common = {"kind": kind, "statesets": K, "meshes": rng.choice([1, 17, 64, 64, 300]), "lods": rng.randint(1, 4)}
    if kind in ("view", "flat"):
        n = _log(rng, 2_000, 10_000_000 if kind == "view" else 5_000_000)
        b, i = shapes1(n)
        return {**common, "drawables": n, "block": b, "items": i}
    if kind in ("frame", "levels"):
        n = _log(rng, 2_000, 8_000_000 if kind == "frame" else 3_000_000)
        depth = rng.randint(2, 4)
        c = {**common, "drawables": n, "depth": depth, "roots": _log(rng, 1, max(2, min(1000, n // 8)))}
        if kind == "levels":
            c["views"] = rng.randint(1, 8)
        b, i = rng.choice([(256, 4), (512, 4), (256, 8)])
        return {**c, "block": b, "items": i}
    if kind == "views":
        v = _log(rng, 2, 256)
        b, i = rng.choice([(256, 4), (512, 4), (256, 8)])
        return {**common, "drawables": _log(rng, 10_000, min(4_000_000, 600_000_000 // v)), "views": v, "block": b,
                "items": i}
    if kind in ("scenes", "served"):
        b, i = rng.choice([(256, 4), (512, 4), (256, 8)])
        return {"kind": kind, "scenes": rng.randint(2, 48), "smallest": 5_000,
                "largest": _log(rng, 50_000, 2_000_000), "max_views": rng.randint(1, 16) if kind == "scenes" else
                rng.randint(1, 4), "statesets": K, "meshes": 64, "layout": rng.randrange(1 << 20), "block": b, "items": i}
    if kind == "gather":
        n = _log(rng, 1_000, 8_000_000)
        return {"kind": kind, "drawables": n, "statesets": K, "level": 3 if n > 1_000_000 else rng.choice([2, 3]),
                "geometries": rng.choice([16, 64, 300])}
    n = _log(rng, 20_000, 4_000_000)
    b, i = shapes1(n)
    return {**common, "drawables": min(_log(rng, 8, 4096), n // 8), "instances": n, "nodes": _log(rng, 100, 80_000),
            "block": b, "items": i}


# --------------------------------------------------------------------------------------------- inputs


def _rng(seed, stream):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1_000_003 + stream) & 0x7FFFFFFFFFFFFFFF)
    return g


def _uniform(g, n, comps=1):
    return torch.rand((n, comps), generator=g, device=DEV, dtype=torch.float32)


def rotation_translation(g, n, span=50.0):
    """n column-major float mat4: a uniform random rotation and a translation U[-span, span]^3."""
    u = _uniform(g, n, 6)
    a, b = torch.sqrt(1.0 - u[:, 0]), torch.sqrt(u[:, 0])
    x, y = a * torch.sin(2 * math.pi * u[:, 1]), a * torch.cos(2 * math.pi * u[:, 1])
    z, w = b * torch.sin(2 * math.pi * u[:, 2]), b * torch.cos(2 * math.pi * u[:, 2])
    m = torch.zeros((n, 16), device=DEV, dtype=torch.float32)
    m[:, 0], m[:, 1], m[:, 2] = 1 - 2 * (y * y + z * z), 2 * (x * y + z * w), 2 * (x * z - y * w)
    m[:, 4], m[:, 5], m[:, 6] = 2 * (x * y - z * w), 1 - 2 * (x * x + z * z), 2 * (y * z + x * w)
    m[:, 8], m[:, 9], m[:, 10] = 2 * (x * z + y * w), 2 * (y * z - x * w), 1 - 2 * (x * x + y * y)
    m[:, 12:15] = span * (2 * u[:, 3:6] - 1)
    m[:, 15] = 1.0
    return m


def scale_translation(g, n, span=500.0):
    """n column-major float mat4: a uniform scale exp(U[ln 0.1, ln 2]) and a translation U[-span, span]^3."""
    u = _uniform(g, n, 4)
    m = torch.zeros((n, 16), device=DEV, dtype=torch.float32)
    m[:, 0] = m[:, 5] = m[:, 10] = torch.exp(math.log(0.1) + u[:, 0] * math.log(20.0))
    m[:, 12:15] = span * (2 * u[:, 1:4] - 1)
    m[:, 15] = 1.0
    return m


def mesh_table(seed, count, lods):
    """cadrMesh[count] on the host: centres within half a unit, radius U[0.5, 2.5), `lods` LODs of falling size."""
    r = np.random.RandomState((int(seed) * 7919 + 17) & 0x7FFFFFFF)
    m = np.zeros(count, N.MESH_DTYPE)
    m["center"] = r.uniform(-0.5, 0.5, (count, 3)).astype(np.float32)
    m["radius"] = r.uniform(0.5, 2.5, count).astype(np.float32)
    m["lodCount"] = lods
    m["vertexOffset"] = r.randint(0, 1 << 20, count)
    size = r.randint(36, 3001, count)
    first = 0
    for k in range(lods):
        m["indexCount"][:, k] = np.maximum(12, (size >> (2 * k)) // 3 * 3)
        m["firstIndex"][:, k] = first + np.concatenate([[0], np.cumsum(m["indexCount"][:-1, k])])
        first += int(m["indexCount"][:, k].sum())
    return m


def to_device(a: np.ndarray) -> torch.Tensor:
    """The bytes of a numpy array in device memory."""
    return torch.from_numpy(np.frombuffer(np.ascontiguousarray(a).tobytes(), np.uint8).copy()).to(DEV)


def statesets_of(g, n, K):
    """Drawable order (grouped by StateSet, each drawable's StateSet random) and the StateSets' sizes."""
    if K == 1:
        return torch.arange(n, device=DEV), np.array([n], np.uint32)
    ss = torch.randint(0, K, (n,), generator=g, device=DEV)
    counts = torch.bincount(ss, minlength=K).cpu().numpy().astype(np.uint32)
    return torch.sort(ss, stable=True).indices, counts


def level_sizes(leaves, depth, roots):
    """Nodes per level of a tree with `roots` roots and an equal fan-out below them."""
    f = max(1.0, (leaves / roots) ** (1.0 / (depth - 1))) if depth > 1 else 1.0
    sizes = [min(leaves, max(1, int(round(roots * f ** d)))) for d in range(depth - 1)] + [leaves]
    return [int(s) for s in sizes]


def tree_inputs(seed, stream, sizes, K):
    """[(local matrices, parent indices or None)] per level; the leaves in StateSet order."""
    out, order, counts = [], None, np.array([sizes[-1]], np.uint32)
    for d, n in enumerate(sizes):
        g = _rng(seed, stream + d)
        last = d == len(sizes) - 1
        if last:
            order, counts = statesets_of(_rng(seed, stream + 90), n, K)
        parent = None
        if d > 0:
            node = order if last else torch.arange(n, device=DEV)
            parent = (node * sizes[d - 1] // n).to(torch.int32)
        out.append((rotation_translation(g, n), parent))
    return out, counts


def cameras(seed, count, box):
    """cadrView[count]: eyes in a box, random directions, vertical fields of view of 40 to 90 degrees."""
    return cull.make_views(scenes.random_cameras(int(seed) & 0xFFFFFFFF, 20, 0, count, box))


class Memory:
    """A torch tensor where the driver's classes take a device buffer."""

    def __init__(self, t):
        self.tensor, self.address = t, t.data_ptr()

    def close(self):
        pass


class Outputs:
    """Commands and counts of a cull job, zeroed (slots past a count are never written)."""

    def __init__(self, views, stride, K):
        self.stride = stride
        self.cmd = torch.zeros((views * stride, 5), device=DEV, dtype=torch.int32)
        self.cnt = torch.zeros((views, K), device=DEV, dtype=torch.int32)
        self.commands, self.counts = Memory(self.cmd), Memory(self.cnt)


class SceneInMemory:
    """What a cull job reads: spheres, mesh indices, mesh table, tiles."""

    def __init__(self, n, counts, meshes, mesh_index, spheres):
        self.n, self.K, self.stateset_counts, self.num_meshes = n, len(counts), counts, len(meshes)
        self.host_meshes = meshes
        self.meshes, self.mesh_index, self.spheres = Memory(to_device(meshes)), Memory(mesh_index), Memory(spheres)
        self._tiles = {}

    def tiles(self, tile):
        if tile not in self._tiles:
            t = cull.build_tiles(self.stateset_counts, tile)
            self._tiles[tile] = (Memory(to_device(t)), len(t))
        return self._tiles[tile]


def flat_spheres(world, meshes, mesh_index):
    """World spheres under a scale and a translation, in torch."""
    m = torch.from_numpy(np.concatenate([meshes["center"], meshes["radius"][:, None]], 1)).to(DEV)[mesh_index.long()]
    s = m * world[:, :1]
    s[:, :3] += world[:, 12:15]
    return s.contiguous()


def mesh_indices(seed, stream, n, count):
    return torch.randint(0, count, (n,), generator=_rng(seed, stream), device=DEV, dtype=torch.int32)


def level_desc(local, world, n, parent=None, parent_world=None, parent_count=0):
    lv = np.zeros(1, N.LEVEL_DTYPE)
    lv["localMatrices"], lv["worldMatrices"], lv["count"] = local.data_ptr(), world.data_ptr(), n
    if parent is not None:
        lv["parentIndex"], lv["parentWorld"], lv["parentCount"] = parent.data_ptr(), parent_world.data_ptr(), parent_count
    return lv


class State:
    def __init__(self, **kw):
        self.__dict__.update(kw)


# ---------------------------------------------------------------------------------- prepare, per kind


def _config(case):
    return cull.make_config(case["block"], case["items"])


def prepare_view(case, seed):
    n, K = case["drawables"], case["statesets"]
    meshes = mesh_table(seed, case["meshes"], case["lods"])
    mi = mesh_indices(seed, 3, n, len(meshes))
    counts = statesets_of(_rng(seed, 5), n, K)[1]
    world = scale_translation(_rng(seed, 4), n)
    flat = case["kind"] == "flat"
    spheres = torch.zeros((n, 4), device=DEV) if flat else flat_spheres(world, meshes, mi)
    ds = SceneInMemory(n, counts, meshes, mi, spheres)
    out = Outputs(1, n, K)
    batch = cull.CullBatch(_config(case), [(ds, cameras(seed, 1, 100.0), out)])
    return State(kind=case["kind"], ds=ds, world=world if flat else None, out=out, batch=batch, spheres=spheres)


def run_view(s):
    s.batch.run_view()
    return {"commands": s.out.cmd, "counts": s.out.cnt}


def run_flat(s):
    ds = s.ds
    N.check(N.load().cadrComputeWorldSpheres(s.world.data_ptr(), ds.mesh_index.address, ds.meshes.address,
                                             ds.num_meshes, ds.n, ds.spheres.address, None))
    s.batch.run_view()
    return {"spheres": s.spheres, "commands": s.out.cmd, "counts": s.out.cnt}


def tree_levels(inputs):
    """World arrays and descriptors of a tree's levels, root first.  A root's world matrices are its local
    ones, so the level below reads those and shares the root level's launch."""
    worlds, descs = [], []
    for d, (local, parent) in enumerate(inputs):
        n = len(local)
        world = torch.zeros((n, 16), device=DEV)
        if d == 0:
            descs.append(level_desc(local, world, n))
        else:
            above = inputs[0][0] if d == 1 else worlds[d - 1]
            descs.append(level_desc(local, world, n, parent, above, len(above)))
        worlds.append(world)
    return worlds, descs


def prepare_frame(case, seed):
    sizes = level_sizes(case["drawables"], case["depth"], case["roots"])
    inputs, counts = tree_inputs(seed, 10, sizes, case["statesets"])
    meshes = mesh_table(seed, case["meshes"], case["lods"])
    n = sizes[-1]
    mi = mesh_indices(seed, 3, n, len(meshes))
    levels = case["kind"] == "levels"
    spheres = torch.zeros((n if levels else 1, 4), device=DEV)
    ds = SceneInMemory(n, counts, meshes, mi, spheres)
    worlds, descs = tree_levels(inputs)
    V = case["views"] if levels else 1
    out = Outputs(V, n, len(counts))
    batch = cull.CullBatch(_config(case), [(ds, cameras(seed, V, 100.0), out)])
    s = State(kind=case["kind"], inputs=inputs, worlds=worlds, ds=ds, out=out, batch=batch, spheres=spheres, descs=descs)
    if levels:
        lv = descs[-1]
        lv["meshIndex"], lv["meshes"], lv["numMeshes"], lv["spheres"] = (mi.data_ptr(), ds.meshes.address,
                                                                         len(meshes), spheres.data_ptr())
    else:
        s.launches = depth_launches([descs[:-1]])
    return s


def depth_launches(trees):
    """Propagation launches over many trees' inner levels: the roots together with the level below them, then
    one launch per depth.  [(device descriptors, host descriptors)]"""
    deepest = max(len(t) for t in trees)
    groups = [[lv for t in trees for lv in t[:2]]] + [[t[d] for t in trees if d < len(t)] for d in range(2, deepest)]
    out = []
    for g in groups:
        if g:
            host = np.concatenate(g)
            out.append((to_device(host), host))
    return out


def run_frame(s):
    lib = N.load()
    for dev, host in s.launches:
        N.check(lib.cadrPropagateTransformsBatch(dev.data_ptr(), N.ptr(host), len(host), None))
    s.batch.run_fused(s.descs[-1])
    return {"worlds": s.worlds, "commands": s.out.cmd, "counts": s.out.cnt}


def run_levels(s):
    lib = N.load()
    for lv in s.descs:
        N.check(lib.cadrPropagateTransforms(N.ptr(lv), None))
    s.batch.run()
    return {"worlds": s.worlds, "spheres": s.spheres, "commands": s.out.cmd, "counts": s.out.cnt}


def prepare_views(case, seed):
    n, K, V = case["drawables"], case["statesets"], case["views"]
    meshes = mesh_table(seed, case["meshes"], case["lods"])
    mi = mesh_indices(seed, 3, n, len(meshes))
    # the drawables of a two-level tree, StateSet by StateSet in tree order: a tile holds neighbours
    sizes = [max(1, n // 10_000), max(1, n // 100), n]
    inputs, counts = tree_inputs(seed, 10, sizes, K)
    pos = [m[:, 12:15] for m, _ in inputs]
    at = pos[2] + pos[1][inputs[2][1].long()] + pos[0][inputs[1][1].long()][inputs[2][1].long()]
    radius = torch.from_numpy(meshes["radius"]).to(DEV)[mi.long()]
    spheres = torch.cat([at, radius[:, None]], 1).contiguous()
    ds = SceneInMemory(n, counts, meshes, mi, spheres)
    out = Outputs(V, n, len(counts))
    batch = cull.CullBatch(_config(case), [(ds, cameras(seed, V, 600.0), out)])
    return State(kind="views", ds=ds, out=out, batch=batch)


def run_views(s):
    s.batch.run()
    return {"commands": s.out.cmd, "counts": s.out.cnt}


def layout(case):
    """(drawables, depth, lods, cameras) per scene: the case's own, whatever the seed."""
    r = random.Random(case["layout"])
    got = []
    for _ in range(case["scenes"]):
        n = _log(r, case["smallest"], case["largest"])
        got.append((n, r.randint(1, 4), r.randint(1, 4), r.randint(1, case["max_views"])))
    return got


def prepare_scenes(case, seed):
    K, M = case["statesets"], case["meshes"]
    specs = layout(case)
    trees = case["kind"] == "scenes"
    # one allocation per kind of output, a part of it per scene (16-byte steps)
    commands = torch.zeros((sum(n * v for n, _, _, v in specs), 5), device=DEV, dtype=torch.int32)
    counts_all = torch.zeros((sum(v for *_, v in specs), K), device=DEV, dtype=torch.int32)
    total = sum(n for n, *_ in specs)
    worlds_all = torch.zeros((total, 16), device=DEV) if trees else None
    entries, inner, leaves, keep = [], [], [], []
    at_cmd = at_cnt = at_leaf = 0
    for i, (n, depth, lods, V) in enumerate(specs):
        meshes = mesh_table(seed + 31 * i, M, lods)
        mi = mesh_indices(seed, 1000 * i + 3, n, M)
        if trees:
            f = max(1, math.ceil(n ** (1.0 / depth) - 1e-9))
            sizes = [n]
            for _ in range(depth - 1):
                sizes.append(-(-sizes[-1] // f))
            inputs, counts = tree_inputs(seed, 1000 * i + 10, sizes[::-1], K)
            spheres = torch.zeros((1, 4), device=DEV)
            worlds, descs = tree_levels(inputs[:-1])
            world = worlds_all[at_leaf:at_leaf + n]
            local, parent = inputs[-1]
            if depth == 1:
                leaf = level_desc(local, world, n)
            else:
                above = inputs[0][0] if depth == 2 else worlds[-1]
                leaf = level_desc(local, world, n, parent, above, len(above))
            inner.append(descs)
            leaves.append(leaf)
            keep.append((inputs, worlds))
        else:
            counts = statesets_of(_rng(seed, 1000 * i + 5), n, K)[1]
            spheres = flat_spheres(scale_translation(_rng(seed, 1000 * i + 4), n), meshes, mi)
        ds = SceneInMemory(n, counts, meshes, mi, spheres)
        out = State(stride=n, commands=Memory(commands[at_cmd:at_cmd + n * V]), counts=Memory(counts_all[at_cnt:at_cnt + V]))
        entries.append((ds, cameras(seed + 77 * i, V, 200.0), out))
        at_cmd, at_cnt, at_leaf = at_cmd + n * V, at_cnt + V, at_leaf + n
    batch = cull.CullBatch(_config(case), entries)
    s = State(kind=case["kind"], batch=batch, entries=entries, keep=keep, commands=commands, counts=counts_all,
              worlds=worlds_all)
    if trees:
        s.launches = depth_launches(inner) if any(inner) else []
        batch.set_leaves(np.concatenate(leaves))
    return s


def run_scenes(s):
    lib = N.load()
    for dev, host in s.launches:
        N.check(lib.cadrPropagateTransformsBatch(dev.data_ptr(), N.ptr(host), len(host), None))
    s.batch.run_fused_batch()
    return {"worlds": s.worlds, "commands": s.commands, "counts": s.counts}


def run_served(s):
    s.batch.run()
    return {"commands": s.commands, "counts": s.counts}


REGION = 1 << 32


def region(nbytes):
    """Device memory at a 4-GiB boundary: the low half of every address in it is the same wherever it lies."""
    whole = torch.empty(nbytes + REGION, device=DEV, dtype=torch.uint8)
    skip = -whole.data_ptr() % REGION
    part = whole[skip:skip + nbytes]
    part.zero_()
    return part


def handle_tables(mem, at, level, first, addresses):
    """Writes the tables that resolve handles first, first + 1, ... to `addresses` (int64) at offset `at` of mem,
    root table first; returns the offset behind them."""
    T = 2048
    base, hmax = mem.data_ptr(), first + len(addresses) - 1
    words = mem.view(torch.int64)
    lo, hi = first // T, hmax // T
    root, at = at, at + 8 * T
    if level == 3:
        mlo, mhi = lo // T, hi // T
        mid, at = at, at + 8 * T * (mhi - mlo + 1)
    leaf, at = at, at + 8 * T * (hi - lo + 1)
    words[leaf // 8 + first - lo * T:leaf // 8 + hmax - lo * T + 1] = addresses
    where = base + leaf + 8 * T * torch.arange(hi - lo + 1, device=DEV)
    if level == 2:
        words[root // 8 + lo:root // 8 + hi + 1] = where
    else:
        words[mid // 8 + lo - mlo * T:mid // 8 + hi - mlo * T + 1] = where
        words[root // 8 + mlo:root // 8 + mhi + 1] = base + mid + 8 * T * torch.arange(mhi - mlo + 1, device=DEV)
    return at


# vertex, index and shader data, which the pass hands on and never reads, lie at addresses of their own
FAR_DATA = 0x6A0000000000


def geometry_records(seed, G, lods=4):
    """PrimitiveSet records {count, first} of G geometries, 4 each."""
    r = np.random.RandomState((int(seed) * 31 + 5) & 0x7FFFFFFF)
    ps = np.zeros((G, 4, 2), np.uint32)
    ps[:, :, 0] = r.randint(1, 1 << 17, (G, 4))
    ps[:, :, 1] = r.randint(0, 1 << 30, (G, 4))
    return torch.from_numpy(ps.reshape(-1).view(np.int32)).to(DEV)


def drawable_records(g, n, G, first, list_handle):
    """DrawableGpuData[n] as int64[n, 6]: a random geometry and PrimitiveSet each, MatrixList handles as given."""
    geom = torch.randint(0, G, (n,), generator=g, device=DEV)
    offset = 8 * torch.randint(0, 4, (n,), generator=g, device=DEV)
    rec = torch.empty((n, 6), device=DEV, dtype=torch.int64)
    rec[:, 0], rec[:, 1], rec[:, 4] = first + 3 * geom, first + 3 * geom + 1, first + 3 * geom + 2
    rec[:, 2], rec[:, 3], rec[:, 5] = list_handle, first + 3 * G + n, offset
    return rec


def gather_memory(seed, n, G, first, level):
    """Handle tables, PrimitiveSet records and one 128-byte MatrixList per drawable."""
    ps = geometry_records(seed, G)
    tables = 8 * 2048 * (4 + (first + 3 * G + n) // 2048 - first // 2048 + (2 if level == 3 else 0))
    ps_at = -(-tables // 256) * 256
    ml_at = -(-(ps_at + 64 * G) // 256) * 256
    mem = region(ml_at + 128 * n)
    base = mem.data_ptr()
    mem.view(torch.int32)[ps_at // 4:ps_at // 4 + 16 * G].view(G, 16)[:, :8] = ps.view(G, 8)
    ml = mem.view(torch.int32)[ml_at // 4:].view(n, 32)
    ml[:, 0] = torch.randint(1, 9, (n,), generator=_rng(seed, 8), device=DEV, dtype=torch.int32)
    ml[:, 1] = 8
    g = torch.arange(G, device=DEV)
    a = torch.empty(3 * G + n + 1, device=DEV, dtype=torch.int64)
    a[0:3 * G:3], a[1:3 * G:3], a[2:3 * G:3] = FAR_DATA + 4096 * g, FAR_DATA + 4096 * g + 2048, base + ps_at + 64 * g
    a[3 * G:3 * G + n] = base + ml_at + 128 * torch.arange(n, device=DEV)
    a[3 * G + n] = FAR_DATA + (1 << 36)
    handle_tables(mem, 0, level, first, a)
    return mem


def prepare_gather(case, seed):
    n, G, level = case["drawables"], case["geometries"], case["level"]
    first = (1 << 22) + 12_345 if level == 3 else 1
    mem = gather_memory(seed, n, G, first, level)
    # MatrixLists in the order the drawables were made, the list in StateSet order
    order = statesets_of(_rng(seed, 5), n, case["statesets"])[0]
    records = drawable_records(_rng(seed, 6), n, G, first, first + 3 * G + order)
    edits = max(1, n // 1000)
    slots = torch.randperm(n, generator=_rng(seed, 7), device=DEV)[:edits].contiguous()
    edited = drawable_records(_rng(seed, 9), edits, G, first, records[slots, 2])
    edited[:, 3] = records[0, 3]
    indirect = torch.zeros((n, 4), device=DEV, dtype=torch.int32)
    pointers = torch.zeros((n, 4), device=DEV, dtype=torch.int64)
    push = N.PushConstants(mem.data_ptr(), records.data_ptr(), indirect.data_ptr(), pointers.data_ptr())
    return State(kind="gather", mem=mem, records=records, slots=slots.to(torch.int32), edited=edited, push=push,
                 level=level, n=n, indirect=indirect, pointers=pointers)


def run_gather(s):
    lib = N.load()
    N.check(lib.cadrScatterDrawables(s.records.data_ptr(), s.n, s.edited.data_ptr(), s.slots.data_ptr(), len(s.slots),
                                     None))
    N.check(lib.cadrProcessDrawables(ctypes.byref(s.push), s.level, s.n, None))
    return {"list": s.records, "indirect": s.indirect, **pointer_outputs(s.pointers)}


def pointer_outputs(pointers):
    """Vertex, index and drawable-data pointers; of the MatrixList's, the half that does not say where in
    device memory this process's lists happen to lie."""
    return {"vertex_index": pointers[:, :2], "matrix_list": pointers.view(torch.int32)[:, 4], "data": pointers[:, 3]}


class CullItems(ctypes.Structure):
    _fields_ = [(f, ctypes.c_uint64) for f in ("handleTable", "drawableList", "itemBase", "itemDrawable", "meshes",
                                               "spheres", "meshIndex", "numDrawables", "numItems")] + \
               [("handleLevel", ctypes.c_uint32), ("numMeshes", ctypes.c_uint32)]


def facade_functions():
    lib = N.load()
    u64, u32, ptr = ctypes.c_uint64, ctypes.c_uint32, ctypes.c_void_p
    lib.cadrBuildMeshTable.argtypes = [u64, u32, u64, u32, u64, ptr]
    lib.cadrBuildCullItems.argtypes = [ctypes.POINTER(CullItems), ptr]
    lib.cadrFinishCullCommands.argtypes = [u64, u64, u64, u32, u32, u32, u64, u64, u64, u64, u64, u64, ptr]
    return lib


class Plan:
    def __init__(self, levels):
        h = ctypes.c_void_p(0)
        N.check(N.load().cadrTransformPlanCreate(N.ptr(levels), len(levels), None, ctypes.byref(h)))
        self.handle = h.value

    def __del__(self):
        if getattr(self, "handle", None):
            N.load().cadrTransformPlanDestroy(self.handle)


def instance_inputs(case, seed):
    """Inner level, and the instances grouped by drawable: (roots, inner local, inner parents, leaf local, leaf
    parents, instances per drawable, StateSet of each drawable)."""
    D, n, nodes, K = case["drawables"], case["instances"], case["nodes"], case["statesets"]
    roots = rotation_translation(_rng(seed, 10), max(1, nodes // 100))
    inner = rotation_translation(_rng(seed, 11), nodes)
    inner_parent = (torch.arange(nodes, device=DEV) * len(roots) // nodes).to(torch.int32)
    # every instance of the scene graph, in its order, belongs to a random drawable; none is empty
    owner = torch.randint(0, D, (n,), generator=_rng(seed, 12), device=DEV)
    owner[:D] = torch.arange(D, device=DEV)
    per = torch.bincount(owner, minlength=D).cpu().numpy()
    node = torch.sort(owner, stable=True).indices
    leaf_parent = (node * nodes // n).to(torch.int32)
    leaf = rotation_translation(_rng(seed, 13), n)
    ss = np.sort(np.random.RandomState((int(seed) * 13 + 1) & 0x7FFFFFFF).randint(0, K, D))
    return roots, inner, inner_parent, leaf, leaf_parent, per, ss


def list_offsets(per):
    """Byte offset of each MatrixList (64-byte header, then the matrices) in one buffer, and its size."""
    size = 64 + 64 * per.astype(np.int64)
    return np.concatenate([[0], np.cumsum(size)[:-1]]), int(size.sum())


def prepare_instances(case, seed):
    lib = facade_functions()
    D, n, K, M = case["drawables"], case["instances"], case["statesets"], case["meshes"]
    roots, inner, inner_parent, leaf, leaf_parent, per, ss = instance_inputs(case, seed)
    offs, lists_bytes = list_offsets(per)
    first, level = 1, 2
    lists = torch.zeros(lists_bytes // 4, device=DEV, dtype=torch.float32)
    heads = torch.from_numpy(offs // 4).to(DEV)
    lists.view(torch.int32)[heads] = torch.from_numpy(per.astype(np.int32)).to(DEV)
    lists.view(torch.int32)[heads + 1] = torch.from_numpy(per.astype(np.int32)).to(DEV)
    # handles: 3 per geometry, one MatrixList per drawable, one drawable-data block
    mem = region(8 * 2048 * 8 + 64 * M + 4096)
    base, ps_at = mem.data_ptr(), 8 * 2048 * 8
    mem.view(torch.int32)[ps_at // 4:ps_at // 4 + 16 * M].view(M, 16)[:, :8] = geometry_records(seed, M).view(M, 8)
    g = torch.arange(M, device=DEV)
    a = torch.empty(3 * M + D + 1, device=DEV, dtype=torch.int64)
    a[0:3 * M:3], a[1:3 * M:3], a[2:3 * M:3] = FAR_DATA + 4096 * g, FAR_DATA + 4096 * g + 2048, base + ps_at + 64 * g
    a[3 * M:3 * M + D] = lists.data_ptr() + torch.from_numpy(offs).to(DEV)
    a[3 * M + D] = FAR_DATA + (1 << 36)
    handle_tables(mem, 0, level, first, a)
    # drawables: one geometry each, the PrimitiveSet of LOD 0, the mesh index in the padding word
    mesh_of = torch.randint(0, M, (D,), generator=_rng(seed, 14), device=DEV)
    records = torch.zeros((D, 6), device=DEV, dtype=torch.int64)
    for c in range(2):
        records[:, c] = first + 3 * mesh_of + c
    records[:, 2], records[:, 3] = first + 3 * M + torch.arange(D, device=DEV), first + 3 * M + D
    records[:, 4], records[:, 5] = first + 3 * mesh_of + 2, mesh_of << 32
    meshes = mesh_table(seed, M, case["lods"])
    src = np.zeros(M, np.dtype([("handle", "<u8"), ("offset", "<u4"), ("lods", "<u4"), ("sphere", "<f4", (4,))]))
    src["handle"], src["lods"] = first + 3 * np.arange(M) + 2, case["lods"]
    src["sphere"][:, :3], src["sphere"][:, 3] = meshes["center"], meshes["radius"]
    # items: the instances, drawable by drawable, StateSet by StateSet
    item_base = torch.from_numpy(np.concatenate([[0], np.cumsum(per)[:-1]]).astype(np.int32)).to(DEV)
    item_drawable = torch.repeat_interleave(torch.arange(D, device=DEV, dtype=torch.int32),
                                            torch.from_numpy(per).to(DEV))
    counts = np.bincount(ss, weights=per, minlength=K).astype(np.uint32)
    range_base = torch.from_numpy(np.concatenate([[0], np.cumsum(counts)[:-1]]).astype(np.int32)).to(DEV)
    mi = torch.zeros(n, device=DEV, dtype=torch.int32)
    spheres = torch.zeros((n, 4), device=DEV)
    ds = SceneInMemory(n, counts, meshes, mi, spheres)   # the mesh table is rewritten by each frame
    out = Outputs(1, n, K)
    batch = cull.CullBatch(_config(case), [(ds, cameras(seed, 1, 100.0), out)])
    inner_world = torch.zeros_like(inner)
    inner_desc = level_desc(inner, inner_world, len(inner), inner_parent, roots, len(roots))
    lv = np.zeros(D, N.LEVEL_DTYPE)
    starts = np.concatenate([[0], np.cumsum(per)[:-1]]).astype(np.uint64)
    lv["localMatrices"] = leaf.data_ptr() + 64 * starts
    lv["parentIndex"] = leaf_parent.data_ptr() + 4 * starts
    lv["parentWorld"], lv["parentCount"] = inner_world.data_ptr(), len(inner)
    lv["worldMatrices"] = lists.data_ptr() + offs.astype(np.uint64) + np.uint64(64)
    lv["count"] = per
    torch.cuda.synchronize()
    plan = Plan(lv)
    indirect = torch.zeros((D, 4), device=DEV, dtype=torch.int32)
    pointers = torch.zeros((D, 4), device=DEV, dtype=torch.int64)
    draw_pointers = torch.zeros((n, 4), device=DEV, dtype=torch.int64)
    items = CullItems(base, records.data_ptr(), item_base.data_ptr(), item_drawable.data_ptr(), ds.meshes.address,
                      spheres.data_ptr(), mi.data_ptr(), D, n, level, M)
    push = N.PushConstants(base, records.data_ptr(), indirect.data_ptr(), pointers.data_ptr())
    return State(kind="instances", lib=lib, keep=(mem, roots, inner, inner_parent, leaf, leaf_parent, records, item_base,
                                                  item_drawable, mi), inner_world=inner_world, inner_desc=inner_desc,
                 lists=lists, plan=plan, sources=to_device(src), ds=ds, out=out, batch=batch, spheres=spheres,
                 indirect=indirect, pointers=pointers, draw_pointers=draw_pointers, items=items, push=push,
                 range_base=range_base, D=D, n=n, K=K, M=M, base=base, level=level, item_base=item_base,
                 item_drawable=item_drawable)


def run_instances(s):
    lib, ds = s.lib, s.ds
    N.check(lib.cadrPropagateTransforms(N.ptr(s.inner_desc), None))
    N.check(lib.cadrPropagateTransformsPlanned(s.plan.handle, None))
    N.check(lib.cadrProcessDrawables(ctypes.byref(s.push), s.level, s.D, None))
    N.check(lib.cadrBuildMeshTable(s.base, s.level, s.sources.data_ptr(), s.M, ds.meshes.address, None))
    N.check(lib.cadrBuildCullItems(ctypes.byref(s.items), None))
    s.batch.run_view()
    N.check(lib.cadrFinishCullCommands(s.out.cmd.data_ptr(), s.out.cnt.data_ptr(), s.range_base.data_ptr(), 1, s.K, s.n,
                                       s.item_base.data_ptr(), s.item_drawable.data_ptr(), s.n, s.pointers.data_ptr(),
                                       s.D, s.draw_pointers.data_ptr(), None))
    return {"inner": s.inner_world, "lists": s.lists, "spheres": s.spheres, "indirect": s.indirect,
            "commands": s.out.cmd, "counts": s.out.cnt, "vertex_index": s.draw_pointers[:, :2],
            "data": s.draw_pointers[:, 3]}


PREPARE = {"view": prepare_view, "flat": prepare_view, "frame": prepare_frame, "levels": prepare_frame,
           "views": prepare_views, "scenes": prepare_scenes, "served": prepare_scenes, "gather": prepare_gather,
           "instances": prepare_instances}
RUN = {"view": run_view, "flat": run_flat, "frame": run_frame, "levels": run_levels, "views": run_views,
       "scenes": run_scenes, "served": run_served, "gather": run_gather, "instances": run_instances}


def prepare(case, seed):
    s = PREPARE[case["kind"]](case, int(seed))
    torch.cuda.synchronize()
    return s


def run(state):
    return RUN[state.kind](state)


# ----------------------------------------------------------------------------------------------- work

SEEN = 0.15      # share of a scene's drawables that a camera sees, about: a command of 20 bytes each
TEST = 30.0      # operations of a sphere's view coordinates and plane tests


def work(case):
    kind = case["kind"]
    if kind in ("view", "flat"):
        n = case["drawables"]
        b = n * (4 + 20 * SEEN) + n * (64 + 16 if kind == "flat" else 16)
        return {"bytes": b, "flops": n * (TEST + (40 if kind == "flat" else 0))}
    if kind in ("frame", "levels"):
        sizes = level_sizes(case["drawables"], case["depth"], case["roots"])
        n, V = sizes[-1], case.get("views", 1)
        b = 128 * sum(sizes) + 4 * sum(sizes[1:]) + 4 * n + V * 20 * SEEN * n + (16 * n if kind == "levels" else 0)
        return {"bytes": b, "flops": 112 * sum(sizes[1:]) + 40 * n + TEST * n * V}
    if kind == "views":
        n, V = case["drawables"], case["views"]
        return {"bytes": 20 * n + 20 * SEEN * n * V, "flops": TEST * n * V}
    if kind in ("scenes", "served"):
        b = f = 0
        for n, _, _, V in layout(case):
            b += n * (136 if kind == "scenes" else 20) + 20 * SEEN * n * V
            f += n * (150 if kind == "scenes" else 0) + TEST * n * V
        return {"bytes": b, "flops": f}
    if kind == "gather":
        # record, MatrixList handle and count read, command and pointers written; the edited records
        n = case["drawables"]
        return {"bytes": n * (48 + 8 + 4 + 48) + 96 * max(1, n // 1000), "flops": 0}
    n, m = case["instances"], case["nodes"]
    return {"bytes": 132 * (n + m) + n * (4 + 20) + SEEN * n * (20 + 64), "flops": 112 * (n + m) + (40 + TEST) * n}


# ---------------------------------------------------------------------------------------------- exact


def product(parent, local):
    """Column-major mat4 products in float64, in parts that stay small."""
    out = torch.empty_like(local)
    for c in range(0, len(local), 1 << 20):
        a, b = parent[c:c + (1 << 20)].view(-1, 4, 4), local[c:c + (1 << 20)].view(-1, 4, 4)
        r = out[c:c + (1 << 20)].view(-1, 4, 4)
        r.copy_(sum(a[:, None, k, :] * b[:, :, k, None] for k in range(4)))
    return out


def sphere_of(world, meshes, mesh_index):
    """World spheres in float64: centre transformed, radius times the longest column."""
    m = torch.from_numpy(np.concatenate([meshes["center"], meshes["radius"][:, None]], 1)).to(DEV).double()[mesh_index.long()]
    w = world.view(-1, 4, 4)
    c = sum(w[:, k, :3] * m[:, k, None] for k in range(3)) + w[:, 3, :3]
    r = w[:, :3, :3].square().sum(2).max(1).values.sqrt() * m[:, 3]
    return torch.cat([c, r[:, None]], 1)


def exact_worlds(inputs):
    worlds = []
    for local, parent in inputs:
        local = local.double()
        worlds.append(local if parent is None else product(worlds[-1][parent.long()], local))
    return worlds


def exact(case, seed):
    kind, seed = case["kind"], int(seed)
    if kind == "flat":
        meshes = mesh_table(seed, case["meshes"], case["lods"])
        mi = mesh_indices(seed, 3, case["drawables"], len(meshes))
        world = scale_translation(_rng(seed, 4), case["drawables"]).double()
        return {"spheres": sphere_of(world, meshes, mi), "commands": None, "counts": None}
    if kind in ("frame", "levels"):
        sizes = level_sizes(case["drawables"], case["depth"], case["roots"])
        worlds = exact_worlds(tree_inputs(seed, 10, sizes, case["statesets"])[0])
        got = {"worlds": worlds, "commands": None, "counts": None}
        if kind == "levels":
            meshes = mesh_table(seed, case["meshes"], case["lods"])
            got["spheres"] = sphere_of(worlds[-1], meshes, mesh_indices(seed, 3, sizes[-1], len(meshes)))
        return got
    if kind == "scenes":
        parts = []
        for i, (n, depth, _, _) in enumerate(layout(case)):
            f = max(1, math.ceil(n ** (1.0 / depth) - 1e-9))
            sizes = [n]
            for _ in range(depth - 1):
                sizes.append(-(-sizes[-1] // f))
            parts.append(exact_worlds(tree_inputs(seed, 1000 * i + 10, sizes[::-1], case["statesets"])[0])[-1])
        return {"worlds": torch.cat(parts), "commands": None, "counts": None}
    if kind == "instances":
        roots, inner, inner_parent, leaf, leaf_parent, per, ss = instance_inputs(case, seed)
        inner_world = product(roots.double()[inner_parent.long()], inner.double())
        world = product(inner_world[leaf_parent.long()], leaf.double())
        offs, nbytes = list_offsets(per)
        lists = torch.zeros(nbytes // 64, 16, device=DEV, dtype=torch.float64)
        rows = torch.ones(nbytes // 64, device=DEV, dtype=torch.bool)
        heads = torch.from_numpy(offs // 64).to(DEV)
        rows[heads] = False
        lists[rows] = world
        count = torch.from_numpy(per.astype(np.int32)).to(DEV).view(torch.float32).double()
        lists[heads, 0], lists[heads, 1] = count, count
        meshes = mesh_table(seed, case["meshes"], case["lods"])
        D = case["drawables"]
        mesh_of = torch.randint(0, len(meshes), (D,), generator=_rng(seed, 14), device=DEV)
        mi = torch.repeat_interleave(mesh_of, torch.from_numpy(per).to(DEV))
        return {"inner": inner_world, "lists": lists.view(-1), "spheres": sphere_of(world, meshes, mi), "indirect": None,
                "commands": None, "counts": None, "vertex_index": None, "data": None}
    return None
