"""The cull launches on both sides of the rules that choose how they run, bit for bit against the oracle: two
launches on one workspace each time, so that the first leaves the workspace as the second needs it."""
import numpy as np
import pytest

import oracle
from cadr_amd import _native as N
from cadr_amd import cull, scenes
from cadr_amd.device import synchronize

pytestmark = pytest.mark.gpu


def _jobs(specs):
    """(device scene, views, outputs, spheres, scene) per (drawables, StateSets, meshes, views)."""
    out = []
    for i, (n, K, M, V) in enumerate(specs):
        scene = scenes.plain_scene(n, seed=scenes.SEED_BASE + 900 + i, num_statesets=K, num_meshes=M)
        ds = cull.DeviceScene(scene)
        ds.propagate()
        views = cull.make_views(scenes.random_cameras(77 + i, 20, 0, V, 200.0))
        out.append((ds, views, cull.CullOutputs(V, ds.n, ds.K), oracle.propagate_scene(scene)[1], scene))
    return out


def _check(jobs, what):
    for ds, views, out, spheres, scene in jobs:
        cmds, counts = out.download()
        ec, en = oracle.cull(spheres, scene.mesh_index, scene.meshes, scene.stateset_counts, views, cmd_dtype=N.CMD_DTYPE)
        assert np.array_equal(counts, en), f"{what}: counts differ"
        got = cull.valid_commands(cmds, counts, scene.stateset_counts)
        exp = cull.valid_commands(ec, en, scene.stateset_counts)
        for v in range(len(got)):
            for k in range(len(scene.stateset_counts)):
                assert got[v][k].tobytes() == exp[v][k].tobytes(), f"{what}: view {v} StateSet {k}"


def _run(specs, block, items, run, flags=0):
    jobs = _jobs(specs)
    batch = cull.CullBatch(cull.make_config(block, items, flags=flags), [j[:3] for j in jobs])
    for k in range(2):
        for _, _, out, _, _ in jobs:
            out.counts.fill_u32(0xDEADBEEF)
            out.commands.fill_u32(0)
        run(batch)
        synchronize()
        batch.workspace.check()
        _check(jobs, f"{specs} {block}x{items} launch {k}")
    batch.close()
    for ds, _, out, _, _ in jobs:
        out.close()
        ds.close()


# ticket shards: 1 below 256 workgroups, then more as the tiles get smaller and the workgroups more, the last
# runs of 8 tiles cut off at every remainder
@pytest.mark.parametrize("tiles,K", [(255, 1), (256, 1), (263, 3), (513, 64), (1031, 1), (4099, 7)])
@pytest.mark.parametrize("block,items", [(256, 2), (256, 4)])
def test_ticket_shards(gpu, tiles, K, block, items):
    n = (tiles - K) * block * items + 5
    print(f"{n} drawables, {K} StateSets, {block}x{items}", flush=True)
    _run([(n, K, 64, 1)], block, items, lambda b: b.run_view())
    _run([(n, K, 64, 1)], block, items, lambda b: b.run())


# a wave's list of visible items: empty, full, one over a chunk of 64 commands; mesh tables on both sides of the
# staged size; the persistent loop (1024 x 8 past 256 tiles)
@pytest.mark.parametrize("block,items,n,K", [(256, 2, 1, 1), (256, 4, 1023, 1), (256, 4, 1025, 2), (512, 16, 8193, 1),
                                             (1024, 1, 4097, 3), (1024, 8, 8191, 1), (1024, 8, 2_200_003, 5)])
@pytest.mark.parametrize("meshes", [64, 65])
def test_one_view_lists(gpu, block, items, n, K, meshes):
    print(f"{n} drawables, {K} StateSets, {meshes} meshes, {block}x{items}", flush=True)
    eye, up = (0.0, 0.0, 2500.0), (0.0, 1.0, 0.0)
    views = cull.make_views([scenes.Camera(eye, (0.0, 0.0, d), up, 1.2, 1.0, 0.1, 6000.0, 1080.0, (40.0, 8.0, 0.5))
                             for d in (-1.0, 1.0)] + scenes.random_cameras(5, 20, 0, 2, 100.0))
    (ds, _, out, spheres, scene), = _jobs([(n, K, meshes, 1)])
    for v in range(len(views)):  # everything, nothing, and two parts
        view = views[v:v + 1].copy()
        batch = cull.CullBatch(cull.make_config(block, items), [(ds, view, out)])
        batch.run_view()
        synchronize()
        batch.workspace.check()
        _check([(ds, view, out, spheres, scene)], f"{block}x{items} view {v}")
        batch.close()
    out.close()
    ds.close()


# job offsets: worked out by the workgroups in chunks of 64 jobs, by a kernel of their own past 256
@pytest.mark.parametrize("jobs", [2, 64, 65, 256, 257])
def test_job_offsets(gpu, jobs):
    print(f"{jobs} jobs", flush=True)
    specs = [(1 + (j * 37) % 90 + (600 if j % 50 == 3 else 0), 1 + j % 3, 8, 1 + (67 if j == 1 else j % 4))
             for j in range(jobs)]
    _run(specs, 256, 2, lambda b: b.run())


# few views: 1, 2 and 4 at a time, the last group cut off, mesh tables staged (one job) and not; CULL_WHOLE_TILES
# takes more than four views to the many-view kernel, whose view groups end at 32 and 64
@pytest.mark.parametrize("block,items", [(256, 2), (256, 4), (256, 8), (512, 4)])
@pytest.mark.parametrize("flags", [0, N.CULL_WHOLE_TILES])
@pytest.mark.parametrize("specs", [[(5000, 3, 64, 1)], [(5000, 2, 65, 2), (1, 1, 9, 1), (2049, 4, 300, 2)],
                                   [(4097, 1, 64, 3)], [(900, 5, 7, 4), (3000, 1, 64, 1)], [(3001, 2, 64, 5)],
                                   [(2500, 3, 80, 33), (2500, 1, 64, 2)], [(1025, 1, 64, 65)]])
def test_few_and_many_views(gpu, block, items, flags, specs):
    print(f"{specs} {block}x{items} flags {flags}", flush=True)
    _run(specs, block, items, lambda b: b.run(), flags)


def test_many_views_boundary_spheres(gpu):
    """Spheres within ulps of every plane, through the many-view kernel's estimate."""
    from test_cull import _boundary_spheres
    rng = np.random.default_rng(3)
    views = cull.make_views(scenes.random_cameras(11, 20, 0, 8, 100.0))
    spheres = _boundary_spheres(views, 40, rng)
    n = spheres.shape[0]
    scene = scenes.plain_scene(n, num_statesets=1)
    ds = cull.DeviceScene(scene)
    ds.upload_spheres(spheres)
    out = cull.CullOutputs(len(views), n, 1)
    batch = cull.CullBatch(cull.make_config(256, 8, flags=N.CULL_WHOLE_TILES), [(ds, views, out)])
    batch.run()
    synchronize()
    _check([(ds, views, out, spheres, scene)], "boundary spheres")
    batch.close()
    out.close()
    ds.close()


# one-view launches of at most one tile a compute unit run the widest shape of their tile size
@pytest.mark.parametrize("block,items,fanouts", [(256, 4, (4, 256, 256)), (256, 4, (4, 256, 257)),
                                                 (256, 8, (8, 256, 256)), (256, 8, (8, 256, 257)), (512, 2, (3, 7, 11))])
def test_fused_shape_by_tiles(gpu, block, items, fanouts):
    print(f"{fanouts} {block}x{items}", flush=True)
    scene = scenes.tree_scene(fanouts, seed=scenes.SEED_BASE + 950, num_statesets=1, lod_count=3)
    worlds, spheres = oracle.propagate_scene(scene)
    ds = cull.DeviceScene(scene)
    descs = ds.level_descs(spheres=False)
    views = cull.make_views(scenes.random_cameras(9, 20, 0, 1, 100.0))
    out = cull.CullOutputs(1, ds.n, ds.K)
    batch = cull.CullBatch(cull.make_config(block, items), [(ds, views, out)])
    for lv in descs[:-1]:
        N.check(N.load().cadrPropagateTransforms(N.ptr(lv), None))
    for k in range(2):
        batch.run_fused(descs[-1])
        synchronize()
        batch.workspace.check()
        _check([(ds, views, out, spheres, scene)], f"fused {block}x{items} launch {k}")
    assert ds.world_matrices(-1).tobytes() == worlds[-1].tobytes()
    batch.close()
    out.close()
    ds.close()


def test_deferred_look_back_over_many_tiles(gpu):
    """Jobs of more tiles than workgroups, one and two views: each workgroup stores an item after it has taken the next."""
    _run([(2_000_003, 3, 64, 2), (500_001, 5, 64, 1), (70, 1, 3, 2)], 256, 2, lambda b: b.run())
    _run([(2_500_003, 1, 64, 1)], 256, 4, lambda b: b.run_view())


# batched launches of at most one tile a compute unit run 256 x 8 tiles with 512 threads
@pytest.mark.parametrize("tiles", [1, 256, 257])
@pytest.mark.parametrize("views", [1, 3, 18])
def test_batch_shape_by_tiles(gpu, tiles, views):
    _run([(tiles * 2048 - 5, 1, 64, views)], 256, 8, lambda b: b.run())


# fused batches: few tiles are cut by four views (each item computes its leaves again, one of them stores them), more
# tiles and CULL_WHOLE_TILES are not
@pytest.mark.parametrize("block,items,flags,fanouts", [(256, 4, 0, (3, 50, 21)), (256, 4, N.CULL_WHOLE_TILES, (3, 50, 21)),
                                                       (256, 8, 0, (2, 30, 40)), (512, 4, N.CULL_WHOLE_TILES, (2, 30, 40)),
                                                       (256, 4, 0, (2, 300, 260))])
def test_fused_batch_view_groups(gpu, block, items, flags, fanouts):
    print(f"{fanouts} {block}x{items} flags {flags}", flush=True)
    jobs, leaves, worlds = [], [], []
    for j, V in enumerate((9, 2, 70)):
        scene = scenes.tree_scene((fanouts[0] + j,) + fanouts[1:], seed=scenes.SEED_BASE + 970 + j, num_statesets=3)
        w, spheres = oracle.propagate_scene(scene)
        ds = cull.DeviceScene(scene)
        descs = ds.level_descs(spheres=False)
        for lv in descs[:-1]:
            N.check(N.load().cadrPropagateTransforms(N.ptr(lv), None))
        views = cull.make_views(scenes.random_cameras(13 + j, 20, 0, V, 150.0))
        jobs.append((ds, views, cull.CullOutputs(V, ds.n, ds.K), spheres, scene))
        leaves.append(descs[-1])
        worlds.append(w[-1])
    batch = cull.CullBatch(cull.make_config(block, items, flags=flags), [j[:3] for j in jobs])
    batch.set_leaves(np.concatenate(leaves))
    for k in range(2):
        batch.run_fused_batch()
        synchronize()
        batch.workspace.check()
        _check(jobs, f"fused batch launch {k}")
    for (ds, _, out, _, _), w in zip(jobs, worlds):
        assert ds.world_matrices(-1).tobytes() == w.tobytes()
        out.close()
    batch.close()
    for ds, *_ in jobs:
        ds.close()


# jobs without views first, in the middle and last, of one tile and of many, beside jobs of few and many views: such a
# job has no look-back chains and no outputs, and the others' are what they are without it
NO_VIEWS = [(70_001, 1, 64, 0), (9000, 2, 64, 70), (1, 1, 8, 0), (70_001, 3, 65, 0), (5000, 1, 64, 2), (70_001, 1, 64, 0)]


@pytest.mark.parametrize("block,items,flags", [(256, 4, N.CULL_WHOLE_TILES), (256, 8, N.CULL_WHOLE_TILES), (256, 16, 0),
                                               (512, 2, 0), (128, 8, 0)])
def test_jobs_without_views_many(gpu, block, items, flags):
    """The many-view kernel (shapes without a few-view one, or whole tiles for 70 views)."""
    print(f"{block}x{items} flags {flags}", flush=True)
    _run(NO_VIEWS, block, items, lambda b: b.run(), flags)


@pytest.mark.parametrize("block,items", [(256, 2), (256, 4), (256, 8), (512, 4)])
@pytest.mark.parametrize("specs", [
    [(70_001, 1, 64, 0)],                                                                   # nothing but that
    [(70_001, 1, 64, 0), (9000, 2, 64, 1), (70_001, 3, 8, 0), (5, 1, 9, 1), (30_001, 1, 64, 0)],  # one view at a time
    [(70_001, 1, 64, 0), (9000, 2, 64, 2), (70_001, 3, 8, 0), (5, 1, 9, 1), (30_001, 1, 64, 0)],  # two
    NO_VIEWS])                                                                              # four
def test_jobs_without_views_few(gpu, block, items, specs):
    print(f"{specs} {block}x{items}", flush=True)
    _run(specs, block, items, lambda b: b.run())


@pytest.mark.parametrize("views", [1, 2])
def test_jobs_without_views_past_the_inline_offsets(gpu, views):
    """More than 256 jobs, whose offsets a kernel of its own works out: every third without views."""
    specs = [(1 + (j * 41) % 90 + (3000 if j % 50 == 3 else 0), 1 + j % 3, 8, 0 if j % 3 == 0 else 1 + j % views)
             for j in range(260)]
    _run(specs, 256, 2, lambda b: b.run())


def test_jobs_without_views_fused(gpu):
    """Fused launches write the leaf level of such a job too."""
    jobs, leaves, worlds = [], [], []
    for j, V in enumerate((0, 3, 0, 70, 0)):
        scene = scenes.tree_scene((3 + j, 50, 21), seed=scenes.SEED_BASE + 990 + j, num_statesets=2)
        w, spheres = oracle.propagate_scene(scene)
        ds = cull.DeviceScene(scene)
        descs = ds.level_descs()
        for lv in descs[:-1]:
            N.check(N.load().cadrPropagateTransforms(N.ptr(lv), None))
        views = cull.make_views(scenes.random_cameras(17 + j, 20, 0, V, 150.0))
        jobs.append((ds, views, cull.CullOutputs(V, ds.n, ds.K), spheres, scene))
        leaves.append(descs[-1])
        worlds.append(w[-1])
    batch = cull.CullBatch(cull.make_config(256, 4), [j[:3] for j in jobs])
    batch.set_leaves(np.concatenate(leaves))
    batch.run_fused_batch()
    synchronize()
    batch.workspace.check()
    _check(jobs, "fused batch with jobs without views")
    for (ds, _, out, spheres, _), w in zip(jobs, worlds):
        assert ds.world_matrices(-1).tobytes() == w.tobytes()
        assert ds.download_spheres().tobytes() == spheres.tobytes()
        out.close()
    batch.close()
    for ds, *_ in jobs:
        ds.close()


# leaf levels whose world matrices take the local ones' place: a tile's matrices are computed by one work item, whatever
# the views and tiles (few tiles: cut by four views otherwise; more than 64 views: by 64)
@pytest.mark.parametrize("block,items,fanouts,views", [(256, 4, (3, 50, 21), (5, 64, 33)), (256, 4, (2, 40, 30), (9, 2, 70)),
                                                       (512, 4, (2, 30, 40), (64, 17)), (256, 8, (4, 40, 30), (64,)),
                                                       (256, 4, (2, 300, 260), (130,))])
def test_fused_batch_in_place(gpu, block, items, fanouts, views):
    print(f"{fanouts} {block}x{items} views {views}", flush=True)
    jobs, leaves, worlds = [], [], []
    for j, V in enumerate(views):
        scene = scenes.tree_scene((fanouts[0] + j,) + fanouts[1:], seed=scenes.SEED_BASE + 1010 + j, num_statesets=3)
        w, spheres = oracle.propagate_scene(scene)
        ds = cull.DeviceScene(scene)
        descs = ds.level_descs(spheres=False)
        for lv in descs[:-1]:
            N.check(N.load().cadrPropagateTransforms(N.ptr(lv), None))
        descs[-1]["worldMatrices"] = descs[-1]["localMatrices"]
        cams = cull.make_views(scenes.random_cameras(23 + j, 20, 0, V, 150.0))
        jobs.append((ds, cams, cull.CullOutputs(V, ds.n, ds.K), spheres, scene))
        leaves.append(descs[-1])
        worlds.append(w[-1])
    batch = cull.CullBatch(cull.make_config(block, items), [j[:3] for j in jobs])
    batch.set_leaves(np.concatenate(leaves))
    batch.run_fused_batch()
    synchronize()
    batch.workspace.check()
    _check(jobs, "fused batch in place")
    for (ds, _, out, _, _), w in zip(jobs, worlds):
        n, local = ds.levels[-1][0], ds.levels[-1][1]
        assert local.download(np.float32, n * 16).reshape(n, 16).tobytes() == w.tobytes()
        out.close()
    batch.close()
    for ds, *_ in jobs:
        ds.close()


@pytest.mark.parametrize("tiles,views,error", [(0x40000000, 16, "too few status words"), (0xfffffff0, 8, "too few status words"),
                                               (0xffffffff, 1, "too many tiles")])
def test_work_item_limit_is_that_of_whole_tiles(gpu, tiles, views, error):
    """Tickets are 32 bits.  Jobs whose tiles only have too many items when cut by four views are not refused for it: the
    call goes on to the next check, the workspace's status words, which ends it here (nothing is launched)."""
    import ctypes
    jobs = np.zeros(1, N.JOB_DTYPE)
    jobs[0] = (16, 16, 16, 16, 16, 16, 16, 100, tiles, 1, views, 100, 1)
    ws = cull.Workspace(16, 1)
    config = cull.make_config(256, 4)
    with pytest.raises(N.CadrError, match=error):
        N.check(N.load().cadrCullBatch(ctypes.byref(config), 16, N.ptr(jobs), 1, ws.handle, None))
    ws.close()


@pytest.mark.parametrize("meshes", [1 << 19, (1 << 19) + 77])
def test_mesh_tables_past_the_list_entries(gpu, meshes):
    """A list entry holds 19 bits of mesh index; the meshes of a larger table are read again when commands are stored."""
    print(f"{meshes} meshes", flush=True)
    _run([(30_001, 3, meshes, 1)], 256, 4, lambda b: b.run_view())
    _run([(30_001, 3, meshes, 1)], 1024, 1, lambda b: b.run_view())
    _run([(9000, 2, meshes, 3), (700, 1, 9, 1)], 256, 2, lambda b: b.run())
    _run([(9000, 2, meshes, 70)], 256, 8, lambda b: b.run(), N.CULL_WHOLE_TILES)
