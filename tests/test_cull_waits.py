"""Bounded look-back waits: a caller-built tile list that names a predecessor
no tile publishes makes every launch end anyway, and the workspace reports
CADR_ERROR_TIMEOUT.  The condition is forced from the host: a tile list
without the first tile of its StateSet and a 1-ms wait limit, so each kernel
exits after its waits give up.  Well-formed launches on the same workspace
stay bit-exact against the oracle."""
import numpy as np
import pytest

import oracle
from cadr_amd import _native as N
from cadr_amd import cull, scenes
from cadr_amd.device import DeviceBuffer, synchronize

pytestmark = pytest.mark.gpu

N_DRAWABLES = 3000


@pytest.fixture(scope="module")
def small(gpu):
    scene = scenes.plain_scene(N_DRAWABLES)
    ds = cull.DeviceScene(scene)
    ds.propagate()
    _, spheres = oracle.propagate_scene(scene)
    yield scene, ds, spheres
    ds.close()


def _job(ds, tiles_buf, num_tiles, views_buf, num_views, out):
    jobs = np.zeros(1, dtype=N.JOB_DTYPE)
    jobs[0] = (ds.spheres.address, ds.mesh_index.address, ds.meshes.address, tiles_buf.address, views_buf.address,
               out.commands.address, out.counts.address, ds.n, num_tiles, ds.K, num_views, out.stride,
               ds.num_meshes)
    return jobs


@pytest.mark.parametrize("path", ["view", "batch"])
def test_missing_predecessor_times_out_and_workspace_recovers(small, path):
    import ctypes
    scene, ds, spheres = small
    config = cull.make_config(256, 4)
    tile = cull.tile_size(config)
    good = cull.build_tiles(scene.stateset_counts, tile)
    assert good.shape[0] == 3 and int(good[0]["stateSetAndFlags"]) & N.TILE_FIRST
    bad = good[1:].copy()  # tiles 1 and 2: both wait (through chain 0) on a tile that is not in the list
    print(f"missing-predecessor tile list, {path} kernel, 1 ms wait limit", flush=True)
    views = cull.make_views([scenes.DEFAULT_CAMERA])
    vb = DeviceBuffer.from_array(views)
    good_b, bad_b = DeviceBuffer.from_array(good), DeviceBuffer.from_array(bad)
    out = cull.CullOutputs(1, ds.n, ds.K)
    ws = cull.Workspace(16, 1)
    ws.set_wait_limit(1000)
    lib = N.load()

    def launch(tb, nt):
        jobs = _job(ds, tb, nt, vb, 1, out)
        jb = DeviceBuffer.from_array(jobs)
        if path == "view":
            rc = lib.cadrCullView(ctypes.byref(config), jb.address, N.ptr(jobs), ws.handle, None)
        else:
            rc = lib.cadrCullBatch(ctypes.byref(config), jb.address, N.ptr(jobs), 1, ws.handle, None)
        N.check(rc)
        synchronize()
        jb.close()

    exp_cmds, exp_counts = oracle.cull(spheres, scene.mesh_index, scene.meshes, scene.stateset_counts, views,
                                       cmd_dtype=N.CMD_DTYPE)
    # the malformed list ends and is reported once
    launch(bad_b, bad.shape[0])
    with pytest.raises(N.CadrError) as e:
        ws.check()
    assert e.value.code == N.ERROR_TIMEOUT
    ws.check()  # the record was cleared
    # a well-formed launch after it is exact and reports nothing
    launch(good_b, good.shape[0])
    ws.check()
    cmds, counts = out.download()
    assert np.array_equal(counts, exp_counts)
    n = int(exp_counts[0, 0])
    assert cmds[0, :n].tobytes() == exp_cmds[0, :n].tobytes()
    # the record is sticky across later good launches until checked
    launch(bad_b, bad.shape[0])
    launch(good_b, good.shape[0])
    cmds, counts = out.download()
    assert np.array_equal(counts, exp_counts) and cmds[0, :n].tobytes() == exp_cmds[0, :n].tobytes()
    with pytest.raises(N.CadrError) as e:
        ws.check()
    assert e.value.code == N.ERROR_TIMEOUT
    for b in (vb, good_b, bad_b):
        b.close()
    out.close()
    ws.close()


def test_missing_predecessor_in_the_persistent_view_kernel(gpu):
    """The same through the persistent one-view kernel, which runs when a
    view has more tiles than resident workgroups (800k drawables in tiles
    of 1024; two 1024-thread workgroups fit per CU): a list without its first
    tile ends after the 1-ms limit and is reported; the full list then gives
    the oracle's draw list on the same workspace."""
    import ctypes
    scene = scenes.plain_scene(800_000, seed=scenes.SEED_BASE + 23)
    ds = cull.DeviceScene(scene)
    ds.propagate()
    spheres = ds.download_spheres()
    config = cull.make_config(1024, 1)
    good = cull.build_tiles(scene.stateset_counts, cull.tile_size(config))
    assert good.shape[0] > 2 * 256
    bad = good[1:].copy()
    print(f"missing-predecessor tile list, persistent view kernel, {bad.shape[0]} tiles", flush=True)
    views = cull.make_views([scenes.DEFAULT_CAMERA])
    vb = DeviceBuffer.from_array(views)
    good_b, bad_b = DeviceBuffer.from_array(good), DeviceBuffer.from_array(bad)
    out = cull.CullOutputs(1, ds.n, ds.K)
    ws = cull.Workspace(good.shape[0], 1)
    ws.set_wait_limit(1000)
    lib = N.load()

    def launch(tb, nt):
        jobs = _job(ds, tb, nt, vb, 1, out)
        jb = DeviceBuffer.from_array(jobs)
        N.check(lib.cadrCullView(ctypes.byref(config), jb.address, N.ptr(jobs), ws.handle, None))
        synchronize()
        jb.close()

    launch(bad_b, bad.shape[0])
    with pytest.raises(N.CadrError) as e:
        ws.check()
    assert e.value.code == N.ERROR_TIMEOUT
    launch(good_b, good.shape[0])
    ws.check()
    cmds, counts = out.download()
    exp_cmds, exp_counts = oracle.cull(spheres, scene.mesh_index, scene.meshes, scene.stateset_counts, views,
                                       cmd_dtype=N.CMD_DTYPE)
    assert np.array_equal(counts, exp_counts)
    n = int(exp_counts[0, 0])
    assert n > 0 and cmds[0, :n].tobytes() == exp_cmds[0, :n].tobytes()
    for b in (vb, good_b, bad_b):
        b.close()
    out.close()
    ws.close()
    ds.close()


# Launches of several ticket counters (work items of few bytes, 256 workgroups or more): a workgroup that waits long for
# tiles of workgroups that do not run leaves its item, and the launch's last workgroup finishes it.  A tile list in
# reverse order, of more tiles than workgroups fit on the GPU, forces it from the host: every workgroup that runs waits
# for tiles whose tickets nobody has taken.

def _reversed_scene(n, K, tile, fanouts=None):
    scene = (scenes.tree_scene(fanouts, seed=scenes.SEED_BASE + 1100, num_statesets=K) if fanouts else
             scenes.plain_scene(n, seed=scenes.SEED_BASE + 1100, num_statesets=K))
    ds = cull.DeviceScene(scene)
    tiles = cull.build_tiles(scene.stateset_counts, tile)[::-1].copy()
    ds._tiles[tile] = (DeviceBuffer.from_array(tiles), tiles.shape[0])
    return scene, ds, tiles.shape[0]


def _check_outputs(scene, ds, spheres, views, out):
    exp_cmds, exp_counts = oracle.cull(spheres, scene.mesh_index, scene.meshes, scene.stateset_counts, views,
                                       cmd_dtype=N.CMD_DTYPE)
    cmds, counts = out.download()
    assert np.array_equal(counts, exp_counts)
    got = cull.valid_commands(cmds, counts, scene.stateset_counts)
    exp = cull.valid_commands(exp_cmds, exp_counts, scene.stateset_counts)
    for v in range(len(views)):
        for k in range(ds.K):
            assert got[v][k].tobytes() == exp[v][k].tobytes(), f"view {v} StateSet {k}"


@pytest.mark.parametrize("block,items,n,K,views,entry", [
    (512, 2, 1_150_000, 1, 1, "view"),      # one workgroup per tile
    (1024, 1, 600_000, 3, 1, "view"),       # the persistent loop
    (256, 2, 1_050_000, 2, 1, "view"),      # the persistent few-view kernel
    (256, 2, 1_050_000, 1, 2, "batch"),     # two views, four, one item of four and one of two
    (256, 2, 1_050_000, 5, 4, "batch"),
    (256, 2, 700_000, 1, 6, "batch"),
    (512, 2, 600_000, 2, 5, "batch"),       # the many-view kernel
])
def test_tiles_of_workgroups_that_do_not_run(gpu, block, items, n, K, views, entry):
    print(f"{n} drawables, {K} StateSets, {views} views, {block}x{items}, {entry}", flush=True)
    scene, ds, tiles = _reversed_scene(n, K, block * items)
    ds.propagate()
    cams = cull.make_views(scenes.random_cameras(31, 20, 0, views, 200.0))
    out = cull.CullOutputs(views, ds.n, ds.K)
    batch = cull.CullBatch(cull.make_config(block, items), [(ds, cams, out)])
    for _ in range(2):
        out.counts.fill_u32(0xDEADBEEF)
        batch.run_view() if entry == "view" else batch.run()
        synchronize()
        batch.workspace.check()
        _check_outputs(scene, ds, oracle.propagate_scene(scene)[1], cams, out)
    batch.close()
    out.close()
    ds.close()


@pytest.mark.parametrize("block,items,fanouts,K,views,entry", [
    (512, 2, (3, 400, 900), 1, 1, "view"), (256, 4, (1, 1_100_003), 2, 1, "view"), (256, 4, (1_100_003,), 1, 1, "view"),
    (256, 4, (4, 300, 1000), 3, 1, "batch"), (256, 4, (1_100_003,), 1, 2, "batch")])
def test_fused_tiles_of_workgroups_that_do_not_run(gpu, block, items, fanouts, K, views, entry):
    print(f"{fanouts}, {K} StateSets, {views} views, {block}x{items}, {entry}", flush=True)
    scene, ds, tiles = _reversed_scene(0, K, block * items, fanouts)
    worlds, spheres = oracle.propagate_scene(scene)
    descs = ds.level_descs(spheres=False)
    for lv in descs[:-1]:
        N.check(N.load().cadrPropagateTransforms(N.ptr(lv), None))
    cams = cull.make_views(scenes.random_cameras(37, 20, 0, views, 100.0))
    out = cull.CullOutputs(views, ds.n, ds.K)
    batch = cull.CullBatch(cull.make_config(block, items), [(ds, cams, out)])
    if entry == "batch":
        batch.set_leaves(descs[-1])
    for _ in range(2):
        out.counts.fill_u32(0xDEADBEEF)
        batch.run_fused(descs[-1]) if entry == "view" else batch.run_fused_batch()
        synchronize()
        batch.workspace.check()
        _check_outputs(scene, ds, spheres, cams, out)
    assert ds.world_matrices(-1).tobytes() == worlds[-1].tobytes()
    batch.close()
    out.close()
    ds.close()


@pytest.mark.parametrize("block,items,n,K,views", [(256, 4, 600_000, 1, 1), (256, 2, 1_300_000, 64, 1), (1024, 1, 700_000, 7, 1),
                                                   (256, 4, 900_000, 7, 2), (256, 8, 900_000, 1, 4), (512, 2, 500_000, 3, 6)])
def test_impatient_waits_stay_exact(gpu, block, items, n, K, views):
    """A wait limit of 1 us: items are left, by every kernel of several ticket counters, whenever a look-back is not ready at
    once, and no wait gives up."""
    print(f"{n} drawables, {K} StateSets, {views} views, {block}x{items}", flush=True)
    scene = scenes.plain_scene(n, seed=scenes.SEED_BASE + 1101, num_statesets=K)
    ds = cull.DeviceScene(scene)
    ds.propagate()
    spheres = ds.download_spheres()
    cams = cull.make_views(scenes.random_cameras(41, 20, 0, views, 200.0))
    out = cull.CullOutputs(views, ds.n, ds.K)
    batch = cull.CullBatch(cull.make_config(block, items), [(ds, cams, out)])
    batch.workspace.set_wait_limit(1)
    for k in range(3):
        out.counts.fill_u32(0xDEADBEEF)
        batch.run_view() if views == 1 and (k < 2 or block == 1024) else batch.run()
        synchronize()
        batch.workspace.check()
        _check_outputs(scene, ds, spheres, cams, out)
    batch.close()
    out.close()
    ds.close()


def test_sharded_launches_on_two_streams(gpu):
    """Two streams, a workspace each, launches of both in flight together: each takes workgroup slots from the other."""
    from cadr_amd.device import Stream
    jobs = []
    for j, (n, V) in enumerate(((1_500_000, 1), (900_000, 2))):
        scene = scenes.plain_scene(n, seed=scenes.SEED_BASE + 1102 + j, num_statesets=1 + 2 * j)
        ds = cull.DeviceScene(scene)
        ds.propagate()
        cams = cull.make_views(scenes.random_cameras(43 + j, 20, 0, V, 200.0))
        out = cull.CullOutputs(V, ds.n, ds.K)
        jobs.append((scene, ds, cams, out, cull.CullBatch(cull.make_config(256, 2 + 2 * j), [(ds, cams, out)]), Stream()))
    synchronize()
    for k in range(8):
        for scene, ds, cams, out, batch, stream in jobs:
            batch.run_view(stream.handle) if len(cams) == 1 and k % 2 else batch.run(stream.handle)
    synchronize()
    for scene, ds, cams, out, batch, stream in jobs:
        batch.workspace.check()
        _check_outputs(scene, ds, ds.download_spheres(), cams, out)
        batch.close()
        stream.close()
        out.close()
        ds.close()
