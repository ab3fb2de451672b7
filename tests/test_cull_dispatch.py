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


def _run(specs, block, items, run):
    jobs = _jobs(specs)
    batch = cull.CullBatch(cull.make_config(block, items), [j[:3] for j in jobs])
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
