"""Batched propagation of one, two and three levels (one and two load their descriptors at once, more scan the
counts), at the edges of the 64-node units, against the oracle."""
import numpy as np
import pytest

import oracle
from cadr_amd import _native as N
from cadr_amd.device import DeviceBuffer, synchronize

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts", [(1,), (64,), (65,), (0, 1), (63, 0), (64, 65), (129, 1), (70000, 3), (1, 64, 0), (65, 0, 200)])
@pytest.mark.parametrize("spheres", [False, True])
def test_batch_of_few_levels(gpu, counts, spheres):
    print(f"{counts} spheres {spheres}", flush=True)
    rng = np.random.default_rng(sum(counts))
    parents = rng.standard_normal((7, 16)).astype(np.float32)
    meshes = np.zeros(3, N.MESH_DTYPE)
    meshes["radius"], meshes["lodCount"], meshes["center"] = [1.0, 2.0, 0.5], 1, rng.standard_normal((3, 3))
    pb, mb = DeviceBuffer.from_array(parents), DeviceBuffer.from_array(meshes)
    levels, kept = np.zeros(len(counts), N.LEVEL_DTYPE), []
    for l, n in enumerate(counts):
        local = rng.standard_normal((n, 16)).astype(np.float32)
        parent = rng.integers(0, 9, n).astype(np.uint32)   # 7 and 8 act as roots
        mi = rng.integers(0, 4, n).astype(np.uint32)       # 3: outside the table
        root = l == 1
        bufs = [DeviceBuffer.from_array(a) for a in (local, parent, mi)] + [DeviceBuffer(max(64 * n, 16)),
                                                                           DeviceBuffer(max(16 * n, 16))]
        levels[l] = (bufs[0].address, bufs[1].address, 0 if root else pb.address, bufs[3].address, n, bufs[2].address,
                     mb.address, bufs[4].address if spheres else 0, 3, 7)
        kept.append((local, parent, mi, root, bufs))
    dev = DeviceBuffer.from_array(levels)
    N.check(N.load().cadrPropagateTransformsBatch(dev.address, N.ptr(levels), len(counts), None))
    synchronize()
    for l, (local, parent, mi, root, bufs) in enumerate(kept):
        n = counts[l]
        if n == 0:
            continue
        world, sph = oracle.propagate_level(local, None if root else parent, None if root else parents, mi, meshes)
        assert bufs[3].download(np.float32, 16 * n).tobytes() == np.ascontiguousarray(world).tobytes(), f"level {l}"
        if spheres:
            assert bufs[4].download(np.float32, 4 * n).tobytes() == np.ascontiguousarray(sph).tobytes(), f"level {l}"
