"""Ray tickets of a persistent launch: the first grid's worth by lane, the rest
in units of 256 dealt to eight groups of blocks, each with a counter, and
through each block's pool.  Every ray is traced exactly
once whatever the count, grid and refill threshold: hits equal those of small
traces that never use the counter, bit for bit, on repeated launches."""
import numpy as np
import pytest

from luxcore_amd import device as D
from luxcore_amd import scenes
from luxcore_amd.raytypes import HIT_DTYPE

pytestmark = pytest.mark.gpu

PIECE = 16384   # below one block per CU: handed out by lane alone


@pytest.fixture(scope="module")
def workload(gpu_device):
    dev = gpu_device
    sc = dev.scene_bvh(scenes.heightfield_scene(cells=64, n_spheres=2), layout=2)
    rng = np.random.Generator(np.random.PCG64(11))
    rays = scenes.random_rays(400003, (-20, -20, -5), (20, 20, 12), rng)
    rays["flags"][rng.random(rays.size) < 0.3] = 1
    init = np.zeros(rays.size, HIT_DTYPE)
    init["t"] = np.arange(rays.size)   # masked rays keep this
    want = np.concatenate([dev.trace_numpy(sc, rays[a:a + PIECE], hits_init=init[a:a + PIECE])
                           for a in range(0, rays.size, PIECE)])
    yield dev, sc, rays, init, want
    sc.close()


# one block per CU = cu_count * block lanes; offsets from it in rays: the
# remainders of waves, of blocks, of units and of rounds of units
@pytest.mark.parametrize("block", [64, 256])
@pytest.mark.parametrize("offset", [-1, 0, 1, 63, 64, 65, 255, 256, 257, 2047, 2048, 2049, 65537, 200001])
@pytest.mark.parametrize("refill", [1, 16, 64])
def test_every_ray_once(workload, block, offset, refill):
    dev, sc, rays, init, want = workload
    n = dev.cu_count * block + offset
    rb, o = dev.upload(rays[:n]), D.trace_opts(block, 8, 1, refill)
    for _ in range(2):   # the counter is rewound by the launch before
        hb = dev.upload(init[:n])
        dev.trace(sc, rb, hb, n, 0, o)
        dev.sync()
        assert np.array_equal(dev.download(hb, HIT_DTYPE, n), want[:n])
        hb.free()
    rb.free()


@pytest.mark.parametrize("counts", [(1, 65536, 7), (100003, 1, 200000), (65536, 65536)])
def test_every_ray_once_batched(workload, counts):
    dev, sc, rays, init, want = workload
    starts = np.cumsum([0] + list(counts))
    bufs = [(dev.upload(rays[a:b]), dev.upload(init[a:b]), int(b - a)) for a, b in zip(starts[:-1], starts[1:])]
    dev.trace_batch([(sc, r, h, n, 0) for r, h, n in bufs], D.trace_opts(256, 8, 1, 16))
    dev.sync()
    for (r, h, n), a in zip(bufs, starts):
        assert np.array_equal(dev.download(h, HIT_DTYPE, n), want[a:a + n])
        r.free()
        h.free()
