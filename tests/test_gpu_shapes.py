"""Launch shapes at the limits of what is accepted: the LDS stack's largest
sizes trace, what does not fit with a block's lanes is refused whatever the
number of rays, and the no-alloc trace of small launches (rays shared among
lanes from the start) gives lrh_trace's records."""
import numpy as np
import pytest

from luxcore_amd import device as D
from luxcore_amd import scenes
from luxcore_amd.raytypes import HIT_DTYPE

pytestmark = pytest.mark.gpu

COUNTS = [1, 7, 17, 4097, 20011, 120001]


@pytest.fixture(scope="module", params=[0, 2])
def workload(request, gpu_device):
    sc = gpu_device.scene_bvh([scenes.soup_scene(3000, extent=10.0, seed=3)], layout=request.param)
    rng = np.random.Generator(np.random.PCG64(6))
    rays = scenes.random_rays(max(COUNTS), (0, 0, 0), (10, 10, 10), rng)
    rays["flags"][rng.random(rays.size) < 0.1] = 1
    yield gpu_device, sc, rays
    sc.close()


@pytest.mark.parametrize("count", COUNTS)
@pytest.mark.parametrize("block,lds", [(256, 32), (128, 64), (64, 64), (256, 4)])
def test_largest_lds_stacks_trace(workload, count, block, lds):
    dev, sc, rays = workload
    init = np.zeros(count, HIT_DTYPE)
    want = dev.trace_numpy(sc, rays[:count], hits_init=init)
    got = dev.trace_numpy(sc, rays[:count], opts=D.trace_opts(block, lds), hits_init=init)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("count", COUNTS)
@pytest.mark.parametrize("block,lds", [(0, 64), (256, 64)])
def test_lds_stack_beyond_a_block_is_refused(workload, count, block, lds):
    dev, sc, rays = workload
    with pytest.raises(D.LrhError, match="exceed 64 KiB"):
        dev.trace_numpy(sc, rays[:count], opts=D.trace_opts(block, lds))


@pytest.mark.parametrize("count", COUNTS)
@pytest.mark.parametrize("query", [0, 1])
def test_noalloc_of_small_launches(workload, count, query):
    dev, sc, rays = workload
    init = np.zeros(count, HIT_DTYPE)
    init["t"] = 7.0   # masked rays keep this
    want = dev.trace_numpy(sc, rays[:count], query=query, hits_init=init)
    rb, hb = dev.upload(rays[:count]), dev.upload(init)
    D.check(D.lib().lrh_trace_noalloc(sc.h, rb.ptr, hb.ptr, count, query, None))
    dev.sync()
    assert np.array_equal(dev.download(hb, HIT_DTYPE, count), want)
    rb.free()
    hb.free()


@pytest.mark.parametrize("count", [30011, 49152])
def test_noalloc_of_a_small_launch_on_a_capped_grid(gpu_device, count):
    """The shared start over a tree whose spill stacks leave room for fewer
    lanes than it asks for: the rest of the rays come through the tickets."""
    dev = gpu_device
    sc = dev.scene_bvh(scenes.plain_scene(seed=1, n_random=20000), layout=2)
    lane_bytes = 8 * (7 * (sc.info()["maxDepth"] + 2) + 4 - 8)
    assert 128 * 1024 * 1024 // lane_bytes < 8 * count
    rays = scenes.plain_rays(count, seed=17)
    init = np.zeros(count, HIT_DTYPE)
    for query in (0, 1):
        want = dev.trace_numpy(sc, rays, query=query, hits_init=init)
        rb, hb = dev.upload(rays), dev.upload(init)
        D.check(D.lib().lrh_trace_noalloc(sc.h, rb.ptr, hb.ptr, count, query, None))
        dev.sync()
        assert np.array_equal(dev.download(hb, HIT_DTYPE, count), want)
        rb.free()
        hb.free()
    sc.close()
