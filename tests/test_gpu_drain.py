"""The drain, in which the last rays of a wave (and all rays of a small launch)
are shared among lanes: the same hits as the counting variant, which has no
drain, bit for bit, any-hit ones too.  Counts at the edges of a wave's, a
group's and a small launch's rays; rings of four entries, so that shared pushes
and pops go through the spill array."""
import numpy as np
import pytest

from luxcore_amd import device as D
from luxcore_amd import scenes
from luxcore_amd.raytypes import HIT_DTYPE

pytestmark = pytest.mark.gpu

COUNTS = [1, 2, 7, 8, 9, 15, 16, 17, 64, 65, 4097, 49152, 49153, 65536, 65537, 120001]


@pytest.fixture(scope="module")
def single(gpu_device):
    meshes = [scenes.soup_scene(3000, extent=10.0, seed=3), scenes.icosphere_l6(2.0, (5, 5, 5))]
    rng = np.random.Generator(np.random.PCG64(6))
    rays = scenes.random_rays(max(COUNTS), (0, 0, 0), (10, 10, 10), rng)
    rays["maxt"][::5] = 3.0
    rays["mint"][::7] = -2.0
    rays["flags"][rng.random(rays.size) < 0.1] = 1
    out = {layout: gpu_device.scene_bvh(meshes, layout=layout, max_leaf=8) for layout in (0, 1, 2)}
    yield gpu_device, out, rays
    for s in out.values():
        s.close()


@pytest.fixture(scope="module")
def instanced(gpu_device):
    sc = scenes.instanced_scene(n_inst=60, motion_frac=0.3, freq=8, extent=6.0, seed=4)
    rays = scenes.instanced_rays(max(COUNTS), extent=6.0, seed=8)
    out = {layout: gpu_device.scene_mbvh(sc, layout=layout) for layout in (0, 1, 2)}
    yield gpu_device, out, rays
    for s in out.values():
        s.close()


def both(dev, sc, rays, query, opts):
    n = rays.size
    init = np.zeros(n, HIT_DTYPE)
    init["t"] = 7.0   # masked rays keep this
    rb, hb = dev.upload(rays), dev.upload(init)
    dev.trace_counters(sc, rb, hb, n, query, opts)
    want = dev.download(hb, HIT_DTYPE, n)
    dev.upload(init, hb)
    dev.trace(sc, rb, hb, n, query, opts)
    dev.sync()
    got = dev.download(hb, HIT_DTYPE, n)
    rb.free()
    hb.free()
    return got, want


@pytest.mark.parametrize("layout", [0, 1, 2])
@pytest.mark.parametrize("count", COUNTS)
@pytest.mark.parametrize("query", [0, 1])
def test_single_level(single, layout, count, query):
    dev, sc, rays = single
    for opts in (None, D.trace_opts(256, 4), D.trace_opts(64, 64)):
        got, want = both(dev, sc[layout], rays[:count], query, opts)
        assert np.array_equal(got, want)


@pytest.mark.parametrize("layout", [0, 1, 2])
@pytest.mark.parametrize("count", COUNTS)
@pytest.mark.parametrize("query", [0, 1])
def test_two_level(instanced, layout, count, query):
    dev, sc, rays = instanced
    for opts in (None, D.trace_opts(256, 4)):
        got, want = both(dev, sc[layout], rays[:count], query, opts)
        assert np.array_equal(got, want)


@pytest.mark.parametrize("layout", [0, 2])
def test_batched(single, layout):
    dev, sc, rays = single
    cuts = [0, 3, 100, 9000, 70001]
    for query in (0, 1):
        bufs = []
        for a, b in zip(cuts[:-1], cuts[1:]):
            bufs.append((dev.upload(rays[a:b]), dev.upload(np.zeros(b - a, HIT_DTYPE)), b - a))
        dev.trace_batch([(sc[layout], r, h, n, query) for r, h, n in bufs], D.trace_opts(256, 4))
        dev.sync()
        for (r, h, n), a in zip(bufs, cuts):
            want = np.zeros(n, HIT_DTYPE)
            dev.upload(want, h2 := dev.alloc(20 * n))
            dev.trace_counters(sc[layout], r, h2, n, query)
            assert np.array_equal(dev.download(h, HIT_DTYPE, n), dev.download(h2, HIT_DTYPE, n))
            for x in (r, h, h2):
                x.free()
