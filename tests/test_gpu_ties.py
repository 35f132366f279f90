"""Hits at exactly equal distances.  Five coincident copies of every triangle
(or object): which copy a ray reports depends on the order of its visits, and
that order is the ray's own, whatever launch it is part of.  The counting
kernel (64 rays a wave, no drain), small launches (a ray shared among lanes
from the start), large ones (shared at the end of a wave), batches of one query
kind and of both give the same record, bit for bit, launch after launch.
Some rays start inside many boxes (equal entry distances), some at a negative
mint (negative ones)."""
import numpy as np
import pytest

from luxcore_amd import device as D
from luxcore_amd import scenes
from luxcore_amd.raytypes import HIT_DTYPE

pytestmark = pytest.mark.gpu

COUNTS = [5, 3000, 50000, 250001]
COPIES = 5


def make_rays(n, extent, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    rays = scenes.random_rays(n, (-extent,) * 3, (extent,) * 3, rng)
    rays["time"] = rng.random(n, dtype=np.float32)
    rays["mint"][::3] = -np.float32(extent)
    rays["maxt"][::5] = np.float32(extent) / 2
    return rays


@pytest.fixture(scope="module", params=[0, 1, 2])
def single(request, gpu_device):
    sc = gpu_device.scene_bvh([scenes.soup_scene(700, extent=4.0, seed=3, mean_edge=0.6)] * COPIES,
                              layout=request.param, max_leaf=2)
    yield gpu_device, sc, make_rays(max(COUNTS), 4.0, 21)
    sc.close()


@pytest.fixture(scope="module", params=[0, 1, 2])
def instanced(request, gpu_device):
    one = scenes.instanced_scene(n_inst=30, motion_frac=0.3, freq=4, extent=6.0, seed=4)
    n_keys = np.diff(one.key_off)
    sc = scenes.InstancedScene(
        one.meshes, np.tile(one.obj_mesh, COPIES), np.tile(one.obj_kind, COPIES), np.tile(one.obj_mat, (COPIES, 1, 1)),
        np.concatenate([[0], np.cumsum(np.tile(n_keys, COPIES))]).astype(np.uint32), np.tile(one.key_times, COPIES),
        np.tile(one.key_mats, (COPIES, 1, 1)))
    dsc = gpu_device.scene_mbvh(sc, layout=request.param)
    yield gpu_device, dsc, make_rays(max(COUNTS), 6.0, 22)
    dsc.close()


def check(dev, sc, rays, query):
    n = rays.size
    rb, other = dev.upload(rays), dev.alloc(20 * n)
    hb = dev.alloc(20 * n)

    def hits():
        dev.sync()
        return dev.download(hb, HIT_DTYPE, n)

    dev.trace_counters(sc, rb, hb, n, query)
    want = hits()
    assert (want["meshIndex"] != 0xffffffff).any()
    for opts in (None, D.trace_opts(256, 4, 1, 64), D.trace_opts(64, 64, 0, 1)):
        for _ in range(2):
            dev.trace(sc, rb, hb, n, query, opts)
            assert np.array_equal(hits(), want)
    for q in (0, 1):
        dev.trace_batch([(sc, rb, hb, n, query), (sc, rb, other, n, q)])
        assert np.array_equal(hits(), want)
    for b in (rb, hb, other):
        b.free()


@pytest.mark.parametrize("count", COUNTS)
@pytest.mark.parametrize("query", [0, 1])
def test_single_level(single, count, query):
    dev, sc, rays = single
    print(f"[case] ties single {count} {query}", flush=True)
    check(dev, sc, rays[:count], query)


@pytest.mark.parametrize("count", COUNTS)
@pytest.mark.parametrize("query", [0, 1])
def test_two_level(instanced, count, query):
    dev, sc, rays = instanced
    print(f"[case] ties two-level {count} {query}", flush=True)
    check(dev, sc, rays[:count], query)
