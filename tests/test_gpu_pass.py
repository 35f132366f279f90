"""What a traversal pass may vary without changing a hit: the reciprocals of
very long and short directions, leaves tested in parts, and batches of one
query kind or of both (each its own kernel)."""
import numpy as np
import pytest

from luxcore_amd import device as D
from luxcore_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def soup(gpu_device):
    mesh = scenes.soup_scene(4000, extent=10.0, seed=3)
    rng = np.random.Generator(np.random.PCG64(5))
    rays = scenes.random_rays(20011, (0, 0, 0), (10, 10, 10), rng, mint=0.0)
    out = {layout: gpu_device.scene_bvh([mesh], layout=layout, max_leaf=8) for layout in (0, 1, 2)}
    yield gpu_device, out, rays
    for s in out.values():
        s.close()


# a power of two scales every product of the triangle test exactly, so the
# hit is the same and t scales; above 1e30 (2^100) the box test divides, below
# it takes the hardware reciprocal
@pytest.mark.parametrize("layout", [0, 1, 2])
@pytest.mark.parametrize("exponent", [-30, 1, 60, 99, 100, 101, 105])
def test_scaled_directions(soup, layout, exponent):
    dev, sc, rays = soup
    want = dev.trace_numpy(sc[layout], rays)
    scaled = rays.copy()
    scaled["d"] *= np.float32(2.0) ** exponent
    got = dev.trace_numpy(sc[layout], scaled)
    got["t"] *= np.float32(2.0) ** exponent
    assert np.array_equal(got, want)
    one = rays.copy()   # a single huge component
    one["d"][:, 1:] = 0
    one["d"][:, 0] = np.float32(2.0) ** exponent
    unit = one.copy()
    unit["d"][:, 0] = 1
    a, b = dev.trace_numpy(sc[layout], one), dev.trace_numpy(sc[layout], unit)
    a["t"] *= np.float32(2.0) ** exponent
    assert np.array_equal(a, b)


@pytest.mark.parametrize("layout", [0, 1, 2])
@pytest.mark.parametrize("leaf_tris", [1, 2, 3, 7, 8])
def test_leaves_in_parts(soup, layout, leaf_tris):
    dev, sc, rays = soup
    want = dev.trace_numpy(sc[layout], rays, opts=D.trace_opts(leaf_tris=8))
    assert np.array_equal(dev.trace_numpy(sc[layout], rays, opts=D.trace_opts(leaf_tris=leaf_tris)), want)


@pytest.mark.parametrize("layout", [0, 1, 2])
@pytest.mark.parametrize("queries", [(0, 0), (1, 1), (0, 1)])
def test_batches_of_each_query_kind(soup, layout, queries):
    dev, sc, rays = soup
    want = [dev.trace_numpy(sc[layout], rays, query=q) for q in queries]
    rb = dev.upload(rays)
    hb = [dev.alloc(20 * rays.size) for _ in queries]
    dev.trace_batch([(sc[layout], rb, h, rays.size, q) for h, q in zip(hb, queries)])
    dev.sync()
    for h, w in zip(hb, want):
        assert np.array_equal(dev.download(h, w.dtype, rays.size), w)
        h.free()
    rb.free()
