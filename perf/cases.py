"""The work that users of the intersection device have it do, as measurable cases.

Every case goes through the public entry points (luxcore_amd.device and
luxcore_amd.scenes): ray buffers traced against resident scenes, batches of
them, path-tracing passes, tree builds and edits.  Scenes come from this
repository's own generators at the sizes its tests and benchmark use; rays,
matrices, cameras and random numbers are drawn from the seed.

Outputs are hit records (20 bytes: t, b1, b2, meshIndex, triangleIndex) or path
records.  The device promises hit records that equal the reference's bit for
bit, so a record is returned as its five 32-bit words, with t of closest hits
also as a float; a ray that meets two triangles at exactly the same t (a shared
edge) may report either, and an any-hit ray may report any triangle that blocks
it, so a small share of the words may differ between correct versions.
"""
import math

import numpy as np
import torch

from luxcore_amd import device as D
from luxcore_amd import scenes as S

NULL = 0xFFFFFFFF
_DEV = None
_SCENES = {}   # resident geometry of this process, by what it is made of
_EXACT_TESTS = 3e9  # ray-triangle pairs that exact() goes through by brute force


def _dev():
    global _DEV
    if _DEV is None:
        torch.cuda.init()
        torch.zeros(1, device="cuda")
        _DEV = D.Device(0)
    return _DEV


class _Buf:
    """A torch tensor as the ray, hit or path buffer of a call."""

    def __init__(self, t):
        self.t = t
        self.ptr = t.data_ptr()


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the smallest buffer an engine hands over: one 64x64 tile of incoherent rays, default build options
        {"name": "trace_small", "kind": "trace", "scene": "terrain", "size": 256, "layout": 0, "rays": "bounce",
         "count": 4096, "query": 0},
        # camera rays of a full HD frame over a mid-size terrain (coherent), default build options
        {"name": "trace_primary", "kind": "trace", "scene": "terrain", "size": 1024, "layout": 0, "rays": "primary",
         "count": 1920 * 1080, "query": 0},
        # shadow rays of a wavefront with ended paths in it (masked rays), an odd count, any hit
        {"name": "trace_shadow", "kind": "trace", "scene": "terrain", "size": 1024, "layout": 2, "rays": "shadow",
         "count": 500001, "query": 1},
        # the headline: one diffuse bounce per pixel of a full HD frame over 26,238,080 triangles, 8-wide nodes
        {"name": "trace_bounce", "kind": "trace", "scene": "terrain", "size": 3240, "layout": 2, "rays": "bounce",
         "count": 1920 * 1080, "query": 0},
        # two-level: 1,000 instances of a 50,000-triangle mesh, 200 of them moving, 4Mi rays with their own times
        {"name": "trace_motion", "kind": "trace", "scene": "instances", "size": 1000, "layout": 2, "rays": "uniform",
         "count": 1 << 22, "query": 0},
        # many buffers of uneven sizes over several resident scenes in one replayed launch, mixed queries
        {"name": "batch", "kind": "batch", "buffers": 24, "largest": 1 << 20, "scenes": 5, "layout": 2},
        # a path-tracing pass of an interactive view: 1280x720, 8 vertices, a shadow ray per vertex
        {"name": "render", "kind": "render", "width": 1280, "height": 720, "depth": 8, "layout": 0, "spheres": 6},
        # wavefronts of several small path-tracing sessions over different scenes, batched step by step
        {"name": "serve", "kind": "serve", "sessions": 6, "side": 256, "depth": 5, "layout": 2, "scenes": 4},
        # the shading steps alone: three steps of a 1280x720 wavefront over recorded hits
        {"name": "shade", "kind": "shade", "count": 1280 * 720, "steps": 3},
        # geometry that changes each frame: the tree rebuilt on the GPU from host meshes, then traced
        {"name": "rebuild", "kind": "rebuild", "scene": "terrain", "size": 700, "builder": 1, "layout": 2,
         "count": 262144},
        # a deforming figure: the higher-quality device build of a small mesh, then a tile of rays
        {"name": "rebuild_ploc", "kind": "rebuild", "scene": "sphere", "size": 50, "builder": 2, "layout": 0,
         "count": 65536},
        # an animation frame: every instance moves, the root tree is refitted, then traced
        {"name": "refit", "kind": "refit", "size": 1000, "layout": 2, "count": 262144},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["trace", "trace", "trace", "trace", "batch", "render", "serve", "shade", "rebuild", "refit"])
    layout = rng.choice([0, 2])
    if kind == "trace":
        scene = rng.choice(["terrain", "terrain", "soup", "spheres", "instances"])
        rays = rng.choice(["bounce", "primary", "shadow"]) if scene == "terrain" else "uniform"
        size = {"terrain": (64, 1200), "soup": (10000, 500000), "spheres": (10000, 1000000),
                "instances": (20, 1000)}[scene]
        return {"kind": kind, "scene": scene, "size": _log_uniform(rng, *size), "layout": layout, "rays": rays,
                "count": _log_uniform(rng, 4096, 1 << 22 if scene != "soup" else 1 << 20), "query": rng.randrange(2)}
    if kind == "batch":
        return {"kind": kind, "buffers": rng.randint(3, 40), "largest": _log_uniform(rng, 1 << 14, 1 << 19),
                "scenes": rng.randint(1, 5), "layout": layout}
    if kind == "render":
        return {"kind": kind, "width": _log_uniform(rng, 100, 1280), "height": _log_uniform(rng, 60, 720),
                "depth": rng.randint(2, 8), "layout": layout, "spheres": rng.randint(1, 12)}
    if kind == "serve":
        return {"kind": kind, "sessions": rng.randint(1, 8), "side": _log_uniform(rng, 48, 256),
                "depth": rng.randint(2, 6), "layout": layout, "scenes": rng.randint(1, 4)}
    if kind == "shade":
        return {"kind": kind, "count": _log_uniform(rng, 4096, 2000000), "steps": rng.randint(1, 3)}
    if kind == "rebuild":
        scene = rng.choice(["terrain", "sphere"])
        return {"kind": kind, "scene": scene, "size": _log_uniform(rng, *((32, 700) if scene == "terrain" else (8, 120))),
                "builder": rng.choice([1, 2]), "layout": layout, "count": _log_uniform(rng, 4096, 1 << 20)}
    return {"kind": kind, "size": _log_uniform(rng, 20, 1000), "layout": layout, "count": _log_uniform(rng, 4096, 1 << 20)}


# ---------------------------------------------------------------------------
# resident scenes: built once per process, as a renderer keeps them
# ---------------------------------------------------------------------------
def _terrain(size):
    return S.heightfield_scene(cells=size, n_spheres=64 if size >= 2000 else 16 if size >= 512 else 2)


def _batch_meshes(k):
    return S.batch_scenes(sizes=S.BATCH_SCENE_TRIS[:k])


def _room(spheres):
    rng = np.random.Generator(np.random.PCG64(17))
    meshes = [S.box_mesh()]
    for _ in range(spheres):
        r = rng.uniform(0.6, 1.3)
        meshes.append(S.geodesic_sphere(32, r, rng.uniform(r + 0.2, 9.8 - r, 3)))
    return meshes


def _resident(*key):
    """(meshes or instanced scene, device scene(s)) of a key, made on first use."""
    if key not in _SCENES:
        dev, what, size, layout = _dev(), key[0], key[1], key[2]
        if what == "terrain":
            m = _terrain(size)
            _SCENES[key] = (m, dev.scene_bvh(m, layout=layout))
        elif what == "soup":
            m = [S.soup_scene(size, seed=100)]
            _SCENES[key] = (m, dev.scene_bvh(m, layout=layout))
        elif what == "spheres":
            m = [S.sphere_grid_scene(max(2000, size), seed=101)]
            _SCENES[key] = (m, dev.scene_bvh(m, layout=layout))
        elif what == "instances":
            m = S.instanced_scene(n_inst=size)
            _SCENES[key] = (m, dev.scene_mbvh(m, layout=layout))
        elif what == "batch":
            m = _batch_meshes(size)
            _SCENES[key] = (m, [dev.scene_bvh(x, layout=layout) for x in m])
        elif what == "room":
            m = _room(size)
            _SCENES[key] = (m, dev.scene_bvh(m, layout=layout))
    return _SCENES[key]


# ---------------------------------------------------------------------------
# rays, made on the GPU
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 2654435761 % (1 << 62) + 12345)
    return g


def _rand(g, *shape):
    return torch.rand(*shape, device="cuda", generator=g)


def _rays(o, d, mint=1e-4, maxt=math.inf, time=0.0, masked=None):
    r = torch.zeros(o.shape[0], 12, device="cuda")
    r[:, 0:3] = o
    r[:, 3:6] = d
    r[:, 6] = mint
    r[:, 7] = maxt
    r[:, 8] = time
    if masked is not None:
        r.view(torch.int32)[:, 9] = masked.to(torch.int32)
    return r


def _sphere_dirs(g, n):
    z = 1.0 - 2.0 * _rand(g, n)
    phi = 2.0 * math.pi * _rand(g, n)
    r = torch.sqrt(torch.clamp(1.0 - z * z, min=0.0))
    return torch.stack([r * torch.cos(phi), r * torch.sin(phi), z], 1)


def _cosine_dirs(g, n):
    """Cosine-weighted directions around the unit normals n."""
    m = n.shape[0]
    v = _sphere_dirs(g, m) * 0.9999 + n   # a unit vector plus a point of the unit sphere
    return v / v.norm(dim=1, keepdim=True)


def _epsilon(p):
    """The offset a ray's mint takes from its origin (128 ulps, within [1e-5, 0.1])."""
    up = (p.contiguous().view(torch.int32) + 0x80).view(torch.float32)
    return (up - p).abs().clamp(1e-5, 1e-1).amax(dim=1)


def _uniform_rays(g, n, lo, hi, time=False):
    return _rays(lo + (hi - lo) * _rand(g, n, 3), _sphere_dirs(g, n), time=_rand(g, n) if time else 0.0)


def _camera_frame(g):
    """A full HD camera above the terrain, turned about it by the seed."""
    a = float(_rand(g, 1)) * 2 * math.pi
    eye = torch.tensor([30.0 * math.sin(a), -30.0 * math.cos(a), 45.0], device="cuda")
    look = torch.tensor([-8.0 * math.sin(a), 8.0 * math.cos(a), 0.0], device="cuda")
    return eye, look


def _camera_dirs(g, eye, look, n):
    """n pixel directions in row order of a 16:9 view, jittered inside the pixels."""
    h = max(1, int(round(math.sqrt(n * 9 / 16))))
    w = -(-n // h)
    f = look - eye
    f = f / f.norm()
    right = torch.linalg.cross(f, torch.tensor([0.0, 0.0, 1.0], device="cuda"))
    right = right / right.norm()
    up = torch.linalg.cross(right, f)
    i = torch.arange(n, device="cuda")
    j = _rand(g, 2, n)
    th = math.tan(math.radians(36.0) / 2)
    px = ((i % w) + j[0]) / w * 2 - 1
    py = 1 - ((i // w) + j[1]) / h * 2
    d = f + (px * (th * 16 / 9))[:, None] * right + (py * th)[:, None] * up
    return d / d.norm(dim=1, keepdim=True)


def _terrain_points(meshes, size, xy):
    """Points on the heightfield above xy and its normals there, from its vertices."""
    n = size + 1
    v = torch.from_numpy(meshes[0].verts).cuda()
    lo, hi = v[0, 0:2], v[-1, 0:2]
    g = ((xy - lo) / (hi - lo)).clamp(0.0, 0.999999) * size
    ij = g.floor().clamp(0, size - 1).long()
    fx, fy = (g[:, 0] - ij[:, 0])[:, None], (g[:, 1] - ij[:, 1])[:, None]
    k = ij[:, 0] * n + ij[:, 1]
    v00, v10, v01, v11 = v[k], v[k + n], v[k + 1], v[k + n + 1]
    a = fx >= fy
    p = torch.where(a, v00 + fx * (v10 - v00) + fy * (v11 - v10), v00 + fy * (v01 - v00) + fx * (v11 - v01))
    nrm = torch.where(a, torch.linalg.cross(v10 - v00, v11 - v00), torch.linalg.cross(v11 - v00, v01 - v00))
    nrm = nrm / nrm.norm(dim=1, keepdim=True)
    return p, torch.where(nrm[:, 2:3] < 0, -nrm, nrm)


def _trace_rays(case, seed, meshes):
    g, n = _gen(seed), case["count"]
    if case["scene"] == "instances":
        return _uniform_rays(g, n, -100.0, 100.0, time=True)
    if case["rays"] == "uniform":
        return _uniform_rays(g, n, 0.0, 100.0)
    eye, look = _camera_frame(g)
    d = _camera_dirs(g, eye, look, n)
    if case["rays"] == "primary":
        return _rays(eye.expand(n, 3), d)
    # the surface points that the pixels look at, in pixel order
    p, nrm = _terrain_points(meshes, case["size"], eye[:2] + d[:, :2] * (-eye[2] / d[:, 2])[:, None])
    if case["rays"] == "bounce":
        return _rays(p, _cosine_dirs(g, nrm), mint=_epsilon(p))
    # shadow: toward a 1x1 light above the terrain; an eighth of the paths have ended
    light = torch.tensor([0.0, 0.0, 30.0], device="cuda").expand(n, 3).clone()
    light[:, :2] += _rand(g, n, 2) - 0.5
    v = light - p
    dist = v.norm(dim=1)
    eps = _epsilon(p)
    return _rays(p, v / dist[:, None], mint=eps, maxt=dist - 2 * eps, masked=_rand(g, n) < 0.125)


def _hits(n):
    return torch.zeros(n, 5, device="cuda")


def _hit_outputs(h, closest=None):
    """The records' words, and t of the first `closest` records (default: all)."""
    out = {"record": h.view(torch.int32)}
    if closest != 0:
        out["t"] = h[:closest, 0]
    return out


# ---------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------
def _upload(a):
    return _Buf(torch.from_numpy(np.ascontiguousarray(a).view(np.uint8).reshape(-1).copy()).cuda())


def _area_light(lo, hi, z, le):
    q = np.array([[lo, lo, z], [hi, lo, z], [hi, hi, z], [lo, hi, z]], np.float32)
    lt = np.zeros(2, D.LIGHT_DTYPE)
    for k, t in enumerate(((0, 2, 1), (0, 3, 2))):
        lt[k]["p0"], lt[k]["e1"], lt[k]["e2"], lt[k]["le"] = q[t[0]], q[t[1]] - q[t[0]], q[t[2]] - q[t[0]], le
    return lt


def _grey(n, kd=0.6):
    m = np.zeros(n, D.MATERIAL_DTYPE)
    m["kd"] = kd
    return m


def prepare(case, seed):
    return {"trace": _prepare_trace, "batch": _prepare_batch, "render": _prepare_render, "serve": _prepare_serve,
            "shade": _prepare_shade, "rebuild": _prepare_rebuild, "refit": _prepare_refit}[case["kind"]](case, seed)


def run(state):
    return state["run"](state)


def _prepare_trace(case, seed):
    meshes, scene = _resident(case["scene"], case["size"], case["layout"])
    return {"run": _run_trace, "case": case, "scene": scene, "rays": _Buf(_trace_rays(case, seed, meshes)),
            "hits": _Buf(_hits(case["count"]))}


def _run_trace(s):
    _dev().trace(s["scene"], s["rays"], s["hits"], s["case"]["count"], s["case"]["query"])
    return _hit_outputs(s["hits"].t, 0 if s["case"]["query"] else None)


def _batch_counts(case):
    """Buffer sizes, scenes and queries of a batch: log-uniform from 4Ki rays up, the largest first."""
    rng = np.random.Generator(np.random.PCG64(case["buffers"] * 1000003 + case["largest"]))
    counts = np.exp(rng.uniform(math.log(4096), math.log(case["largest"]), case["buffers"])).astype(int)
    counts[0] = case["largest"]
    spec = [(int(rng.integers(0, case["scenes"])), int(c), int(rng.integers(0, 2))) for c in counts]
    return sorted(spec, key=lambda x: x[2])   # closest-hit buffers first in the hit array


def _prepare_batch(case, seed):
    _, scenes = _resident("batch", case["scenes"], case["layout"])
    g = _gen(seed)
    spec = _batch_counts(case)
    rays = [_Buf(_uniform_rays(g, c, 0.0, 100.0)) for _, c, _ in spec]
    hits = _Buf(_hits(sum(c for _, c, _ in spec)))
    views, at = [], 0
    for _, c, _ in spec:
        views.append(_Buf(hits.t[at:at + c]))
        at += c
    torch.cuda.synchronize()
    batch = _dev().batch([(scenes[k], rays[i], views[i], c, q) for i, (k, c, q) in enumerate(spec)])
    batch.capture()
    return {"run": _run_batch, "case": case, "batch": batch, "hits": hits, "keep": (rays, views),
            "closest": sum(c for _, c, q in spec if q == 0)}


def _run_batch(s):
    s["batch"].replay()
    return _hit_outputs(s["hits"].t, s["closest"])


def _path_outputs(p):
    """Throughput, radiance and pending light as floats; depth, alive and the ended mark as words."""
    return {"path": p[:, 0:9], "path_words": p.view(torch.int32)[:, 9:12]}


def _prepare_render(case, seed):
    meshes, scene = _resident("room", case["spheres"], case["layout"])
    n = case["width"] * case["height"]
    g = _gen(seed)
    eye = (1.0 + 8.0 * _rand(g, 3)).cpu().numpy() * np.array([1, 0.05, 0.5]) + np.array([0, 0.3, 2.0])
    mats = _grey(len(meshes), 0.7)
    mats["kd"] *= np.random.Generator(np.random.PCG64(int(seed) % (1 << 31))).uniform(0.5, 1.0, (len(meshes), 3))
    buf = lambda words: _Buf(torch.zeros(n, words, device="cuda"))  # noqa: E731
    return {"run": _run_render, "case": case, "scene": scene, "n": n, "eye": [float(x) for x in eye],
            "seed": int(seed) % (1 << 62) + 1, "mats": _upload(mats), "nm": len(meshes),
            "lights": _upload(_area_light(3.5, 6.5, 9.9, 12.0)), "rays": [buf(12), buf(12)], "shadow": buf(12),
            "hits": buf(5), "shits": buf(5), "paths": buf(12)}


def _run_render(s):
    dev, n, c = _dev(), s["n"], s["case"]
    a, b = s["rays"]
    dev.camera_rays(a, s["eye"], (5.0, 6.0, 4.0), vfov_deg=60.0, width=c["width"], height=c["height"])
    dev.paths_init(s["paths"], n)
    for k in range(c["depth"]):
        dev.trace(s["scene"], a, s["hits"], n, 0)
        if k:
            dev.trace(s["scene"], s["shadow"], s["shits"], n, 1)
        dev.shade(s["scene"], s["mats"], s["nm"], s["lights"], 2, a, s["hits"], s["shits"] if k else None, s["paths"],
                  b, s["shadow"], n, max_depth=c["depth"], rr_depth=3, rr_survive=0.7, seed=s["seed"])
        a, b = b, a
    return _path_outputs(s["paths"].t)


def _prepare_serve(case, seed):
    meshes, scenes = _resident("batch", case["scenes"], case["layout"])
    n, g = case["side"] ** 2, _gen(seed)
    sessions = []
    for i in range(case["sessions"]):
        buf = lambda words: _Buf(torch.zeros(n, words, device="cuda"))  # noqa: E731
        p = _rand(g, 2, 3).cpu().numpy()
        sessions.append({"scene": scenes[i % len(scenes)], "eye": [float(x) for x in p[0] * 100.0],
                         "look": [float(x) for x in 30.0 + 40.0 * p[1]], "seed": int(seed) % (1 << 60) + 7 * i,
                         "rays": [buf(12), buf(12)], "shadow": buf(12), "hits": buf(5), "shits": buf(5)})
    paths = torch.zeros(case["sessions"] * n, 12, device="cuda")
    for i, x in enumerate(sessions):
        x["paths"] = _Buf(paths[i * n:(i + 1) * n])
    return {"run": _run_serve, "case": case, "n": n, "sessions": sessions, "paths": paths, "mats": _upload(_grey(1)),
            "lights": _upload(_area_light(35.0, 65.0, 150.0, 30.0))}


def _run_serve(s):
    dev, n, c = _dev(), s["n"], s["case"]
    for x in s["sessions"]:
        dev.camera_rays(x["rays"][0], x["eye"], x["look"], width=c["side"], height=c["side"])
        dev.paths_init(x["paths"], n)
    for k in range(c["depth"]):
        a, b = k % 2, 1 - k % 2
        items = [(x["scene"], x["rays"][a], x["hits"], n, 0) for x in s["sessions"]]
        if k:
            items += [(x["scene"], x["shadow"], x["shits"], n, 1) for x in s["sessions"]]
        dev.trace_batch(items)
        dev.shade_batch([(x["scene"], x["rays"][a], x["hits"], x["shits"] if k else None, x["paths"], x["rays"][b],
                          x["shadow"], n, c["depth"], 3, 0.7, x["seed"], 0) for x in s["sessions"]],
                        s["mats"], 1, s["lights"], 2)
    return _path_outputs(s["paths"])


def _shade_inputs(case, seed):
    """Per step: rays that meet random triangles of the room's spheres at their recorded hits (one in eight a
    miss), and what became of the step's shadow rays (half of them blocked)."""
    g, n = _gen(seed), case["count"]
    meshes = _room(6)[1:]
    tri = torch.from_numpy(np.concatenate([m.verts[m.tris.astype(np.int64)] for m in meshes])).cuda()
    base = np.cumsum([0] + [m.ntris for m in meshes])
    owner = torch.from_numpy(np.repeat(np.arange(len(meshes)), [m.ntris for m in meshes])).cuda()
    first = torch.from_numpy(base[:-1]).cuda()
    steps = []
    for _ in range(case["steps"]):
        k = torch.randint(0, tri.shape[0], (n,), device="cuda", generator=g)
        u = _rand(g, 2, n)
        su = u[0].sqrt()
        b1, b2 = (su * (1 - u[1]))[:, None], (su * u[1])[:, None]
        p = tri[k, 0] + b1 * (tri[k, 1] - tri[k, 0]) + b2 * (tri[k, 2] - tri[k, 0])
        d = _sphere_dirs(g, n)
        t = 0.5 + 4.0 * _rand(g, n)
        miss = _rand(g, n) < 0.125
        h = torch.zeros(n, 5, device="cuda")
        h[:, 0] = torch.where(miss, math.inf, t)
        h[:, 1], h[:, 2] = b1[:, 0], b2[:, 0]
        w = h.view(torch.int32)
        w[:, 3] = torch.where(miss, -1, owner[k].int())
        w[:, 4] = torch.where(miss, -1, (k - first[owner[k]]).int())
        sh = torch.zeros(n, 5, device="cuda")
        sh.view(torch.int32)[:, 3] = torch.where(_rand(g, n) < 0.5, -1, 0).int()
        steps.append({"rays": _rays(p - t[:, None] * d, d, mint=1e-4), "hits": h, "shits": sh, "tri": k})
    return meshes, tri, steps


def _shade_mats(seed):
    m = _grey(6)
    m["kd"] = np.random.Generator(np.random.PCG64(int(seed) % (1 << 31))).uniform(0.3, 0.9, (6, 3))
    m["le"][5] = 2.0
    return m


def _prepare_shade(case, seed):
    meshes, _, steps = _shade_inputs(case, seed)
    if "shade" not in _SCENES:
        _SCENES["shade"] = _dev().scene_bvh(meshes)
    n = case["count"]
    buf = lambda words: _Buf(torch.zeros(n, words, device="cuda"))  # noqa: E731
    return {"run": _run_shade, "case": case, "scene": _SCENES["shade"], "seed": int(seed) % (1 << 62) + 1,
            "steps": [{k: _Buf(x[k]) for k in ("rays", "hits", "shits")} for x in steps], "mats": _upload(_shade_mats(seed)),
            "lights": _upload(_area_light(3.5, 6.5, 9.9, 12.0)), "paths": buf(12), "next": [buf(12), buf(12)],
            "shadow": buf(12)}


def _run_shade(s):
    dev, c = _dev(), s["case"]
    dev.paths_init(s["paths"], c["count"])
    for k, x in enumerate(s["steps"]):
        dev.shade(s["scene"], s["mats"], 6, s["lights"], 2, x["rays"], x["hits"], x["shits"] if k else None, s["paths"],
                  s["next"][k % 2], s["shadow"], c["count"], max_depth=8, rr_depth=1, rr_survive=0.7, seed=s["seed"])
    nxt = s["next"][(c["steps"] - 1) % 2].t
    return {"path": s["paths"].t[:, 0:9], "path_words": s["paths"].t.view(torch.int32)[:, 9:12],
            "next": nxt[:, 0:9], "next_flags": nxt.view(torch.int32)[:, 9],
            "shadow": s["shadow"].t[:, 0:9], "shadow_flags": s["shadow"].t.view(torch.int32)[:, 9]}


def _deformed(case, seed):
    """The frame's geometry: the same meshes moved and reshaped by the seed, as host arrays."""
    if case["scene"] == "terrain":
        key = ("meshes", "terrain", case["size"])
        if key not in _SCENES:
            _SCENES[key] = _terrain(case["size"])
    else:
        key = ("meshes", "sphere", case["size"])
        if key not in _SCENES:
            _SCENES[key] = [S.displaced_sphere(freq=case["size"])]
    rng = np.random.Generator(np.random.PCG64(int(seed) % (1 << 31)))
    out = []
    for m in _SCENES[key]:
        v = m.verts.copy()
        ph = rng.uniform(0, 2 * np.pi, 2).astype(np.float32)
        v[:, 2] += np.float32(0.02 * np.abs(v).max()) * np.sin(v[:, 0] * np.float32(0.7) + ph[0]) * np.cos(v[:, 1] + ph[1])
        out.append(S.Mesh(v, m.tris))
    return out


def _rebuild_rays(case, seed, meshes):
    g, n = _gen(seed), case["count"]
    if case["scene"] == "sphere":
        o = _sphere_dirs(g, n) * 3.0
        d = _sphere_dirs(g, n) * 0.8 - o
        return _rays(o, d / d.norm(dim=1, keepdim=True))
    eye, look = _camera_frame(g)
    d = _camera_dirs(g, eye, look, n)
    p, nrm = _terrain_points(meshes, case["size"], eye[:2] + d[:, :2] * (-eye[2] / d[:, 2])[:, None])
    return _rays(p, _cosine_dirs(g, nrm), mint=_epsilon(p))


def _prepare_rebuild(case, seed):
    meshes = _deformed(case, seed)
    return {"run": _run_rebuild, "case": case, "meshes": meshes, "rays": _Buf(_rebuild_rays(case, seed, meshes)),
            "hits": _Buf(_hits(case["count"]))}


def _run_rebuild(s):
    c, dev = s["case"], _dev()
    scene = dev.scene_bvh(s["meshes"], layout=c["layout"], builder=c["builder"])
    dev.trace(scene, s["rays"], s["hits"], c["count"], 0)
    scene.close()
    return _hit_outputs(s["hits"].t)


def _moved(sc, seed):
    """Every object turned and shifted a little: new instance matrices and motion keys."""
    rng = np.random.Generator(np.random.PCG64(int(seed) % (1 << 31)))
    n = len(sc.obj_mesh)
    a = rng.uniform(-0.3, 0.3, n)
    M = np.tile(np.eye(4), (n, 1, 1))
    M[:, 0, 0], M[:, 0, 1], M[:, 1, 0], M[:, 1, 1] = np.cos(a), -np.sin(a), np.sin(a), np.cos(a)
    M[:, :3, 3] = rng.uniform(-5.0, 5.0, (n, 3))
    mats = sc.obj_mat.astype(np.float64).copy()
    mats[:, :3, :] = np.einsum("nij,njk->nik", M[:, :3, :3], mats[:, :3, :])
    mats[:, :3, 3] += M[:, :3, 3]
    owner = np.repeat(np.arange(n), np.diff(sc.key_off.astype(np.int64)))
    keys = sc.key_mats.astype(np.float64)
    if len(owner):
        keys = np.einsum("nij,njk->nik", keys, np.linalg.inv(M[owner]))
    return S.InstancedScene(sc.meshes, sc.obj_mesh, sc.obj_kind, mats.astype(np.float32), sc.key_off, sc.key_times,
                            keys.astype(np.float32))


def _prepare_refit(case, seed):
    key = ("instanced", case["size"])
    if key not in _SCENES:
        _SCENES[key] = S.instanced_scene(n_inst=case["size"])
    sc = _SCENES[key]
    return {"run": _run_refit, "case": case, "scene": _dev().scene_mbvh(sc, layout=case["layout"]),
            "edit": _moved(sc, seed), "rays": _Buf(_uniform_rays(_gen(seed), case["count"], -100.0, 100.0, time=True)),
            "hits": _Buf(_hits(case["count"]))}


def _run_refit(s):
    c, dev = s["case"], _dev()
    s["scene"].refit(s["edit"])
    dev.trace(s["scene"], s["rays"], s["hits"], c["count"], 0)
    out = _hit_outputs(s["hits"].t)
    out["boxes"] = s["scene"].object_boxes(c["size"])
    return out


# ---------------------------------------------------------------------------
# what each case cannot do without
# ---------------------------------------------------------------------------
def _mesh_sizes(case):
    """(vertices, triangles) of a rebuild's meshes."""
    if case["scene"] == "sphere":
        return 10 * case["size"] ** 2 + 2, 20 * case["size"] ** 2
    k = 64 if case["size"] >= 2000 else 16 if case["size"] >= 512 else 2
    return (case["size"] + 1) ** 2 + k * 40962, 2 * case["size"] ** 2 + k * 81920


def work(case):
    """Ray records read and hit records written once; for the steps around a trace the path state as well, and for
    builds and edits the geometry read and the tree's triangle records written.  The nodes and triangles that the rays
    have to meet depend on the rays and are not counted."""
    kind = case["kind"]
    if kind == "trace":
        return {"bytes": 68 * case["count"], "flops": 0}
    if kind == "batch":
        return {"bytes": 68 * sum(c for _, c, _ in _batch_counts(case)), "flops": 0}
    step = 2 * 68 + 2 * 20 + 3 * 48 + 48   # traces of both buffers; hits, ray, path read; path and two rays written
    if kind == "render":
        return {"bytes": case["width"] * case["height"] * case["depth"] * step, "flops": 0}
    if kind == "serve":
        return {"bytes": case["sessions"] * case["side"] ** 2 * case["depth"] * step, "flops": 0}
    if kind == "shade":
        return {"bytes": case["count"] * (48 + case["steps"] * (2 * 48 + 2 * 20 + 3 * 48)), "flops": 0}
    if kind == "rebuild":
        v, t = _mesh_sizes(case)
        return {"bytes": 12 * v + 12 * t + 48 * t + 68 * case["count"], "flops": 0}
    return {"bytes": case["size"] * (16 + 64 + 24) + 68 * case["count"], "flops": 0}


def tolerance(case):
    """Closest-hit records are bit-exact up to ties: traced over two different trees (4-wide and 8-wide nodes, so
    another visiting order) t never differed, and at most 4.1e-6 of a case's record words did.  Which blocker an
    any-hit ray reports depends on the visiting order: 1.0e-4 of the words over the two trees for shadow rays, 1.7e-2
    for rays among large overlapping triangles, so a version that visits in a slightly other order stays far below the
    latter.  Path records of whole passes were the same over the two trees; a tie on the way would change a path
    altogether, so a few may differ.  Shading runs the same fp32 operations in the same order."""
    if case["kind"] in ("render", "serve"):
        return {"rel": 1e-3, "max": 0.9, "differ": 1e-4}
    if case["kind"] == "shade":
        return {"rel": 1e-6, "max": 1e-4, "differ": 1e-5}
    if case["kind"] == "batch" or case.get("query"):
        return {"rel": 1e-6, "max": 1e-5, "differ": 5e-3}
    return {"rel": 1e-6, "max": 1e-5, "differ": max(2e-5, 12 / (5 * case["count"]))}


# ---------------------------------------------------------------------------
# 64-bit results
# ---------------------------------------------------------------------------
def exact(case, seed):
    if case["kind"] == "trace" and case["scene"] in ("terrain", "soup", "spheres") and case["query"] == 0:
        return _exact_trace(case, seed)
    if case["kind"] == "shade":
        return _exact_shade(case, seed)
    return None


def _exact_trace(case, seed):
    tris = {"terrain": lambda: _mesh_sizes(case)[1], "soup": lambda: case["size"],
            "spheres": lambda: max(2000, case["size"])}[case["scene"]]()
    if tris * case["count"] > _EXACT_TESTS:
        return None
    meshes = {"terrain": lambda: _terrain(case["size"]), "soup": lambda: [S.soup_scene(case["size"], seed=100)],
              "spheres": lambda: [S.sphere_grid_scene(max(2000, case["size"]), seed=101)]}[case["scene"]]()
    rays = _trace_rays(case, seed, meshes)
    p = torch.from_numpy(np.concatenate([m.verts[m.tris.astype(np.int64)] for m in meshes])).cuda().double()
    p0, e1, e2 = p[:, 0], p[:, 1] - p[:, 0], p[:, 2] - p[:, 0]
    out = torch.empty(case["count"], device="cuda", dtype=torch.float64)
    step = max(1, int(2e7 // p.shape[0]))
    for a in range(0, case["count"], step):
        r = rays[a:a + step]
        o, d = r[:, None, 0:3].double(), r[:, None, 3:6].double()
        s1 = torch.linalg.cross(d, e2[None])
        div = (s1 * e1).sum(-1)
        s = o - p0
        b1 = (s * s1).sum(-1) / div
        s2 = torch.linalg.cross(s, e1[None].expand_as(s))
        b2 = (d * s2).sum(-1) / div
        t = (e2 * s2).sum(-1) / div
        lo, hi = r[:, 6:7].double(), r[:, 7:8].double()
        ok = (b1 >= 0) & (b2 >= 0) & (1 - b1 - b2 >= 0) & (t >= lo) & (t < hi)
        best = torch.where(ok, t, math.inf).amin(1)
        out[a:a + step] = torch.where(torch.isfinite(best), best, hi[:, 0])
        if r.view(torch.int32)[:, 9].any():
            out[a:a + step][r.view(torch.int32)[:, 9] != 0] = 0.0
    return {"t": out, "record": None}


def _pcg(v):
    m = 0xFFFFFFFF
    s = (v * 747796405 + 2891336453) & m
    w = (((s >> ((s >> 28) + 4)) ^ s) * 277803737) & m
    return (w >> 22) ^ w


def _uniform(seed, pix, depth, dim):
    """The random number of (seed, pixel, depth, dimension): a 32-bit hash, its upper 24 bits."""
    h = _pcg((seed >> 32) ^ _pcg(pix ^ _pcg(depth * 16 + dim)))
    return (_pcg((seed & 0xFFFFFFFF) ^ h) >> 8).double() / 16777216.0


def _exact_shade(case, seed):
    _, tri, steps = _shade_inputs(case, seed)
    n, f8 = case["count"], torch.float64
    mats, lights = _shade_mats(seed), _area_light(3.5, 6.5, 9.9, 12.0)
    kds, les = (torch.from_numpy(mats[k].astype(np.float64)).cuda() for k in ("kd", "le"))
    lt = {k: torch.from_numpy(lights[k].astype(np.float64)).cuda() for k in ("p0", "e1", "e2", "le")}
    rr, pi_inv, two_pi = float(np.float32(0.7)), float(np.float32(0.31830988)), float(np.float32(6.2831853))
    thr = torch.ones(n, 3, device="cuda", dtype=f8)
    rad, dl = torch.zeros_like(thr), torch.zeros_like(thr)
    depth = torch.zeros(n, device="cuda", dtype=torch.long)
    alive = torch.ones(n, device="cuda", dtype=torch.bool)
    pix = torch.arange(n, device="cuda")
    sd = int(seed) % (1 << 62) + 1
    nxt = [torch.zeros(n, 9, device="cuda", dtype=f8) for _ in range(2)]
    masked = torch.tensor([0.0, 0, 0, 0, 0, 1.0, 0, 0, 0], device="cuda", dtype=f8).expand(n, 9)
    shadow = torch.zeros_like(nxt[0])
    for k, x in enumerate(steps):
        words = x["hits"].view(torch.int32)
        if k:
            free = (x["shits"].view(torch.int32)[:, 3] == -1)[:, None]
            rad = torch.where(free, rad + dl, rad)
        dl = torch.zeros_like(dl)
        live = alive & (words[:, 3] != -1)
        ray, m = x["rays"].double(), words[:, 3].long().clamp(min=0)
        kd, le = kds[m], les[m]
        v = tri[x["tri"]].double()
        nr = torch.linalg.cross(v[:, 1] - v[:, 0], v[:, 2] - v[:, 0])
        nr = nr / nr.norm(dim=1, keepdim=True)
        nr = torch.where((nr * ray[:, 3:6]).sum(1, keepdim=True) > 0, -nr, nr)
        t = torch.where(live, x["hits"][:, 0], 0.0).double()
        p = ray[:, 0:3] + ray[:, 3:6] * t[:, None]
        eps = _epsilon(p.float()).double()
        rad = torch.where((live & (depth == 0))[:, None], rad + thr * le, rad)
        u = [_uniform(sd, pix, depth, j) for j in range(6)]
        j = (u[3] * 2).long().clamp(max=1)
        su = u[4].sqrt()
        w = lt["p0"][j] + (su * (1 - u[5]))[:, None] * lt["e1"][j] + (su * u[5])[:, None] * lt["e2"][j] - p
        d2 = (w * w).sum(1)
        dist = d2.sqrt()
        wn = w / dist[:, None]
        ln = torch.linalg.cross(lt["e1"][j], lt["e2"][j])
        lnl = ln.norm(dim=1)
        cos_s, cos_l = (nr * wn).sum(1), (ln * wn).sum(1).abs() / lnl
        lit = live & (cos_s > 0) & (cos_l > 0) & (dist > 4 * eps)
        gain = cos_s * cos_l * (0.5 * lnl * 2) / d2 * pi_inv
        dl = torch.where(lit[:, None], thr * kd * lt["le"][j] * gain[:, None], dl)
        zero = torch.zeros_like(eps)
        shadow = torch.where(lit[:, None], torch.cat([p, wn, torch.stack([eps, dist - 2 * eps, zero], 1)], 1), masked)
        go = live & (depth + 1 < 8)
        roulette = depth + 1 >= 1
        go = go & (~roulette | (u[2] < rr))
        thr = torch.where((go & roulette)[:, None], thr / rr, thr)
        r, phi = u[0].sqrt(), two_pi * u[1]
        lx, ly, lz = r * torch.cos(phi), r * torch.sin(phi), (1 - u[0]).clamp(min=0).sqrt()
        sg = torch.where(nr[:, 2] >= 0, 1.0, -1.0).double()
        a = -1 / (sg + nr[:, 2])
        b = nr[:, 0] * nr[:, 1] * a
        t0 = torch.stack([1 + sg * nr[:, 0] ** 2 * a, sg * b, -sg * nr[:, 0]], 1)
        t1 = torch.stack([b, sg + nr[:, 1] ** 2 * a, -nr[:, 1]], 1)
        d = lx[:, None] * t0 + ly[:, None] * t1 + lz[:, None] * nr
        d = d / d.norm(dim=1, keepdim=True)
        thr = torch.where(go[:, None], thr * kd, thr)
        out = torch.cat([p, d, torch.stack([eps, torch.full_like(eps, math.inf), zero], 1)], 1)
        nxt[k % 2] = torch.where(go[:, None], out, masked)
        depth = torch.where(live, depth + 1, depth)
        alive = go
    return {"path": torch.cat([thr, rad, dl], 1), "path_words": None, "next": nxt[(case["steps"] - 1) % 2],
            "next_flags": None, "shadow": shadow, "shadow_flags": None}
