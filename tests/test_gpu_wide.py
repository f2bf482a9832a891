"""The walk over the four-wide nodes against the walk over the binary ones, bit for bit: a traced ray buffer
goes over the wide nodes, a counted one over the binary ones, and the wavefront engine takes the binary nodes
when their top is staged in LDS. Scenes where ties, flat boxes, rounding or the wide format's limits decide."""
import numpy as np
import pytest

from photon_amd import gpu, host
from photon_amd.types import RAY_DTYPE, Material, RenderSettings

from gpu_util import trace_on_gpu, uploaded

pytestmark = pytest.mark.gpu


def _mesh(scale=1.0, offset=0.0, twice=False, n=900, flat=False, max_leaf=0, seed=3):
    """Random small triangles, or a floor of axis-aligned ones; `twice`: every triangle again, in a second mesh."""
    rng = np.random.default_rng(seed)
    if flat:
        k = int(np.sqrt(n / 2))
        x, z = np.meshgrid(np.arange(k), np.arange(k))
        corner = np.stack([x, np.zeros_like(x), z], -1).reshape(-1, 1, 3).astype(np.float64)
        quad = np.array([[0, 0, 0], [1, 0, 0], [1, 0, 1], [0, 0, 0], [1, 0, 1], [0, 0, 1]], float)
        p = (corner + quad).reshape(-1, 3) / k * 2 - 1
    else:
        p = (rng.uniform(-1, 1, (n, 1, 3)) + rng.normal(0, 0.08, (n, 3, 3))).reshape(-1, 3)
    p = (p * scale + offset).astype(np.float32)
    s = host.Scene()
    for _ in range(2 if twice else 1):
        s.add_mesh(p, np.arange(len(p), dtype=np.int32), s.add_material(Material.default()))
    return s.build(max_leaf=max_leaf, traversal_cost=1e9 if max_leaf > 32 else 0.0), p


def _rays(points, n, seed):
    """Rays between points near the vertices `points`, many of them exactly through vertices and edges, along axes,
    from far away, and with upper limits that cut hits off; a few that are not finite."""
    rng = np.random.default_rng(seed)
    lo, hi = points.min(0), points.max(0)
    ext = np.maximum(hi - lo, 1e-6 * np.abs(hi))
    ext = np.maximum(ext, ext.max() * 1e-3)
    tri = points[: len(points) // 3 * 3].reshape(-1, 3, 3)
    t = tri[rng.integers(len(tri), size=n)].astype(np.float64)
    bary = rng.dirichlet(np.ones(3), n)
    edge = rng.random(n) < 0.25
    bary[edge, 0] = 0
    vertex = rng.random(n) < 0.15
    bary[vertex] = [0, 1, 0]
    target = (t * (bary / bary.sum(1, keepdims=True))[..., None]).sum(1)
    o = lo + ext * rng.uniform(-1.0, 2.0, (n, 3))
    far = rng.random(n) < 0.2
    o[far] = target[far] + (o - target)[far] * 10.0 ** rng.uniform(0, 6, (far.sum(), 1))
    on = rng.random(n) < 0.1
    o[on] = t[on, 0]
    d = target - o
    d /= np.maximum(np.linalg.norm(d, axis=1, keepdims=True), 1e-30)
    axis = rng.random(n) < 0.2
    k = rng.integers(3, size=n)
    unit = np.eye(3)[k] * rng.choice([-1.0, 1.0], n)[:, None]
    o[axis] = target[axis] - unit[axis] * ext[k[axis], None]
    d[axis] = unit[axis]
    d[rng.random(n) < 0.03] *= -0.0
    r = np.zeros(n, RAY_DTYPE)
    r["o"], r["d"], r["tmax"] = o, d, 1e30
    cut = rng.random(n) < 0.2
    r["tmax"][cut] = (ext.max() * 10.0 ** rng.uniform(-3, 1, cut.sum())).astype(np.float32)
    r["tmax"][:6] = [0.0, -1.0, np.nan, np.inf, 3e38, 1e-30]
    r["o"][6:9, 0] = [np.nan, 1e16, -np.inf]
    r["d"][9:13, 1] = [np.nan, 1e16, np.inf, 1e-25]
    return r


CASES = {
    "random": dict(),
    "twice": dict(twice=True, n=300),
    "floor": dict(flat=True),
    "floor-twice": dict(flat=True, twice=True, n=400),
    "tiny": dict(scale=1e-6),
    "small-far": dict(scale=1e-2, offset=1e3),
    "large": dict(scale=1e6),
    "beyond-limits": dict(scale=1e16, n=60),
    "large-leaves": dict(n=200, max_leaf=200),
    "one": dict(n=1),
    "five": dict(n=5),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_wide_hits_are_the_binary_hits(name):
    scene, points = _mesh(**CASES[name])
    r = uploaded(scene)
    rays = _rays(points, 40001, seed=len(name))
    want, _ = trace_on_gpu(r, rays, counts=True)
    got = trace_on_gpu(r, rays)
    # The bounds under rays at the tie threshold: limits set to a hit's own distance.
    hit = want["tri"] >= 0
    limited = rays.copy()
    limited["tmax"][hit] = want["t"][hit] * np.where(np.arange(hit.sum()) % 2, np.float32(1), np.float32(1 + 2**-22))
    want2, _ = trace_on_gpu(r, limited, counts=True)
    got2 = trace_on_gpu(r, limited)
    assert name in ("beyond-limits", "tiny") or hit.mean() > 0.1
    assert got.tobytes() == want.tobytes()
    assert got2.tobytes() == want2.tobytes()
    r.close()


@pytest.mark.parametrize("name", ["cornell-c1", "materials", "glass", "soup"])
def test_wide_hits_on_scenes(name):
    scene = host.Scene.spheres(24, box=20.0, alpha_fraction=0.3, seed=5).build() if name == "soup" else host.Scene.builtin(name).build()
    r = uploaded(scene)
    rays = host.camera_rays(scene.camera_view(1.0), 257, 251)
    assert trace_on_gpu(r, rays).tobytes() == trace_on_gpu(r, rays, counts=True)[0].tobytes()
    r.close()


@pytest.mark.parametrize("w,h,spp,split", [(70, 45, 3, 1), (130, 67, 4, 4)])
def test_wavefront_image_over_either_walk(w, h, spp, split):
    """Also a second upload and a light update, which write the triangles again."""
    scene = host.Scene.field(8, seed=2, env_width=64).build()
    cam, rs = scene.camera_view(w / h), RenderSettings.make(w, h, max_depth=8, rr_depth=3, seed=9)
    r = uploaded(scene, w, h, engine=gpu.ENGINE_WAVEFRONT)
    images = []
    for nodes in (0, 64, 0):
        r.set_wavefront_config(block=64, stack_depth=8, path_slots=1000, lds_nodes=nodes, sample_split=split)
        r.reset()
        r.render(cam, rs, spp)
        images.append(r.download_image())
        r.update_lights(scene)
    assert images[0].tobytes() == images[1].tobytes() == images[2].tobytes()
    r.close()


@pytest.mark.parametrize("n", [480, 900])
def test_default_and_configured_launches_alternate(n):
    """Hierarchies on either side of 512 nodes, the line up to which the queues of configured slots walk the binary nodes
    and the default launch's the wide ones: one renderer, in turns, so that each has to find its own launches again."""
    scene = _lit(n=n)
    assert (scene.desc().num_nodes > 512) == (n == 900)
    w, h, spp = 520, 512, 5  # more than 2^20 samples: the default launch runs in bounces
    cam, rs = scene.camera_view(w / h), RenderSettings.make(w, h, max_depth=6, rr_depth=3, seed=4)
    r = uploaded(scene, w, h, engine=gpu.ENGINE_WAVEFRONT)
    default, images = r.wavefront_config(), []
    for cfg in ({}, dict(path_slots=w * h * spp, sample_split=spp)) * 3:
        r.set_wavefront_config(**(cfg or {f: getattr(default, f) for f, _ in default._fields_}))
        r.reset()
        r.render(cam, rs, spp)
        images.append(gpu.copy_device_to_numpy(r.buffer_ptr(gpu.BUF_ACCUM), w * h * 16, np.float32).tobytes())
    assert len(set(images)) == 1
    r.close()


@pytest.mark.parametrize("n", [1, 129, 786431, 786432, 1000003, 1966079, 1966080, 2500007])
def test_any_hit_launches_report_the_same_hits(n):
    """Few any-hit rays run in blocks with deep stacks, more (from 786,432 on) in blocks with short ones, many (from 1,966,080
    on) in a grid with refilled lanes: all report the counting walk's hits."""
    scene = host.Scene.spheres(12, box=12.0, alpha_fraction=0.3, seed=4).build()
    r = uploaded(scene)
    rays = scene.shadow_rays(n, seed=3)
    got = trace_on_gpu(r, rays, anyhit=True)
    want, _ = trace_on_gpu(r, rays, anyhit=True, counts=True)
    assert got.tobytes() == want.tobytes()
    r.close()


def _lit(**kw):
    """A _mesh scene with light from a sky of one colour and from its first triangles, and a camera that sees it."""
    rng = np.random.default_rng(11)
    n, twice, max_leaf = kw.get("n", 300), kw.get("twice", False), kw.get("max_leaf", 0)
    p = (rng.uniform(-1, 1, (n, 1, 3)) + rng.normal(0, 0.15, (n, 3, 3))).reshape(-1, 3).astype(np.float32)
    s = host.Scene()
    dull, lamp = Material.default(), Material.default()
    dull.base_color[:], dull.metallic, dull.double_sided = (0.7, 0.6, 0.5, 1.0), 0.0, 1
    lamp.emission[:], lamp.double_sided = (8.0, 7.0, 6.0), 1
    a, b = s.add_material(dull), s.add_material(lamp)
    for _ in range(2 if twice else 1):
        s.add_mesh(p, np.arange(len(p), dtype=np.int32), a)
    q = (rng.uniform(-1.5, 1.5, (6, 1, 3)) + rng.normal(0, 0.3, (6, 3, 3))).reshape(-1, 3).astype(np.float32)
    s.add_mesh(q, np.arange(len(q), dtype=np.int32), b)
    s.set_env_color((0.3, 0.4, 0.5), 1.0)
    s.set_camera((0.2, 0.3, 4.0), (0, 0, 0), (0, 1, 0), 45.0)
    return s.build(max_leaf=max_leaf, traversal_cost=1e9 if max_leaf > 32 else 0.0)


@pytest.mark.parametrize("kw", [dict(max_leaf=100), dict(twice=True), dict(), dict(twice=True, n=900), dict(n=900)],
                         ids=["no-wide-nodes", "every-triangle-twice", "plain", "every-triangle-twice-900", "plain-900"])
def test_every_path_renders_the_same_image(kw):
    """One image through every kernel that traces paths: the per-pixel one, a sample per lane, bounces over few slots,
    bounces that end one path per thread, the binary nodes' top staged in LDS, and serving among other jobs. Leaves of
    100 triangles have no wide nodes: all of it walks the binary ones. Where every triangle is there twice, every hit is a
    tie that the wide walk leaves to the binary one, in the queues' second pass too. Of 900 triangles a hierarchy has more
    than the 512 nodes up to which the queues of serving and of configured slots walk the binary ones."""
    from oracle import oracle_py

    scene = _lit(**kw)
    w, h, spp = 90, 61, 4
    rs, cam = RenderSettings.make(w, h, max_depth=6, rr_depth=3, seed=3), scene.camera_view(w / h)
    images = {}

    def accum(r):
        return gpu.copy_device_to_numpy(r.buffer_ptr(gpu.BUF_ACCUM), w * h * 16, np.float32).tobytes()

    for name, engine, cfg in (("per-pixel", gpu.ENGINE_MEGAKERNEL, {}), ("direct", gpu.ENGINE_WAVEFRONT, {}),
                              ("bounces", gpu.ENGINE_WAVEFRONT, dict(path_slots=1000, finish_percent=0)),
                              ("finished", gpu.ENGINE_WAVEFRONT, dict(path_slots=3000, finish_percent=100)),
                              ("samples", gpu.ENGINE_WAVEFRONT, dict(path_slots=5000, sample_split=4, refill_lanes=1, finish_percent=0)),
                              ("top", gpu.ENGINE_WAVEFRONT, dict(path_slots=1000, lds_nodes=16, finish_percent=0))):
        r = uploaded(scene, w, h, engine=engine)
        if cfg:
            r.set_wavefront_config(**cfg)
        r.render(cam, rs, spp)
        images[name] = accum(r)
        if name == "per-pixel":
            image = r.download_image()
            ref = oracle_py.render(scene.desc(), cam, rs, spp)
            assert np.mean(np.all(np.abs(image - ref) <= 1e-3 * np.abs(ref) + 1e-6, axis=2)) >= 0.999
            assert image.mean() > 0.05
        r.close()
    for name in images:
        assert images[name] == images["per-pixel"], name
    srv = gpu.Server(path_slots=2000, express_slots=-1, min_items=1)
    other = host.Scene.builtin("materials").build()
    a, b = srv.add_scene(scene), srv.add_scene(other)
    jobs = [srv.submit(a, w, h, spp, cam, max_depth=6, seed=3), srv.submit(b, 64, 40, 3, other.camera_view(1.6), max_depth=6, seed=9)]
    srv.run_until_idle()
    assert srv.result(jobs[0]).tobytes() == image.tobytes()
    alone = gpu.Server(path_slots=2000, express_slots=-1, min_items=1)
    j = alone.submit(alone.add_scene(other), 64, 40, 3, other.camera_view(1.6), max_depth=6, seed=9)
    alone.run_until_idle()
    assert alone.result(j).tobytes() == srv.result(jobs[1]).tobytes()
    alone.close()
    srv.close()


@pytest.mark.parametrize("kw", [dict(max_leaf=100), dict(twice=True)], ids=["no-wide-nodes", "every-triangle-twice"])
def test_real_time_samples_of_scenes_left_to_the_binary_nodes(kw):
    """The one-sample G-buffer kernels: the compact sample's colour is the first sample of the render, and the denoised
    frame traces the same one."""
    scene = _lit(**kw)
    w, h = 75, 50
    rs, cam = RenderSettings.make(w, h, max_depth=5, rr_depth=3, seed=6), scene.camera_view(w / h)
    r = uploaded(scene, w, h)
    r.render(cam, rs, 1)
    first = r.download_image()
    r.close()
    r = uploaded(scene, w, h)
    g = gpu.CompactGBuffer(w, h)
    r.sample_compact(cam, rs, g)
    assert g.planes["color"].numpy(np.float32, (h, w, 3)).tobytes() == first.tobytes()
    r.close()
    r = uploaded(scene, w, h)
    r.render_denoised(cam, cam, rs)
    colour = gpu.copy_device_to_numpy(r.buffer_ptr(gpu.BUF_COLOR), w * h * 16, np.float32, (h, w, 4))
    assert np.ascontiguousarray(colour[..., :3]).tobytes() == first.tobytes()
    r.close()
