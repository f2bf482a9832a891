"""The work that users of the renderer have it do, case by case, for timing one version of the library
against another: ray buffers, progressive renders, real-time frames, the denoiser, scene builds and the
serving loop, from the smallest call to the 1080p render of a million triangles.

`listed()` names the cases, `draw(rng)` gives another one of the same ranges, `prepare` makes what a
program holds before the call (scene uploaded, buffers, views of them), `run` is one pass through the
public entry points of `photon_amd`, `work` the bytes and operations a pass cannot do without,
`tolerance` how far another correct implementation may be, and `exact` the same outputs in 64 bits where
they have such a value.
"""
import ctypes
import math
import random

import numpy as np
import torch

from photon_amd import gpu, host
from photon_amd.types import CameraView, RenderSettings, SvgfSettings

# The launch that the wavefront engine's tuner settles on for the 1080p, 64-sample render of the
# million-triangle field; a program that renders that view again and again keeps it.
TUNED = dict(block=128, stack_depth=8, path_slots=31104000, blocks_per_cu=16, sort_materials=1, use_graph=1, graph_iterations=5,
             refill_lanes=16, lds_nodes=0, ray_bins=1, xcd_parts=1, sample_split=64, finish_percent=10)


def listed():
    return [
        # A picking or visibility query: a few thousand rays into a small room. Launch latency.
        dict(name="rays-cornell-4097", kind="rays", scene="cornell", spheres=0, rays=4097, anyhit=False),
        # Ambient-occlusion-like batches into a small scene, a count that fills no whole block.
        dict(name="rays-soup16k-66001", kind="rays", scene="soup", spheres=16, rays=66001, anyhit=False),
        # The traversal workload: 2048 x 2048 camera rays into 262,144 triangles, a tenth alpha-masked.
        dict(name="rays-soup262k-4m", kind="rays", scene="soup-alpha", spheres=256, rays=2048 * 2048, anyhit=False),
        # Its shadow rays, a million and three.
        dict(name="shadow-soup262k-1m", kind="rays", scene="soup-alpha", spheres=256, rays=1000003, anyhit=True),
        # A thumbnail with the default launch: few paths, many short launches.
        dict(name="render-cornell-64", kind="render", scene="cornell", spheres=0, width=64, height=64, spp=4, depth=8, tuned=False),
        # A preview of metals, plastics and glass under an HDR sky at an odd size, default launch.
        dict(name="render-materials-853", kind="render", scene="materials", spheres=0, width=853, height=479, spp=8, depth=8, tuned=False),
        # The final render: 1080p, 64 samples, 1,048,578 triangles, the launch kept from tuning.
        dict(name="render-field1m-1080p", kind="render", scene="field", spheres=1024, width=1920, height=1080, spp=64, depth=16, tuned=True),
        # A real-time frame: one sample per pixel into the compact G-buffer, then the denoiser on it.
        dict(name="frame-field1m-1600", kind="frame", scene="field", spheres=1024, width=1600, height=900, depth=16),
        # The viewer's frame at an odd window size: traced, denoised and tone-mapped for display.
        dict(name="denoised-field64-853", kind="denoised", scene="field", spheres=64, width=853, height=481, depth=8),
        # The denoiser alone on a caller's float4 G-buffer.
        dict(name="svgf-1600", kind="svgf", width=1600, height=900),
        # A scene edited while the program runs: its hierarchy built on the device.
        dict(name="bvh-65k", kind="bvh", spheres=64),
        # Jobs of mixed size and scene through the serving loop, from submission to their images.
        dict(name="serve-mixed", kind="serve", spheres=64, jobs=8, spp=16),
    ]


def draw(rng):
    def log_int(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    kind = rng.choice(["rays", "rays", "rays", "render", "render", "frame", "denoised", "svgf", "svgf", "bvh"])
    if kind == "rays":
        scene = rng.choice(["cornell", "soup", "soup-alpha"])
        return dict(kind=kind, scene=scene, spheres=0 if scene == "cornell" else log_int(4, 256), rays=log_int(2000, 4000000),
                    anyhit=scene != "cornell" and rng.random() < 0.5)
    if kind == "render":
        scene = rng.choice(["cornell", "materials", "glass", "field"])
        return dict(kind=kind, scene=scene, spheres=log_int(8, 256) if scene == "field" else 0, width=log_int(48, 1280), height=log_int(48, 720),
                    spp=rng.choice([1, 2, 3, 4, 5, 8, 12, 16]), depth=rng.choice([4, 8, 16]), tuned=False)
    if kind in ("frame", "denoised"):
        return dict(kind=kind, scene="field", spheres=log_int(16, 512), width=log_int(200, 1600), height=log_int(120, 900), depth=rng.choice([4, 8, 16]))
    if kind == "svgf":
        return dict(kind=kind, width=log_int(160, 1920), height=log_int(90, 1080))
    return dict(kind=kind, spheres=log_int(4, 250))


# ---- scenes and buffers ------------------------------------------------------------------------------
def _scene(name, spheres, seed):
    if name == "cornell":
        return host.Scene.builtin("cornell-c1").build()
    if name in ("materials", "glass"):
        return host.Scene.builtin(name).build()
    if name == "soup":
        return host.Scene.spheres(spheres, box=100.0 * (spheres / 256.0) ** (1.0 / 3.0), seed=1 + seed).build()
    if name == "soup-alpha":
        return host.Scene.spheres(spheres, box=100.0 * (spheres / 256.0) ** (1.0 / 3.0), alpha_fraction=0.1, seed=1 + seed).build()
    return host.Scene.field(spheres, seed=1 + seed, env_width=2048 if spheres >= 512 else 512).build()


def _triangles(case):
    name = case.get("scene", "soup")
    return {"cornell": 36, "materials": 39746, "glass": 18062}.get(name, 1024 * case.get("spheres", 0) + 2)


class _DevicePlane:
    """Device memory of the library, for torch.as_tensor. The tensor keeps this object, and with it the
    library's object that owns the memory."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = dict(data=(int(ptr), False), shape=tuple(shape), typestr=typestr, version=2)


def _plane(owner, ptr, shape, typestr="<f4"):
    ptr = ptr.value if hasattr(ptr, "value") else ptr
    t = torch.as_tensor(_DevicePlane(owner, ptr, shape, typestr), device="cuda")
    if t.data_ptr() != ptr:
        raise RuntimeError("the tensor is a copy of the plane")
    return t


def _ptr(tensor):
    return ctypes.c_void_p(tensor.data_ptr())


def _views(scene, aspect, first, count, step=0.5):
    """`count` views of the scene's camera turned about its target, `step` degrees apart, from `first` degrees on."""
    c = scene.camera()
    t = c["target"]
    b = [c["position"][i] - t[i] for i in range(3)]
    views = []
    for k in range(count):
        a = math.radians(first + step * k)
        p = (t[0] + math.cos(a) * b[0] + math.sin(a) * b[2], t[1] + b[1], t[2] - math.sin(a) * b[0] + math.cos(a) * b[2])
        scene.set_camera(p, t, c["up"], c["vfov"])
        views.append(scene.camera_view(aspect))
    scene.set_camera(c["position"], t, c["up"], c["vfov"])
    return views


class _State:
    pass


# ---- ray buffers -----------------------------------------------------------------------------------------
def _ray_inputs(case, seed):
    scene = _scene(case["scene"], case["spheres"], seed)
    n = case["rays"]
    if case["anyhit"]:
        rays = scene.shadow_rays(n, seed=2 + seed)
    else:
        side = int(math.ceil(math.sqrt(n)))
        view = _views(scene, 1.0, (seed % 41) * 0.25, 1)[0]
        rays = host.camera_rays(view, side, side)[:n]
    return scene, np.ascontiguousarray(rays)


def _prepare_rays(case, seed):
    scene, rays = _ray_inputs(case, seed)
    s = _State()
    s.renderer = gpu.GpuRenderer()
    ok, err = s.renderer.upload(scene)
    if not ok:
        raise RuntimeError(err)
    s.n, s.anyhit = len(rays), case["anyhit"]
    s.rays = torch.from_numpy(rays.view(np.float32).reshape(-1, 7)).cuda()
    s.hits = torch.zeros((s.n, 4), dtype=torch.float32, device="cuda")
    s.out = dict(t=s.hits[:, 0], tri=s.hits.view(torch.int32)[:, 1], uv=s.hits[:, 2:])
    s.rays_ptr, s.hits_ptr = _ptr(s.rays), _ptr(s.hits)
    return s


def _run_rays(s):
    s.renderer.trace(s.rays_ptr, s.n, s.hits_ptr, anyhit=s.anyhit)
    return s.out


def _exact_rays(case, seed):
    """Every ray against every triangle in 64 bits (closest hit, scenes without alpha masks)."""
    if case["anyhit"] or case["scene"] == "soup-alpha" or case["rays"] * _triangles(case) > 2.5e9:
        return None
    scene, rays = _ray_inputs(case, seed)
    d = scene.desc()
    raw = np.frombuffer((ctypes.c_uint8 * (48 * d.num_tris)).from_address(ctypes.addressof(d.tris.contents)), np.float32).reshape(-1, 12)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    tri = torch.from_numpy(raw.astype(np.float64)).to(dev)
    v0, e1, e2 = tri[:, 0:3], tri[:, 4:7], tri[:, 8:11]
    ray = torch.from_numpy(rays.view(np.float32).reshape(-1, 7).astype(np.float64)).to(dev)
    t_out = torch.full((len(rays),), 1e30, dtype=torch.float64, device=dev)
    uv_out = torch.zeros((len(rays), 2), dtype=torch.float64, device=dev)
    chunk = max(1, min(len(rays), 20000000 // max(1, len(tri))))

    def dot(a, b):
        return (a * b).sum(-1)

    for k in range(0, len(rays), chunk):
        o, dr, tmax = ray[k:k + chunk, None, 0:3], ray[k:k + chunk, None, 3:6], ray[k:k + chunk, 6]
        p = torch.linalg.cross(dr.expand(-1, len(tri), -1), e2.expand(o.shape[0], -1, -1))
        det = dot(e1, p)
        inv = 1.0 / det
        sv = o - v0
        u = dot(sv, p) * inv
        q = torch.linalg.cross(sv, e1.expand(o.shape[0], -1, -1))
        v = dot(dr, q) * inv
        t = dot(e2, q) * inv
        t = torch.where((det.abs() >= 1e-14) & (u >= 0) & (v >= 0) & (u + v <= 1) & (t > 0) & (t < tmax[:, None]), t, math.inf)
        best, at = t.min(dim=1)
        hit = torch.isfinite(best)
        t_out[k:k + chunk][hit] = best[hit]
        rows = torch.arange(len(at), device=dev)
        uv_out[k:k + chunk][hit] = torch.stack([u[rows, at], v[rows, at]], dim=1)[hit]
    return dict(t=t_out, tri=None, uv=uv_out)


# ---- progressive renders -----------------------------------------------------------------------------------
def _prepare_render(case, seed):
    s = _State()
    w, h = case["width"], case["height"]
    scene = _scene(case["scene"], case["spheres"], seed)
    s.renderer = gpu.GpuRenderer()
    ok, err = s.renderer.upload(scene)
    if not ok:
        raise RuntimeError(err)
    s.renderer.resize(w, h)
    if case["tuned"]:
        s.renderer.set_wavefront_config(**TUNED)
    s.camera = _views(scene, w / h, (seed % 41) * 0.25, 1)[0]
    s.settings = RenderSettings.make(w, h, max_depth=case["depth"], rr_depth=3, seed=1 + seed % 100003)
    s.spp = case["spp"]
    s.out = [_plane(s.renderer, s.renderer.buffer_ptr(b), (h, w, 4)) for b in (gpu.BUF_ACCUM, gpu.BUF_ALBEDO, gpu.BUF_NORMAL_DEPTH)]
    return s


def _run_render(s):
    s.renderer.reset()
    s.renderer.render(s.camera, s.settings, s.spp)
    return s.out


# ---- real-time frames ------------------------------------------------------------------------------------------
FRAMES = 8


def _prepare_frame(case, seed):
    s = _State()
    w, h = case["width"], case["height"]
    scene = _scene(case["scene"], case["spheres"], seed)
    s.renderer = gpu.GpuRenderer()
    ok, err = s.renderer.upload(scene)
    if not ok:
        raise RuntimeError(err)
    s.renderer.resize(w, h)
    s.views = _views(scene, w / h, (seed % 41) * 0.25, FRAMES)
    s.views += s.views[-2:0:-1]  # there and back again, half a degree a frame
    s.settings = RenderSettings.make(w, h, max_depth=case["depth"], rr_depth=3, seed=1 + seed % 100003)
    s.svgf_settings = SvgfSettings.make()
    s.frame = 0
    if case["kind"] == "denoised":
        s.out = dict(image=_plane(s.renderer, s.renderer.buffer_ptr(gpu.BUF_DENOISED), (h, w, 4)),
                     display=_plane(s.renderer, s.renderer.display_buffer(), (h, w, 4), "|u1"))
        return s
    s.gbuffer = gpu.CompactGBuffer(w, h)
    s.svgf = gpu.Svgf()
    s.svgf.resize(w, h)
    s.image = torch.zeros((h, w, 4), dtype=torch.float32, device="cuda")
    s.image_ptr = _ptr(s.image)
    s.out = dict(image=s.image)
    for name, dtype, k in gpu.CompactGBuffer.PLANES:
        s.out[name] = _plane(s.gbuffer.planes[name], s.gbuffer.planes[name].ptr, (h, w, k), "<f4" if dtype is np.float32 else "<i4")
    return s


def _next_views(s):
    cur, prev = s.views[s.frame % len(s.views)], s.views[max(0, s.frame - 1) % len(s.views)]
    s.frame += 1
    return cur, prev


def _run_frame(s):
    cur, prev = _next_views(s)
    s.renderer.sample_compact(cur, s.settings, s.gbuffer)
    s.svgf.run_compact(s.gbuffer, cur, prev, s.svgf_settings, s.image_ptr)
    return s.out


def _run_denoised(s):
    cur, prev = _next_views(s)
    s.renderer.render_denoised(cur, prev, s.settings, s.svgf_settings)
    s.renderer.display(s.settings)
    return s.out


# ---- the denoiser on a caller's planes ------------------------------------------------------------------------
# Frames before the timed one: a settled history. (The denoiser treats histories below four frames
# apart; a still view reaches four everywhere at once, up to rounding, and what one rounding decides there
# fades by a fifth a frame.)
WARM_FRAMES = 24


def _orbit_camera(w, h, degrees):
    a = math.radians(degrees)
    eye, aim = np.array([9.0 * math.sin(a), 4.0, 9.0 * math.cos(a)]), np.array([0.0, 1.0, 0.0])
    f = aim - eye
    f /= np.linalg.norm(f)
    r = np.cross(f, [0.0, 1.0, 0.0])
    r /= np.linalg.norm(r)
    c = CameraView()
    c.position[:], c.forward[:], c.right[:], c.up[:] = eye, f, r, np.cross(r, f)
    c.tan_half_fov, c.aspect, c.aperture, c.focus_distance = math.tan(math.radians(22.5)), w / h, 0.0, 1.0
    return c


def _gbuffer(w, h, seed, frame, dev):
    """A frame of spheres over a floor under a sky, one noisy sample per pixel: colour, albedo,
    normal+depth, position+material, emission, four floats per pixel each."""
    cam = _orbit_camera(w, h, (seed % 41) * 0.25 + 0.5 * frame)
    f8 = dict(dtype=torch.float64, device=dev)
    rnd = random.Random(seed)
    balls = [([rnd.uniform(-5, 5), rnd.uniform(0.3, 1.6), rnd.uniform(-5, 5)], rnd.uniform(0.3, 1.2), [rnd.uniform(0.1, 0.9) for _ in range(3)])
             for _ in range(14)]
    x = (torch.arange(w, **f8) + 0.5) / w * 2 - 1
    y = 1 - (torch.arange(h, **f8) + 0.5) / h * 2
    vec = lambda a: torch.tensor(list(a), **f8)  # noqa: E731
    o = vec(cam.position)
    d = vec(cam.forward) + vec(cam.right) * (x * cam.tan_half_fov * cam.aspect)[None, :, None] + vec(cam.up) * (y * cam.tan_half_fov)[:, None, None]
    d = d / d.norm(dim=-1, keepdim=True)
    depth = torch.where(d[..., 1] < -1e-6, -o[1] / d[..., 1].clamp(max=-1e-6), torch.full((h, w), math.inf, **f8))
    depth = torch.where(depth > 60, torch.full_like(depth, math.inf), depth)
    mat = torch.where(torch.isfinite(depth), 0.0, -1.0).to(torch.float64)
    normal = vec([0, 1, 0]).expand(h, w, 3).clone()
    albedo = vec([0.5, 0.5, 0.45]).expand(h, w, 3).clone()
    for k, (c, r, a) in enumerate(balls):
        oc = o - vec(c)
        b = (d * oc).sum(-1)
        disc = b * b - (oc.dot(oc) - r * r)
        t = -b - disc.clamp(min=0).sqrt()
        near = (disc > 0) & (t > 0) & (t < depth)
        depth = torch.where(near, t, depth)
        mat = torch.where(near, float(k + 1), mat)
        normal = torch.where(near[..., None], (o + d * t[..., None] - vec(c)) / r, normal)
        albedo = torch.where(near[..., None], vec(a), albedo)
    hit = mat >= 0
    depth = torch.where(hit, depth, 0.0)
    position = torch.where(hit[..., None], o + d * depth[..., None], o + d * 1e4)
    normal = torch.where(hit[..., None], normal, -d)
    albedo = torch.where(hit[..., None], albedo, 1.0)
    emission = torch.zeros(h, w, 3, **f8)
    emission[mat == 3] = 2.0
    g = torch.Generator(device=dev).manual_seed(seed * 1009 + frame)
    light = (0.2 + 0.8 * (normal * vec([0.5, 0.7, 0.5])).sum(-1).clamp(min=0)) * (torch.rand(h, w, generator=g, **f8) < 0.5) * 2
    light = light * (-torch.log1p(-torch.rand(h, w, generator=g, **f8) * 0.9999))
    colour = torch.where(hit[..., None], albedo * light[..., None] + emission, 0.2 + 0.8 * d[..., 1:2].clamp(min=0).expand(h, w, 3))
    emission = torch.where(hit[..., None], emission, colour)
    one = torch.ones(h, w, 1, **f8)
    planes = [torch.cat([colour, one], -1), torch.cat([albedo, one], -1), torch.cat([normal, depth[..., None]], -1),
              torch.cat([position, mat[..., None]], -1), torch.cat([emission, one], -1)]
    return cam, [p.float().contiguous() for p in planes]


def _prepare_svgf(case, seed):
    s = _State()
    w, h = case["width"], case["height"]
    s.svgf = gpu.Svgf()
    s.svgf.resize(w, h)
    s.settings = SvgfSettings.make()
    s.image = torch.zeros((h, w, 4), dtype=torch.float32, device="cuda")
    s.image_ptr = _ptr(s.image)
    prev = None
    for k in range(WARM_FRAMES + 1):
        cam, s.planes = _gbuffer(w, h, seed, k, "cuda")
        s.previous = prev or cam
        prev = cam
        s.pointers = [_ptr(p) for p in s.planes]
        torch.cuda.synchronize()
        if k < WARM_FRAMES:
            s.svgf.run(*s.pointers, s.previous, s.settings, s.image_ptr)
    s.out = [s.image, _plane(s.svgf, s.svgf.variance_buffer(), (h, w, 4))]
    return s


def _run_svgf(s):
    s.svgf.run(*s.pointers, s.previous, s.settings, s.image_ptr)
    return s.out


def _lum(c):
    return 0.2126 * c[..., 0] + 0.7152 * c[..., 1] + 0.0722 * c[..., 2]


def _shifted(a, dy, dx, clamp=False):
    """a[y + dy, x + dx] and whether that lies in the image (clamped to it otherwise)."""
    h, w = a.shape[:2]
    yy, xx = torch.arange(h, device=a.device) + dy, torch.arange(w, device=a.device) + dx
    inside = ((yy >= 0) & (yy < h))[:, None] & ((xx >= 0) & (xx < w))[None, :]
    return a[yy.clamp(0, h - 1)][:, xx.clamp(0, w - 1)], inside


def _exact_svgf(case, seed):
    """The denoiser in 64 bits: temporal accumulation, variance, five a-trous passes, remodulation."""
    w, h = case["width"], case["height"]
    st = SvgfSettings.make()
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    hist, prev, out = None, None, None
    for frame in range(WARM_FRAMES + 1):
        cam, planes = _gbuffer(w, h, seed, frame, dev)
        colour, albedo, nd, pos, emission = [p.double() for p in planes]
        mat, n, z = pos[..., 3], nd[..., :3], nd[..., 3]
        cur = (colour - emission)[..., :3].clamp(min=0) / albedo[..., :3].clamp(min=1e-3)
        lum = _lum(cur)
        hc, hm, hl, ws = torch.zeros_like(cur), torch.zeros(h, w, 2, dtype=torch.float64, device=dev), torch.zeros_like(lum), torch.zeros_like(lum)
        if hist is not None:
            v = lambda a: torch.tensor(list(a), dtype=torch.float64, device=dev)  # noqa: E731
            rel = pos[..., :3] - v(prev.position)
            zc = (rel * v(prev.forward)).sum(-1)
            ok = (zc > 1e-4) & (mat >= 0)
            zs = torch.where(ok, zc, 1.0)
            px = ((rel * v(prev.right)).sum(-1) / (zs * prev.tan_half_fov * prev.aspect) + 1) * 0.5 * w - 0.5
            py = (1 - (rel * v(prev.up)).sum(-1) / (zs * prev.tan_half_fov)) * 0.5 * h - 0.5
            dist = rel.norm(dim=-1)
            px, py = px.clamp(-1e6, 1e6), py.clamp(-1e6, 1e6)
            x0, y0 = px.floor(), py.floor()
            fx, fy = px - x0, py - y0
            for k in range(4):
                xx, yy = (x0 + (k & 1)).long(), (y0 + (k >> 1)).long()
                take = ok & (xx >= 0) & (yy >= 0) & (xx < w) & (yy < h)
                j = yy.clamp(0, h - 1) * w + xx.clamp(0, w - 1)
                p_il, p_m, p_nd, p_mat = [a.reshape(h * w, -1)[j.reshape(-1)].reshape(h, w, -1) for a in hist]
                take &= (p_mat[..., 0] == mat) & ((p_nd[..., 3] - dist).abs() <= 0.05 * dist + 0.01) & ((p_nd[..., :3] * n).sum(-1) >= 0.9)
                bw = torch.where(take, (fx if k & 1 else 1 - fx) * (fy if k >> 1 else 1 - fy), 0.0)
                hc, hm, hl, ws = hc + p_il[..., :3] * bw[..., None], hm + p_m * bw[..., None], hl + p_il[..., 3] * bw, ws + bw
        have = ws > 1e-3
        wd = torch.where(have, ws, 1.0)
        length = torch.where(have, (hl / wd + 1).clamp(max=64), 1.0)
        ac, am = (1 / length).clamp(min=st.alpha_color), (1 / length).clamp(min=st.alpha_moments)
        hc, hm = hc / wd[..., None], hm / wd[..., None]
        c = torch.where(have[..., None], hc + (cur - hc) * ac[..., None], cur)
        now = torch.stack([lum, lum * lum], -1)
        m = torch.where(have[..., None], hm + (now - hm) * am[..., None], now)
        var = (m[..., 1] - m[..., 0] ** 2).clamp(min=0)
        # Short histories: the 7x7 estimate.
        acc, am1, asum = torch.zeros_like(c), torch.zeros_like(m), torch.zeros_like(var)
        for dy in range(-3, 4):
            for dx in range(-3, 4):
                t_nd, inside = _shifted(nd, dy, dx)
                t_mat, _ = _shifted(mat, dy, dx)
                wt = (n * t_nd[..., :3]).sum(-1).clamp(min=0) ** st.phi_normal * torch.exp(-(t_nd[..., 3] - z).abs() / (0.05 * z + 1e-3))
                wt = torch.where(inside & (t_mat == mat), wt, 0.0)
                acc, am1, asum = acc + _shifted(c, dy, dx)[0] * wt[..., None], am1 + _shifted(m, dy, dx)[0] * wt[..., None], asum + wt
        short = (length < 4) & (mat >= 0) & (asum > 0)
        sd = torch.where(asum > 0, asum, 1.0)
        var = torch.where(short, (am1[..., 1] / sd - (am1[..., 0] / sd) ** 2).clamp(min=0) * (4 / length), var)
        plane = torch.cat([torch.where(short[..., None], acc / sd[..., None], c), var[..., None]], -1)
        kernel, kept = (3 / 8, 1 / 4, 1 / 16), None
        for it in range(st.atrous_iterations):
            step = 1 << it
            pv = torch.zeros_like(var)
            for dy in (-1, 0, 1):
                for dx in (-1, 0, 1):
                    pv = pv + _shifted(plane[..., 3], dy, dx)[0] * (0.25, 0.125, 0.0625)[abs(dx) + abs(dy)]
            grad = 0.5 * torch.maximum((_shifted(z, 0, 1)[0] - _shifted(z, 0, -1)[0]).abs(), (_shifted(z, 1, 0)[0] - _shifted(z, -1, 0)[0]).abs())
            l0, sigma = _lum(plane), st.phi_color * pv.clamp(min=0).sqrt() + 1e-4
            acc, vs, asum = torch.zeros_like(c), torch.zeros_like(var), torch.zeros_like(var)
            for dy in range(-2, 3):
                for dx in range(-2, 3):
                    t, inside = _shifted(plane, dy * step, dx * step)
                    t_nd, t_mat = _shifted(nd, dy * step, dx * step)[0], _shifted(mat, dy * step, dx * step)[0]
                    wt = (n * t_nd[..., :3]).sum(-1).clamp(min=0) ** st.phi_normal
                    wt = wt * torch.exp(-(t_nd[..., 3] - z).abs() / (st.phi_depth * grad * math.hypot(dx, dy) * step + 1e-3 * z + 1e-4))
                    wt = wt * torch.exp(-(_lum(t) - l0).abs() / sigma) * (kernel[abs(dx)] * kernel[abs(dy)])
                    wt = torch.where(inside & (t_mat == mat), wt, 0.0)
                    acc, vs, asum = acc + t[..., :3] * wt[..., None], vs + t[..., 3] * wt * wt, asum + wt
            use = (mat >= 0) & (asum > 0)
            sd = torch.where(asum > 0, asum, 1.0)
            plane = torch.where(use[..., None], torch.cat([acc / sd[..., None], (vs / sd ** 2)[..., None]], -1), plane)
            if it == 0:
                hist = [torch.cat([plane[..., :3], length[..., None]], -1), m, nd, mat[..., None]]
            if it == st.atrous_iterations - 2:
                kept = plane
        image = torch.where((mat >= 0)[..., None], plane[..., :3] * albedo[..., :3].clamp(min=1e-3) + emission[..., :3], colour[..., :3])
        out = [torch.cat([image, torch.ones(h, w, 1, dtype=torch.float64, device=dev)], -1), kept]
        prev = cam
    return out


# ---- scene builds ------------------------------------------------------------------------------------------
def _prepare_bvh(case, seed):
    s = _State()
    raw = host.Scene.spheres(case["spheres"], box=100.0, seed=1 + seed)
    r = raw.raw()
    s.positions = np.ctypeslib.as_array(r.positions, (r.num_vertices * 3,)).reshape(-1, 3).copy()
    s.indices = np.ctypeslib.as_array(r.indices, (r.num_tris * 3,)).reshape(-1, 3).copy()
    return s


def _run_bvh(s):
    nodes, order, _ = gpu.bvh_build(s.positions, s.indices)
    # All the room that the call gives the nodes, of which it uses the front: the same shape for any input.
    whole = nodes if nodes.base is None else nodes.base
    return [whole.view(np.int32).reshape(-1, 16), order]


# ---- serving -----------------------------------------------------------------------------------------------
JOB_SIZES = ((256, 256), (512, 512), (1280, 720), (640, 361))
JOB_DEPTHS = (4, 8, 16)


def _job_spp(case, k):
    return max(1, case["spp"] >> (k % 3))


def _prepare_serve(case, seed):
    s = _State()
    s.server = gpu.Server()
    scenes = [_scene("cornell", 0, seed), _scene("soup-alpha", case["spheres"], seed), _scene("field", case["spheres"], seed)]
    ids = [s.server.add_scene(x) for x in scenes]
    rnd = random.Random(seed)
    s.jobs = []
    for k in range(case["jobs"]):
        w, h = JOB_SIZES[k % len(JOB_SIZES)]
        which = k % 3
        s.jobs.append((ids[which], w, h, _job_spp(case, k), scenes[which].camera_view(w / h),
                       dict(max_depth=JOB_DEPTHS[k % 3], rr_depth=3, seed=rnd.randrange(1 << 31))))
    return s


def _run_serve(s):
    ids = [s.server.submit(*job[:5], **job[5]) for job in s.jobs]
    s.server.run_until_idle()
    return [s.server.result(i) for i in ids]


_KINDS = {
    "rays": (_prepare_rays, _run_rays),
    "render": (_prepare_render, _run_render),
    "frame": (_prepare_frame, _run_frame),
    "denoised": (_prepare_frame, _run_denoised),
    "svgf": (_prepare_svgf, _run_svgf),
    "bvh": (_prepare_bvh, _run_bvh),
    "serve": (_prepare_serve, _run_serve),
}


def prepare(case, seed):
    s = _KINDS[case["kind"]][0](case, seed)
    s.kind = case["kind"]
    return s


def run(state):
    return _KINDS[state.kind][1](state)


def exact(case, seed):
    """Paths follow random decisions that a change of rounding sends elsewhere, and hierarchies are whole
    numbers: those outputs have no 64-bit value. Ray hits and the denoiser do."""
    if case["kind"] == "rays":
        return _exact_rays(case, seed)
    if case["kind"] == "svgf":
        return _exact_svgf(case, seed)
    return None


# Operations that a ray cannot do without: two slab tests (18 each) a level of a balanced tree over
# leaves of four triangles, and two triangle tests (45 each). A path vertex: about 300.
def _ray_flops(tris):
    return 36.0 * max(1.0, math.log2(max(2, tris) / 4.0)) + 90.0


def _scene_bytes(tris):
    """Nodes (64 B, about one for two triangles), triangles (48), indices (12) and half a vertex (32) each."""
    return tris * (32 + 48 + 12 + 16)


def _paths(case, samples):
    """A sample is a camera ray, and in these scenes about one more vertex with its shadow ray."""
    return samples * (2.3 * _ray_flops(_triangles(case)) + 300.0)


def work(case):
    kind, tris = case["kind"], _triangles(case)
    if kind == "rays":
        return {"bytes": case["rays"] * 44 + min(case["rays"] * 400, tris * 80), "flops": case["rays"] * _ray_flops(tris)}
    if kind == "bvh":
        # Positions and indices in, nodes and order out; every triangle is binned once a level on three axes.
        return {"bytes": tris * (12 + 6 + 38 + 4), "flops": tris * math.log2(tris) * 30.0}
    if kind == "serve":
        samples = sum(w * h * _job_spp(case, k) for k in range(case["jobs"]) for w, h in [JOB_SIZES[k % len(JOB_SIZES)]])
        return {"bytes": 3 * _scene_bytes(tris) + samples, "flops": _paths(dict(case, scene="field"), samples)}
    pixels = case["width"] * case["height"]
    if kind == "render":
        return {"bytes": _scene_bytes(tris) + pixels * 48, "flops": _paths(case, pixels * case["spp"])}
    # The denoiser reads five planes and four of history, writes four of history and its image, and filters 25 taps
    # of about 30 operations five times; between passes a frame fits the caches.
    svgf = {"bytes": pixels * 16 * 14, "flops": pixels * 25 * 30 * 5.0}
    if kind == "svgf":
        return svgf
    return {"bytes": svgf["bytes"] + _scene_bytes(tris), "flops": svgf["flops"] + _paths(case, pixels)}


def tolerance(case):
    kind = case["kind"]
    if kind == "bvh":
        return "exact"
    if kind == "rays":
        # Barycentrics in 32 bits are up to 2e-5 from those in 64; the triangle may differ where two tie.
        return {"rel": 8e-5, "differ": 1e-5}
    if kind == "svgf":
        # 1.2e-4 (image) and 4e-4 (variance) from 64 bits: see WARM_FRAMES.
        return {"rel": 1e-3, "max": 0.05}
    if kind == "render" or kind == "serve":
        # The same paths computed on the CPU, whose last bits send a few of them elsewhere: rel 4.2e-5, max 0.012.
        return {"rel": 1.7e-4, "max": 0.05}
    return {"rel": 1e-4, "max": 0.02, "differ": 1e-3}
