"""The walk over the four-wide nodes against the walk over the binary ones, both compiled for the CPU (tests/hipcpu):
more and worse-conditioned rays than the GPU tests send."""
import os
import sys

import numpy as np
import pytest

from photon_amd import host
from photon_amd.types import RAY_DTYPE, Material

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "hipcpu"))

import hipcpu_wide  # noqa: E402


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    return hipcpu_wide.build(str(tmp_path_factory.mktemp("wide")))


def _soup(rng, spread, tilt, n=400):
    """Triangles of about the scene's size, in a box of height `spread` and turned out of its plane by `tilt`."""
    p = rng.uniform(-1, 1, (n, 1, 3)) * [1, spread, 1] + rng.normal(0, 0.3, (n, 3, 3)) * [1, tilt, 1]
    p = p.astype(np.float32)
    s = host.Scene()
    s.add_mesh(p.reshape(-1, 3), np.arange(3 * n, dtype=np.int32), s.add_material(Material.default()))
    return hipcpu_wide.scene_arrays(s.build()), p.astype(np.float64)


def _aimed(rng, p, n, distance, grazing):
    """Rays at points of the triangles, many on edges and at vertices, from about `distance` away, up to `grazing` out of
    the triangle's plane (down to a ten-thousandth of it)."""
    t = p[rng.integers(len(p), size=n)]
    b = rng.dirichlet(np.ones(3), n)
    edge = rng.random(n) < 0.4
    b[edge, 0] = rng.uniform(0, 1e-4, edge.sum()) * (rng.random(edge.sum()) < 0.5)
    b[rng.random(n) < 0.2] = [0, 1, 0]
    x = (t * (b / b.sum(1, keepdims=True))[..., None]).sum(1)
    e1, e2 = t[:, 1] - t[:, 0], t[:, 2] - t[:, 0]
    normal = np.cross(e1, e2)
    normal /= np.linalg.norm(normal, axis=1, keepdims=True)
    d = rng.normal(size=(n, 1)) * e1 + rng.normal(size=(n, 1)) * e2
    d = d / np.linalg.norm(d, axis=1, keepdims=True) + grazing * 10.0 ** rng.uniform(-4, 0, (n, 1)) * rng.choice([-1.0, 1.0], (n, 1)) * normal
    o = (x - d / np.linalg.norm(d, axis=1, keepdims=True) * distance * 10.0 ** rng.uniform(-1, 1, (n, 1))).astype(np.float32)
    d = x - o
    r = np.zeros(n, RAY_DTYPE)
    r["o"], r["d"], r["tmax"] = o, d / np.linalg.norm(d, axis=1, keepdims=True), 1e30
    return r


def _differ(a, b):
    return (a["tri"] != b["tri"]) | (a["t"] != b["t"]) | (a["u"] != b["u"]) | (a["v"] != b["v"])


@pytest.mark.parametrize("distance", [1, 30, 300, 3000, 100000])
def test_hits_from_any_distance_are_the_binary_hits(lib, distance):
    """Angles down to a ten-thousandth of a radian: from far away the errors of a triangle's distance and of its box's are
    as large as the gaps between triangles."""
    rng = np.random.default_rng(distance)
    for spread, tilt in ((1, 1), (1, 1), (0.01, 0.01), (0.1, 0.01)):
        (nodes, tris), p = _soup(rng, spread, tilt)
        rays = _aimed(rng, p, 300000, distance, 1.0)
        for anyhit in (False, True):
            count, want, got, _ = hipcpu_wide.walk(lib, nodes, tris, rays, anyhit)
            assert count > 0 and (want["tri"] >= 0).mean() > 0.8
            assert np.array_equal(want["tri"] >= 0, got["tri"] >= 0) if anyhit else not _differ(want, got).any()


@pytest.mark.parametrize("distance", [0.3, 3, 30, 300, 3000])
def test_hits_along_triangles_planes_differ_only_where_the_distance_is_lost(lib, distance):
    """Rays within 1e-4 to 1e-8 of a triangle's plane. Where the answers differ the binary walk's triangle lies edge-on:
    its distance is off by more than the 2^-10 that boxes are entered behind a hit. That error is at most a few 2^-24 over
    |det| / (|e1| |e2| |d|), which is therefore below 2^-13. Any-hit answers never differ."""
    rng = np.random.default_rng(int(10 * distance))
    for spread, tilt in ((1, 1), (0.01, 0.01)):
        (nodes, tris), p = _soup(rng, spread, tilt)
        rays = _aimed(rng, p, 300000, distance, 1e-4)
        _, want, got, _ = hipcpu_wide.walk(lib, nodes, tris, rays)
        at = np.nonzero(_differ(want, got))[0]
        tri, d = tris[want["tri"][at]].astype(np.float64), rays["d"][at].astype(np.float64)
        e1, e2 = tri[:, 4:7], tri[:, 8:11]
        det = np.abs((np.cross(e1, e2) * d).sum(1))
        assert len(at) <= len(rays) / 2000
        assert np.all(det <= 2.0**-13 * np.linalg.norm(e1, axis=1) * np.linalg.norm(e2, axis=1) * np.linalg.norm(d, axis=1))
        assert np.all(got["t"][at] > want["t"][at])
        _, want, got, _ = hipcpu_wide.walk(lib, nodes, tris, rays, anyhit=True)
        assert np.array_equal(want["tri"] >= 0, got["tri"] >= 0)


def _rays_through(rng, n):
    r = np.zeros(n, RAY_DTYPE)
    d = rng.normal(size=(n, 3))
    r["d"] = d / np.linalg.norm(d, axis=1, keepdims=True)
    r["o"] = rng.uniform(-1, 1, (n, 3)) - 4 * r["d"]
    r["tmax"] = 1e30
    return r


def test_scenes_of_this_librarys_builders_have_wide_nodes(lib):
    for scene in (host.Scene.builtin("cornell-c1"), host.Scene.builtin("materials"), host.Scene.builtin("glass"), host.Scene.spheres(8, box=10.0, seed=3),
                  host.Scene.field(12, seed=2, env_width=64)):
        nodes, tris = hipcpu_wide.scene_arrays(scene.build())
        assert hipcpu_wide.walk(lib, nodes, tris, _rays_through(np.random.default_rng(1), 10))[0] > 0


def test_boxes_that_do_not_nest_are_left_to_the_binary_walk(lib):
    """A caller's hierarchy in which an interior box is smaller than what lies below it: the binary walk misses triangles
    outside of it. A wide node that leaves that box out would find them."""
    rng = np.random.default_rng(4)
    (nodes, tris), _ = _soup(rng, 1, 1)
    rays = _rays_through(rng, 20000)
    count, _, _, _ = hipcpu_wide.walk(lib, nodes, tris, rays)
    assert count > 0
    words = nodes.view(np.int32)
    changed = 0
    for i in range(1, min(40, len(nodes))):
        for side in (0, 8):
            if words[i, side + 7] == 0 and words[i, side + 3] >= 0:  # interior: the middle half of its box
                lo, hi = nodes[i, side:side + 3].copy(), nodes[i, side + 4:side + 7].copy()
                nodes[i, side:side + 3], nodes[i, side + 4:side + 7] = lo + (hi - lo) / 4, hi - (hi - lo) / 4
                changed += 1
    assert changed > 10
    assert hipcpu_wide.walk(lib, nodes, tris, rays)[0] == 0

