"""The 4-wide search against brute force: zero and tiny direction components, flat, tiny and huge scenes."""

import ctypes

import numpy
import pytest

import fresnel_amd as fresnel
import oracle
from oracle import ptr
import scenes
from test_gpu_parity import c1_scene

pytestmark = pytest.mark.gpu


def spheres(n, scale, offset=0.0, radius=0.5):
    def build(device):
        rng = numpy.random.default_rng(n)
        s = fresnel.Scene(device)
        pos = rng.uniform(-2, 2, (n, 3)) * scale + offset
        fresnel.geometry.Sphere(s, position=pos.astype(numpy.float32), radius=radius * scale)
        return s
    return build


def flat(device):
    """Triangles in the planes x = 0, y = 0 and z = 3, polygons in z = 0, spherocylinders along the axes."""
    s = fresnel.Scene(device)
    tri = [[0, -1, -1], [0, 1, -1], [0, -1, 1], [-1, 0, -1], [1, 0, -1], [-1, 0, 1], [-1, -1, 3], [1, -1, 3], [-1, 1, 3]]
    fresnel.geometry.Mesh(s, tri, position=[[0, 0, 0], [0, 0, 2], [3, 0, 0]], orientation=[[1, 0, 0, 0]] * 3)
    fresnel.geometry.Polygon(s, [[-1, -1], [1, -1], [0, 1]], position=[[0, 0], [2, 1], [-2, 0]], angle=[0, 0.5, 1])
    fresnel.geometry.Cylinder(s, points=[[[0, 0, 0], [2, 0, 0]], [[0, 0, 0], [0, 0, -2]], [[0, 1, 0], [0, 1, 0]]],
                              radius=0.1)
    return s


SCENES = {
    'spheres_1': spheres(1, 1.0),
    'spheres_2': spheres(2, 1.0),
    'spheres_3': spheres(3, 1.0),
    'spheres_5': spheres(5, 1.0),
    'spheres_700': spheres(700, 8.0, radius=0.02),
    'spheres_milli': spheres(200, 1e-3),
    'spheres_mega': spheres(200, 1e6),
    'spheres_1e18': spheres(200, 1e18),
    'spheres_aside': spheres(200, 1.0, offset=1000.0),
    'c1': c1_scene,
    'flat': flat,
    'polyhedra': scenes.eight_polyhedra,
    'cylinders': scenes.four_cylinders,
    'box': scenes.box,
    'triangle': scenes.one_triangle,
    'polygons': scenes.rounded_polygons,
}


def rays_of(scene, n, rng):
    """Rays between and along box faces of the scene: all, one or two direction components zero or tiny."""
    ext = scene.get_extents().astype(numpy.float64)
    c, half = (ext[0] + ext[1]) / 2, numpy.maximum((ext[1] - ext[0]) / 2, 0.2 * (ext[1] - ext[0]).max())
    o = c + rng.uniform(-2, 2, (n, 3)) * half
    d = rng.normal(size=(n, 3))
    small = [0.0, -0.0, 1e-45, 2.0**-61, -2.0**-60, 2.0**-59, 1e-12, -1e-6]
    k = rng.integers(0, 4, n)  # 0: as it is, 1: one component small, 2: two, 3: two, and the origin on the scene's planes
    axis = rng.integers(0, 3, n)
    for i in range(n):
        for j in range(3):
            if (k[i] == 1 and j == axis[i]) or (k[i] >= 2 and j != axis[i]):
                d[i, j] = small[rng.integers(len(small))]
                if k[i] == 3:
                    o[i, j] = [0.0, ext[0, j], ext[1, j], c[j]][rng.integers(4)]
    d /= numpy.linalg.norm(d, axis=1, keepdims=True)
    return numpy.ascontiguousarray(numpy.concatenate([o, d], axis=1), dtype=numpy.float32)


@pytest.mark.parametrize('name,tnear', [(name, tnear) for name in sorted(SCENES) for tnear in (0.0, 1e-3)]
                         + [(name, -3.0) for name in ('spheres_1', 'spheres_5', 'flat', 'box', 'cylinders', 'polygons')])
def test_search_equals_brute_force(name, tnear, gpu_device, cpu_device):
    """Geometry, primitive and distance of every ray are the brute-force minimum's, bit for bit."""
    gs, cs = SCENES[name](gpu_device), SCENES[name](cpu_device)
    n = 3000
    rays = rays_of(cs, n, numpy.random.default_rng(5))
    gid, prim, t = gs._scene.debugTrace(rays, tnear)
    L, h = oracle.lib(), cs._scene.handle()
    L.oracle_scene_set_brute(h, 1)
    rg, rp, rt = numpy.zeros(n, numpy.uint32), numpy.zeros(n, numpy.uint32), numpy.zeros(n, numpy.float32)
    L.oracle_trace(h, ptr(rays), n, tnear, ptr(rg, ctypes.c_uint32), ptr(rp, ctypes.c_uint32), ptr(rt), None, 0)
    assert numpy.array_equal(gid, rg)
    assert numpy.array_equal(prim, rp)
    assert numpy.array_equal(t.view(numpy.uint32), rt.view(numpy.uint32))
    assert (rg != 0xffffffff).any()


CUBOID = [[x, y, z] for x in (-0.5, 0.5) for y in (-0.5, 0.5) for z in (-0.25, 0.25)]


def test_edge_lines_of_polyhedra(gpu_device, cpu_device):
    """Rays through the lines of edges beyond the edges' ends, in a dense scene of convex polyhedra.  The reference's plane
    loop ends when the largest entry and smallest exit distance are equal and reports a hit, the planes left unseen, so
    such a ray, though it passes outside, may hit a polyhedron far before its bounding box.  The search then may or may not
    meet that hit before a nearer one culls its box.  Every other hit is the brute-force minimum: a ray that differs from
    brute force has a brute-force hit below that primitive's own culling bound."""
    n, n_rays, side = 3000, 200000, 20.0
    rng = numpy.random.default_rng(8)
    pos = rng.uniform(-side / 2, side / 2, (n, 3)).astype(numpy.float32)
    q = rng.normal(size=(n, 4))
    q = (q / numpy.linalg.norm(q, axis=1, keepdims=True)).astype(numpy.float32)

    def build(device):
        s = fresnel.Scene(device)
        fresnel.geometry.ConvexPolyhedron(s, fresnel.util.convex_polyhedron_from_vertices(CUBOID), position=pos,
                                          orientation=q)
        return s

    # a point on the line of an edge of polyhedron k, past the edge's end; rays through it from 20 to 130 away
    half, radius = numpy.array(CUBOID[-1]), numpy.linalg.norm(CUBOID[-1])
    k = rng.integers(0, n, n_rays)
    p = half * rng.choice([-1, 1], (n_rays, 3))
    axis = rng.integers(0, 3, n_rays)
    p[numpy.arange(n_rays), axis] *= rng.uniform(1, radius / half[axis])
    d = rng.normal(size=(n_rays, 3))
    d /= numpy.linalg.norm(d, axis=1, keepdims=True)

    def rotate(x):
        s, v = q[k].astype(numpy.float64)[:, :1], q[k].astype(numpy.float64)[:, 1:]
        return x + 2 * numpy.cross(v, numpy.cross(v, x) + s * x)

    o = p - d * rng.uniform(20, 130, (n_rays, 1))
    rays = numpy.ascontiguousarray(numpy.concatenate([rotate(o) + pos[k], rotate(d)], axis=1), dtype=numpy.float32)
    gs, cs = build(gpu_device), build(cpu_device)
    gid, prim, t = gs._scene.debugTrace(rays, 1e-3)
    L, h = oracle.lib(), cs._scene.handle()
    L.oracle_scene_set_brute(h, 1)
    rg, rp, rt = (numpy.zeros(n_rays, numpy.uint32), numpy.zeros(n_rays, numpy.uint32),
                  numpy.zeros(n_rays, numpy.float32))
    L.oracle_trace(h, ptr(rays), n_rays, 1e-3, ptr(rg, ctypes.c_uint32), ptr(rp, ctypes.c_uint32), ptr(rt), None, 0)
    hit = rg != 0xffffffff
    # the culling bound of the brute-force winner: its box's slab interval, less 2^-9 of its end and of 3 half extents
    with numpy.errstate(divide='ignore'):
        inv = 1 / rays[:, 3:].astype(numpy.float64)
    a = (pos[rp * hit] - radius - rays[:, :3]) * inv
    b = (pos[rp * hit] + radius - rays[:, :3]) * inv
    tmin, tmax = numpy.minimum(a, b).max(axis=1), numpy.maximum(a, b).min(axis=1)
    bound = tmin - 2.0**-9 * (numpy.maximum(tmax, 0) + 3 * radius)
    below = hit & (rt < bound * (1 + 1e-5))
    differs = (gid != rg) | (prim != rp) | (t.view(numpy.uint32) != rt.view(numpy.uint32))
    print(f"{below.sum()} of {hit.sum()} hits below their own bound, {differs.sum()} rays differ from brute force")
    assert below.any()
    assert not (differs & ~below).any()


# coordinates that are NaN: all three (no ray reaches the primitive's bounds), or x alone (y and z bound it)
@pytest.mark.parametrize('axes', [slice(0, 3), slice(0, 1)])
@pytest.mark.parametrize('kind', ['spheres', 'mixed'])
def test_nan_positions(kind, axes, gpu_device):
    """Primitives at NaN change nothing and are not walked by the rays that come near: the image and the node visits of
    a scene without them."""
    d = gpu_device._device
    images, visits = [], []
    for n_nan in (0, 20000):
        rng = numpy.random.default_rng(6)
        pos = rng.uniform(-4, 4, (1000 + n_nan, 3))
        pos[1000:, axes] = numpy.nan
        s = fresnel.Scene(gpu_device, lights=fresnel.light.cloudy())
        m = fresnel.material.Material(color=(0.3, 0.5, 0.9), roughness=0.5)
        fresnel.geometry.Sphere(s, position=pos, radius=0.3, material=m)
        if kind == 'mixed':
            fresnel.geometry.Cylinder(s, points=[[[-1, 0, 5], [2, 1, 4]]], radius=0.2, material=m)
        s.camera = fresnel.camera.Perspective(position=(3, 4, 12), look_at=(0, 0, 0), up=(0, 1, 0), focus_distance=12,
                                              focal_length=0.5, height=0.4)
        t = fresnel.tracer.Path(gpu_device, w=96, h=72)
        t.seed = 4
        d.countersEnable(True)
        try:
            t.sample(s, samples=4)
            c = d.countersLast()
        finally:
            d.countersEnable(False)
        visits.append((c[1] + c[7]) / (c[0] + c[6]))
        images.append(numpy.array(t.linear_output[:]))
    numpy.testing.assert_array_equal(images[1], images[0])
    # (at x alone NaN the visits of the exact binary search grow by a factor of 2.4 here)
    assert visits[1] < (1.01 if axes == slice(0, 3) else 4) * visits[0]


def test_flat_scene_visits(gpu_device):
    """Secondary rays that leave overlapping polygons in one plane do not walk the boxes they start in."""
    d = gpu_device._device
    rng = numpy.random.default_rng(3)
    s = fresnel.Scene(gpu_device, lights=fresnel.light.cloudy())
    fresnel.geometry.Polygon(s, [[-0.3, -0.3], [0.3, -0.3], [0, 0.3]], position=rng.uniform(-4, 4, (5000, 2)),
                             angle=rng.uniform(0, 6, 5000), color=(0.4, 0.5, 0.6))
    s.camera = fresnel.camera.Orthographic(position=(0, 0, 5), look_at=(0, 0, 0), up=(0, 1, 0), height=8)
    t = fresnel.tracer.Path(gpu_device, w=160, h=120)
    d.countersEnable(True)
    try:
        t.sample(s, samples=4)
        c = d.countersLast()
    finally:
        d.countersEnable(False)
    assert c[0] + c[6] > 10000
    # 1.0 with exact boxes: the root, whose children a ray leaves before tnear unless it grazes the plane
    assert (c[1] + c[7]) / (c[0] + c[6]) < 4


@pytest.mark.parametrize('kind', ['spheres', 'cylinders'])
def test_far_from_the_origin_visits(kind, gpu_device):
    """A scene moved by 2^20 (coordinates in steps of 1/8, exact in both places): about the same node visits."""
    d = gpu_device._device
    visits = []
    for offset in (0, 2**20):
        rng = numpy.random.default_rng(3)
        pos = rng.integers(-120, 120, (20000, 3)) / 8.0 + offset
        s = fresnel.Scene(gpu_device, lights=fresnel.light.cloudy())
        m = fresnel.material.Material(color=(0.3, 0.5, 0.9), roughness=0.5)
        if kind == 'spheres':
            fresnel.geometry.Sphere(s, position=pos, radius=0.5, material=m)
        else:
            end = pos + rng.integers(-8, 8, pos.shape) / 8.0
            fresnel.geometry.Cylinder(s, points=numpy.stack([pos, end], axis=1), radius=0.125, material=m)
        s.camera = fresnel.camera.Orthographic(position=(offset, offset, offset + 64), look_at=(offset, offset, offset),
                                               up=(0, 1, 0), height=32)
        t = fresnel.tracer.Path(gpu_device, w=160, h=120)
        t.seed = 2
        d.countersEnable(True)
        try:
            t.sample(s, samples=4)
            c = d.countersLast()
        finally:
            d.countersEnable(False)
        visits.append((c[1] + c[7]) / (c[0] + c[6]))
    # (the rays' own coordinates are steps of 1/8 there, so the paths differ)
    assert visits[1] < 1.5 * visits[0]
