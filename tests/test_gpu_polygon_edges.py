"""The polygon test's quotients by edge constants as the device holds them: the checker's divisions, bit for bit."""

import ctypes

import numpy
import pytest

import fresnel_amd as fresnel
import oracle
from oracle import ptr

pytestmark = pytest.mark.gpu


def star(n, seed):
    """A star-shaped outline of n vertices."""
    rng = numpy.random.default_rng(seed)
    a = numpy.arange(n) * 2 * numpy.pi / n
    r = rng.uniform(0.3, 1.0, n)
    return numpy.stack([r * numpy.cos(a), r * numpy.sin(a)], axis=1)


POLYGONS = {
    'triangle': [[-1, -1], [1, -1], [0.3, 1]],
    # horizontal and vertical edges
    'steps': [[-1, -1], [1, -1], [1, 0], [0.25, 0], [0.25, 0.5], [-0.5, 0.5], [-0.5, 1], [-1, 1]],
    # repeated vertices (edges of no length, the last one among them) and a vertex on an edge
    'repeated': [[-1, -1], [-1, -1], [1, -1], [1, 1], [1, 1], [1, 1], [0, 1], [-1, 1], [-1, -1]],
    'star_101': star(101, 1),
    'star_1000': star(1000, 2),
    'tiny': 1e-20 * star(7, 3),
}


def build(device, vertices, rounding):
    s = fresnel.Scene(device, lights=fresnel.light.cloudy())
    size = numpy.abs(vertices).max()
    fresnel.geometry.Polygon(s, vertices, position=[[0, 0], [2.5 * size, 0.7 * size]], angle=[0, 0.4],
                             rounding_radius=rounding * size, outline_width=0.04 * size, color=(0.3, 0.5, 0.9))
    s.camera = fresnel.camera.Orthographic(position=(size, 0, 1), look_at=(size, 0, 0), up=(0, 1, 0), height=3 * size)
    return s


@pytest.mark.parametrize('rounding', [0.0, 0.1])
@pytest.mark.parametrize('name', sorted(POLYGONS))
def test_polygon_edges_equal_checker(name, rounding, gpu_device, cpu_device):
    """Rays at vertices, edge midpoints, points on edges and their neighbours; an image with outlines."""
    v = numpy.array(POLYGONS[name], dtype=numpy.float32)
    gs, cs = build(gpu_device, v, rounding), build(cpu_device, v, rounding)
    rng = numpy.random.default_rng(9)
    w = numpy.roll(v, 1, axis=0)
    f = rng.uniform(0, 1, (8 * len(v), 1)).astype(numpy.float32)
    on_edges = numpy.tile(v, (8, 1)) + f * numpy.tile(w - v, (8, 1))
    p = numpy.concatenate([v, (v + w) / 2, on_edges, rng.uniform(-1.2, 1.2, (2000, 2)) * numpy.abs(v).max()])
    p = p.astype(numpy.float32)
    p = numpy.concatenate([p, numpy.nextafter(p, numpy.float32(9)), numpy.nextafter(p, numpy.float32(-9))])
    down = numpy.tile(numpy.float32([0, 0, -1]), (len(p), 1))
    height = numpy.ones((len(p), 1))
    rays = [numpy.concatenate([p, height, down], axis=1)]
    tilted = rng.normal(size=(len(p), 3)) * [0.3, 0.3, 0] + [0, 0, -1]
    tilted /= numpy.linalg.norm(tilted, axis=1, keepdims=True)
    rays.append(numpy.concatenate([p + tilted[:, :2] / tilted[:, 2:], height, tilted], axis=1))
    rays = numpy.ascontiguousarray(numpy.concatenate(rays), dtype=numpy.float32)
    n = len(rays)
    gid, prim, t = gs._scene.debugTrace(rays, 1e-3)
    rg, rp, rt = numpy.zeros(n, numpy.uint32), numpy.zeros(n, numpy.uint32), numpy.zeros(n, numpy.float32)
    oracle.lib().oracle_trace(cs._scene.handle(), ptr(rays), n, 1e-3, ptr(rg, ctypes.c_uint32),
                              ptr(rp, ctypes.c_uint32), ptr(rt), None, 0)
    assert (rg != 0xffffffff).any() and (rg == 0xffffffff).any()
    assert numpy.array_equal(gid, rg) and numpy.array_equal(prim, rp)
    assert numpy.array_equal(t.view(numpy.uint32), rt.view(numpy.uint32))
    images = []
    for device, s in ((gpu_device, gs), (cpu_device, cs)):
        tracer = fresnel.tracer.Path(device, w=181, h=141)
        tracer.seed = 2
        tracer.sample(s, samples=2)
        images.append(numpy.array(tracer.linear_output[:]))
    assert numpy.array_equal(images[0].view(numpy.uint32), images[1].view(numpy.uint32))
