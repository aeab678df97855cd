"""Primary rays searched one by one (many primitives per tile, no lists): the checker's bits, alone and in batches."""

import numpy
import pytest

import bench
import fresnel_amd as fresnel

pytestmark = pytest.mark.gpu


def dense_scene(device, kind, lens, seed=1):
    rng = numpy.random.default_rng(seed)
    s = fresnel.Scene(device, lights=fresnel.light.cloudy())
    m = fresnel.material.Material(color=(0.5, 0.4, 0.1), roughness=0.5)
    if kind == 'cylinders':
        a = rng.uniform(-8, 8, (20000, 3))
        fresnel.geometry.Cylinder(s, points=numpy.stack([a, a + rng.normal(0, 0.3, a.shape)], axis=1), radius=0.05,
                                  material=m)
    elif kind == 'meshes':
        fresnel.geometry.Mesh(s, bench.icosphere(0.4, 2), position=rng.uniform(-6, 6, (80, 3)),
                              orientation=bench.random_quaternions(80, rng), material=m)
    else:
        fresnel.geometry.Polygon(s, [[-0.1, -0.1], [0.1, -0.1], [0, 0.1]], position=rng.uniform(-8, 8, (25000, 2)),
                                 angle=rng.uniform(0, 6, 25000), material=m)
        fresnel.geometry.Sphere(s, position=[[0, 0, 1], [2, 1, 0]], radius=0.5, material=m)
    s.camera = fresnel.camera.Perspective(position=(3, 4, 25), look_at=(0, 0, 0), up=(0, 1, 0), focus_distance=25,
                                          focal_length=0.5, f_stop=0.25 if lens else numpy.inf, height=0.36)
    return s


@pytest.mark.parametrize('kind', ['cylinders', 'meshes', 'polygons'])
@pytest.mark.parametrize('lens,w,h', [(True, 64, 48), (False, 61, 51)])
def test_per_ray_primary_equals_checker(kind, lens, w, h, gpu_device, cpu_device):
    """At 64 x 48 and 16 samples these scenes hold over 16 Mi / (primary rays) primitives per 64 pixels."""
    d = gpu_device._device
    d.tune('tile_min_rays', 1 << 40)
    try:
        s = dense_scene(gpu_device, kind, lens)
        t = fresnel.tracer.Path(gpu_device, w, h)
        t.sample(s, samples=16, light_samples=2)  # (the hierarchy is built)
        d.statsEnable(True)
        t.seed = 3
        t.sample(s, samples=16, light_samples=2)
        assert 'traverse_primary' in d.statsLast()
        d.statsEnable(False)
        jobs = [(dense_scene(gpu_device, kind, lens, seed), fresnel.tracer.Path(gpu_device, w, h)) for seed in (1, 2)]
        for _, tr in jobs:
            tr.seed = 3
            tr.reset()
            tr._tracer.setLightSamples(2)
        fresnel._gpu.batch_render([x._scene for x, _ in jobs], [tr._tracer for _, tr in jobs], 16)
    finally:
        d.statsEnable(False)
        d.tune('tile_min_rays', 1)
    for k, image in enumerate([t] + [tr for _, tr in jobs]):
        c = fresnel.tracer.Path(cpu_device, w, h)
        c.seed = 3
        c.sample(dense_scene(cpu_device, kind, lens, 2 if k == 2 else 1), samples=16, light_samples=2)
        numpy.testing.assert_array_equal(numpy.array(image.linear_output[:]), numpy.array(c.linear_output[:]))
