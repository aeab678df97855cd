"""Tiles with empty candidate lists are taken as background without tracing: whole images, odd sizes, batches."""

import numpy
import pytest

import fresnel_amd as fresnel

pytestmark = pytest.mark.gpu


def corner_scene(device, n=3):
    """A few spheres in one corner of the view, a background of its own: most tiles list nothing."""
    rng = numpy.random.default_rng(n)
    s = fresnel.Scene(device, lights=fresnel.light.cloudy())
    fresnel.geometry.Sphere(s, position=rng.uniform(-1, 1, (n, 3)) + [-3, 2, 0], radius=0.5, color=(0.2, 0.4, 0.9))
    s.camera = fresnel.camera.Orthographic(position=(0, 0, 20), look_at=(0, 0, 0), up=(0, 1, 0), height=8)
    s.background_color = (0.3, 0.1 + 0.01 * n, 0.7)
    s.background_alpha = 0.6
    return s


# whole tiles; strips on both sides; one tile; fewer pixels than a tile
@pytest.mark.parametrize('w,h', [(96, 64), (101, 75), (8, 8), (7, 5)])
@pytest.mark.parametrize('light_samples', [1, 3])
def test_background_tiles_equal_checker(w, h, light_samples, gpu_device, cpu_device):
    """Samples in two calls (the running mean goes on) and a batch of jobs whose rays share claims: the checker's bits."""
    images = {}
    for dev in (gpu_device, cpu_device):
        t = fresnel.tracer.Path(dev, w, h)
        s = corner_scene(dev)
        t.sample(s, samples=5, light_samples=light_samples)
        t.sample(s, samples=2, reset=False, light_samples=light_samples)
        images[dev.mode] = numpy.array(t.linear_output[:])
    numpy.testing.assert_array_equal(images['gpu'], images['cpu'])
    # three jobs, 3 samples each: a job's first ray is no multiple of 64
    jobs = [(corner_scene(gpu_device, n), fresnel.tracer.Path(gpu_device, w, h)) for n in (1, 2, 4)]
    for _, t in jobs:
        t.reset()
        t._tracer.setLightSamples(light_samples)
    fresnel._gpu.batch_render([s._scene for s, _ in jobs], [t._tracer for _, t in jobs], 3)
    for n, (_, t) in zip((1, 2, 4), jobs):
        c = fresnel.tracer.Path(cpu_device, w, h)
        c.sample(corner_scene(cpu_device, n), samples=3, light_samples=light_samples)
        numpy.testing.assert_array_equal(numpy.array(t.linear_output[:]), numpy.array(c.linear_output[:]))
