"""The preview kernel: samples shared by a workgroup's wavefronts, tile lists or packets, every image shape."""

import numpy
import pytest

import fresnel_amd as fresnel
from test_gpu_parity import PRIMARY_SCENES

pytestmark = pytest.mark.gpu


def touching_plane(device):
    """Triangles, polygons and spheres on, touching and behind the plane an orthographic camera's rays start from."""
    s = fresnel.Scene(device, lights=fresnel.light.cloudy())
    tri = [[-3, -3, 0], [3, -3, 0], [-3, 3, 0]]
    fresnel.geometry.Mesh(s, tri, position=[[0, 0, 0], [0.5, 0.5, -1]], orientation=[[1, 0, 0, 0]] * 2, color=(1, 0, 0))
    fresnel.geometry.Sphere(s, position=[[0, 0, -0.5], [1, 1, 0.5], [1, -1, 0], [-1, -1, 2]], radius=0.5)
    fresnel.geometry.Polygon(s, [[-1, -1], [1, -1], [0, 1]], position=[[1.5, 0.5]], angle=[0.3])
    s.camera = fresnel.camera.Orthographic(position=(0, 0, 0), look_at=(0, 0, -1), up=(0, 1, 0), height=6)
    return s


SCENES = dict(PRIMARY_SCENES, touching_plane=touching_plane)


def render(device, scene, w, h, aa_n):
    t = fresnel.tracer.Preview(device, w=w, h=h)
    t._tracer.setAntialiasingN(aa_n)
    t.enable_highlight_warning((0, 1, 1))
    t.render(scene)
    return numpy.array(t.linear_output[:]), numpy.array(t.output[:])


# one pixel; a strip narrower than a tile; whole tiles; tiles with strips on both sides.
# 1 sample (each wavefront has a chunk to itself); 4, 9 and 64 samples (shared; a partial last round).
@pytest.mark.parametrize('w,h,aa_n', [(1, 1, 8), (5, 70, 3), (64, 40, 2), (75, 61, 1), (75, 61, 3)])
@pytest.mark.parametrize('name', sorted(SCENES))
def test_preview_lists_packets_checker(name, w, h, aa_n, gpu_device, cpu_device):
    """Lists and packets give the same bits; the checker's colors agree to the library functions' rounding.

    Hits and outline choices are exact; the lighting calls acosf, sinf and cosf, whose device and host versions
    differ by a few ulp: at most 1e-6 rad in the reflected direction, and the specular lobe's relative slope is at
    most 2 / roughness^2 = 200 per rad at the scenes' smallest roughness, 0.1.
    """
    scene = SCENES[name](gpu_device)
    lists = render(gpu_device, scene, w, h, aa_n)
    try:
        gpu_device._device.tune('tile_min_rays', 1 << 40)
        packets = render(gpu_device, scene, w, h, aa_n)
    finally:
        gpu_device._device.tune('tile_min_rays', 1)
    numpy.testing.assert_array_equal(lists[0], packets[0])
    numpy.testing.assert_array_equal(lists[1], packets[1])
    ref = render(cpu_device, SCENES[name](cpu_device), w, h, aa_n)
    numpy.testing.assert_array_equal(lists[0][..., 3], ref[0][..., 3])
    numpy.testing.assert_allclose(lists[0], ref[0], rtol=4e-4, atol=1e-5)


# 2^18 tiles, every sphere over all of them: lists of 2^27.8 entries; more than the 2^30 they may have; 2^32 + 3 * 2^18, whose
# 32-bit count is 3 * 2^18
@pytest.mark.parametrize('n,lists', [(900, True), (4100, False), (16387, False)])
def test_preview_lists_too_long(n, lists, gpu_device):
    """A scene whose lists would be too long is searched in the hierarchy: the same pixels as with lists off."""
    d = gpu_device._device
    s = fresnel.Scene(gpu_device, lights=fresnel.light.cloudy())
    pos = numpy.random.default_rng(n).uniform(-1, 1, (n, 3))
    fresnel.geometry.Sphere(s, position=pos, radius=5, color=(0.5, 0.5, 0.1))
    s.camera = fresnel.camera.Orthographic(position=(0, 0, 30), look_at=(0, 0, 0), up=(0, 1, 0), height=2)
    preview = fresnel.tracer.Preview(gpu_device, w=4096, h=4096, anti_alias=False)
    path = fresnel.tracer.Path(gpu_device, w=4096, h=4096)

    def images():
        preview.render(s)
        path.seed = 3
        path.sample(s, samples=1)
        return numpy.array(preview.output[:]), numpy.array(path.output[:])

    d.statsEnable(True)
    try:
        preview.render(s)
        assert ('tiles_emit' in d.statsLast()) == lists
    finally:
        d.statsEnable(False)
    got = images()
    try:
        d.tune('primary_tiles', 1)
        expected = images()
    finally:
        d.tune('primary_tiles', 2)
    for a, b in zip(got, expected):
        assert numpy.array_equal(a, b)
