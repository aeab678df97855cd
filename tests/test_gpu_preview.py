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
