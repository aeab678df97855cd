"""Repeated renders of one scene and tracer: what a call leaves out must not show."""

import time

import numpy
import pytest

import bench
import fresnel_amd as fresnel
from fresnel_amd import serve
from test_gpu_parity import c1_scene

pytestmark = pytest.mark.gpu


def test_outputs_read_after_reset_are_clear(gpu_device):
    """reset() queues the clearing of the outputs; every way of reading them waits for it."""
    s = c1_scene(gpu_device, n=300)
    t = fresnel.tracer.Path(gpu_device, w=640, h=480)
    for _ in range(5):
        t.sample(s, samples=2)
        assert t.linear_output[:].any()
        t.reset()
        assert not t.linear_output[:].any()
        t.sample(s, samples=2)
        t.reset()
        assert not t.output[:].any()
        t.sample(s, samples=2)
        t.reset()
        assert not numpy.array(t.output_async(linear=True).wait()).any()
        assert t.histogram()[0].sum() == 0


@pytest.mark.parametrize('tracer', ['Path', 'Preview'])
def test_material_changes_between_renders(tracer, gpu_device):
    """The geometry table is uploaded again when anything in it changed, and only then."""
    s = c1_scene(gpu_device, n=300)
    colors = [(0.9, 0.1, 0.1), (0.1, 0.9, 0.1), (0.1, 0.9, 0.1), (0.9, 0.1, 0.1)]
    images = []
    t = getattr(fresnel.tracer, tracer)(gpu_device, w=96, h=64)
    for c in colors:
        s.geometry[0].material.color = c
        t.seed = 5
        if tracer == 'Path':
            t.sample(s, samples=2)
        else:
            t.render(s)
        images.append(numpy.array(t.linear_output[:]))
    assert numpy.array_equal(images[1], images[2])
    assert numpy.array_equal(images[0], images[3])
    assert not numpy.array_equal(images[0], images[1])
    s.geometry[0].outline_width = 0.3
    t.seed = 5
    t.sample(s, samples=2) if tracer == 'Path' else t.render(s)
    assert not numpy.array_equal(images[3], t.linear_output[:])


@pytest.mark.parametrize('tail_rays', [96 * 64 * 3 - 1, 96 * 64 * 3, 96 * 64 * 3 + 1])
def test_tail_only_batches(tail_rays, gpu_device):
    """A batch of exactly, just under and just over tail_rays paths: the same image."""
    s = c1_scene(gpu_device, n=3000)
    t = fresnel.tracer.Path(gpu_device, w=96, h=64)
    t.seed = 5
    t.sample(s, samples=3)
    ref = numpy.array(t.linear_output[:])
    old = gpu_device._device.tune('tail_rays', tail_rays)
    try:
        for _ in range(2):
            t.seed = 5
            t.sample(s, samples=3)
            numpy.testing.assert_array_equal(t.linear_output[:], ref)
    finally:
        gpu_device._device.tune('tail_rays', old)


@pytest.mark.parametrize('tracer', ['Path', 'Preview'])
def test_color_edits_reach_the_next_render(tracer, gpu_device):
    """All colors of a large unchanged scene rewritten before every render (12 MB of copies, no new table or hierarchy):
    each image is that of a scene built with those colors."""
    n = 1 << 20
    rng = numpy.random.default_rng(4)
    pos = rng.uniform(-40, 40, (n, 3)).astype(numpy.float32)
    colors = [rng.uniform(0, 1, (n, 3)).astype(numpy.float32) for _ in range(2)]

    def build(c):
        s = fresnel.Scene(gpu_device, lights=fresnel.light.cloudy())
        fresnel.geometry.Sphere(s, position=pos, radius=0.4, color=c,
                                material=fresnel.material.Material(primitive_color_mix=1, roughness=0.5))
        s.camera = fresnel.camera.Orthographic(position=(0, 0, 80), look_at=(0, 0, 0), up=(0, 1, 0), height=60)
        return s

    def image(t, s):
        t.seed = 5
        if tracer == 'Path':
            t.sample(s, samples=1)
        else:
            t.render(s)
        return numpy.array(t.linear_output[:])

    def new_tracer():
        return getattr(fresnel.tracer, tracer)(gpu_device, w=320, h=240)

    fresh = [image(new_tracer(), build(c)) for c in colors]
    assert not numpy.array_equal(*fresh)
    s, t = build(colors[0]), new_tracer()
    image(t, s)
    builds = s._scene.bvhInfo()[0]
    for k in range(8):
        s.geometry[0].color[:] = colors[k % 2]
        numpy.testing.assert_array_equal(image(t, s), fresh[k % 2])
    assert s._scene.bvhInfo()[0] == builds


@pytest.mark.parametrize('edit', ['add', 'enable', 'disable', 'disable_spheres'])
def test_served_scene_edited_between_steps(edit, gpu_device):
    """A geometry of another type added to, enabled or disabled in a served scene shows with the next synchronization:
    the request goes on with the scene as it was built, and the next render has the edit."""

    def build():
        s = c1_scene(gpu_device, n=500)
        if edit != 'add':
            mesh(s)
            if edit == 'enable':
                s.geometry[1].disable()
        return s

    def mesh(s):
        fresnel.geometry.Mesh(s, bench.icosphere(2.0, 1), position=[[0, 0, 9], [5, 5, 9]],
                              orientation=[[1, 0, 0, 0]] * 2, color=(0.9, 0.2, 0.1))

    def change(s):
        if edit == 'add':
            mesh(s)
        elif edit == 'enable':
            s.geometry[1].enable()
        elif edit == 'disable':
            s.geometry[1].disable()
        else:
            s.geometry[0].disable()

    def sample(s):
        t = fresnel.tracer.Path(gpu_device, w=72, h=56)
        t.sample(s, samples=6)
        return numpy.array(t.linear_output[:])

    other = c1_scene(gpu_device, n=300, w_seed=3)
    before, alone = sample(build()), sample(other)
    edited = build()
    change(edited)
    after = sample(edited)
    assert not numpy.array_equal(before, after)
    s = build()
    srv = serve.Server(gpu_device, hbm_budget=1 << 34, target_paths=2 * 72 * 56)
    tracers = [fresnel.tracer.Path(gpu_device, w=72, h=56) for _ in range(2)]
    reqs = [srv.submit(scene, t, 6) for scene, t in zip((s, other), tracers)]
    for _ in range(2):
        srv.step()  # both scenes are built
    assert all(r.state == serve.ACTIVE for r in reqs)
    change(s)
    srv.run()
    assert [r.state for r in reqs] == [serve.DONE] * 2
    numpy.testing.assert_array_equal(tracers[0].linear_output[:], before)
    numpy.testing.assert_array_equal(tracers[1].linear_output[:], alone)
    numpy.testing.assert_array_equal(sample(s), after)


def test_counters_after_a_preview_beside_a_server_batch(gpu_device):
    """A preview ends before a served batch has added its work to the device's counters: the next render still starts
    from zero."""
    d = gpu_device._device
    alone = c1_scene(gpu_device, n=300)
    t = fresnel.tracer.Path(gpu_device, w=64, h=48)

    def counts():
        t.seed = 7
        t.sample(alone, samples=2)
        return d.countersLast()

    # few rays that take long: a polygon of 50,000 edges, 64 x 8 pixels
    a = numpy.linspace(0, 2 * numpy.pi, 50000, endpoint=False)
    slow = fresnel.Scene(gpu_device)
    fresnel.geometry.Polygon(slow, numpy.stack([numpy.cos(a), numpy.sin(a)], axis=1), position=[[0, 0]])
    slow.camera = fresnel.camera.Orthographic(position=(0, 0, 1), look_at=(0, 0, 0), up=(0, 1, 0), height=0.1)
    small = fresnel.Scene(gpu_device)
    fresnel.geometry.Sphere(small, position=[[0, 0, 0]], radius=0.5)
    small.camera = fresnel.camera.Orthographic.fit(small)
    preview = fresnel.tracer.Preview(gpu_device, w=8, h=8, anti_alias=False)
    preview.render(small)
    d.countersEnable(True)
    try:
        expected = counts()
        srv = serve.Server(gpu_device, hbm_budget=1 << 34, target_paths=512)
        req = srv.submit(slow, fresnel.tracer.Path(gpu_device, w=64, h=8), 8)
        srv.step()
        preview.render(small)
        assert req.state == serve.ACTIVE
        assert counts() == expected
        srv.run()
        assert req.state == serve.DONE
        assert counts() == expected
    finally:
        d.countersEnable(False)


def test_preview_after_a_batch_that_failed(gpu_device):
    """The second batch of a call is refused (2^32 light-sample paths) while the first one runs: the next call does not
    touch what that one still uses."""
    spheres = c1_scene(gpu_device, n=3000)
    mesh = fresnel.Scene(gpu_device)
    fresnel.geometry.Mesh(mesh, bench.icosphere(1.0, 1), position=[[0, 0, 0]], orientation=[[1, 0, 0, 0]])
    mesh.camera = fresnel.camera.Orthographic.fit(mesh)
    preview = fresnel.tracer.Preview(gpu_device, w=80, h=60)
    path = fresnel.tracer.Path(gpu_device, w=640, h=480)

    def images():
        preview.render(mesh)
        path.seed = 3
        path.sample(spheres, samples=1, light_samples=2)
        return numpy.array(preview.linear_output[:]), numpy.array(path.linear_output[:])

    expected = images()
    refused = fresnel.tracer.Path(gpu_device, w=256, h=256)
    refused._tracer.setLightSamples(65535)
    for _ in range(3):
        path._tracer.setLightSamples(64)
        with pytest.raises(RuntimeError, match='batch too large'):
            fresnel._gpu.batch_render([spheres._scene, mesh._scene], [path._tracer, refused._tracer], 1)
        for a, b in zip(images(), expected):
            numpy.testing.assert_array_equal(a, b)


def test_reading_an_image_does_not_wait_for_other_work(gpu_device):
    """A finished image (of Path.sample or a server) is read at once while clears of other outputs (33 GB) are still
    queued on the device stream; those outputs are read only after theirs."""
    s = c1_scene(gpu_device, n=300)
    sampled, served = [fresnel.tracer.Path(gpu_device, w=64, h=48) for _ in range(2)]
    preview = fresnel.tracer.Preview(gpu_device, w=64, h=48)
    sampled.sample(s, samples=2)
    preview.render(s)
    srv = serve.Server(gpu_device, hbm_budget=1 << 34, target_paths=1 << 16)
    req = srv.submit(s, served, 2)
    srv.run()
    assert req.state == serve.DONE
    images = [numpy.array(t.linear_output[:]) for t in (sampled, served, preview)]
    large = fresnel.tracer.Path(gpu_device, w=4096, h=4096)
    large.output[:]

    def timed(read):
        times = []
        for _ in range(3):
            for _ in range(100):
                large.reset()
            t0 = time.perf_counter()
            read()
            times.append(time.perf_counter() - t0)
            large.histogram()  # waits for the device stream
        return min(times)

    wait = timed(large.histogram)
    for t, image in zip((sampled, served, preview), images):
        assert timed(lambda: t.linear_output[:]) < 0.5 * wait
        numpy.testing.assert_array_equal(t.linear_output[:], image)
    large.sample(s, samples=1)
    for _ in range(20):
        large.reset()
    assert not large.output[:].any()


def test_tile_group_of_polygon_scenes(gpu_device):
    """Polygon scenes take the default tile_group as 2 tiles and every other value as it is: the entries tested differ,
    the images do not."""
    rng = numpy.random.default_rng(2)
    s = fresnel.Scene(gpu_device, lights=fresnel.light.cloudy())
    fresnel.geometry.Polygon(s, [[-0.1, -0.1], [0.1, -0.1], [0, 0.1]], position=rng.uniform(-5, 5, (4000, 2)),
                             angle=rng.uniform(0, 6, 4000), color=(0.2, 0.5, 0.9))
    s.camera = fresnel.camera.Orthographic(position=(0, 0, 5), look_at=(0, 0, 0), up=(0, 1, 0), height=10)
    t = fresnel.tracer.Path(gpu_device, w=203, h=151)
    d = gpu_device._device
    default = d.tune('tile_group', 0)
    assert default == 4
    entries, images = {}, {}
    d.countersEnable(True)
    try:
        for group in (1, 2, 4, 9, 16):
            d.tune('tile_group', group)
            t.seed = 3
            t.sample(s, samples=2)
            entries[group] = d.countersLast()[10]
            images[group] = numpy.array(t.linear_output[:])
    finally:
        d.countersEnable(False)
        d.tune('tile_group', default)
    assert entries[4] == entries[2]
    assert len({entries[g] for g in (1, 2, 9, 16)}) == 4
    for group in images:
        numpy.testing.assert_array_equal(images[group], images[1])


def test_tail_threshold_takes_no_memory(gpu_device):
    """The tail kernel's overflow stacks belong to its resident threads: a threshold of 2^24 rays keeps no request out
    of an 8 GB budget (a stack for each ray would take 10.7 GB in each of two scratches)."""
    s = c1_scene(gpu_device, n=3000)
    alone = fresnel.tracer.Path(gpu_device, w=96, h=64)
    alone.sample(s, samples=3)
    d = gpu_device._device
    old = d.tune('tail_rays', 1 << 24)
    try:
        srv = serve.Server(gpu_device, hbm_budget=8 << 30, target_paths=1 << 20)
        t = fresnel.tracer.Path(gpu_device, w=96, h=64)
        req = srv.submit(s, t, 3)
        srv.run()
        assert req.state == serve.DONE
        numpy.testing.assert_array_equal(t.linear_output[:], alone.linear_output[:])
    finally:
        d.tune('tail_rays', old)
