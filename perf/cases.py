"""The work that users of fresnel_amd have it do, as cases that can be timed and compared.

A case names a scene (geometry type and size), a call and its sizes.  The calls are the public ones:

  preview   `fresnel_amd.preview(scene)`, or a `tracer.Preview` whose linear image is read
  path      `fresnel_amd.pathtrace(scene)`, or `tracer.Path.sample` on a tracer that is kept
  frame     one frame of a trajectory: new positions into `geometry.position`, `Path.sample`, the image
  orbit     an interactive view: for each of four camera poses one sample per pixel, the image and its histogram
  serve     a burst of small requests through `serve.Server`

Every call ends with the image in host memory, as the program that asked for it gets it.
"""

import math

import numpy
import torch

import fresnel_amd as fresnel
from fresnel_amd import serve

# ------------------------------------------------------------------ cases


def listed():
    return [
        # a glance at a small cluster while a scene is set up (no anti-aliasing): latency
        dict(name="preview_glance", call="preview", scene="spheres", n=64, w=200, h=150, aa=False, out="srgb"),
        # the default call, preview(scene), of a few hundred particles; the linear image is kept
        dict(name="preview_default", call="preview", scene="spheres", n=500, w=600, h=370, aa=True, out="linear"),
        # a simulation of hard polyhedra, looked at in a notebook at 720p
        dict(name="preview_polyhedra", call="preview", scene="polyhedra", n=20000, w=1280, h=720, aa=True, out="srgb"),
        # a small figure with soft light: few pixels, several light samples
        dict(name="path_small", call="path", scene="spheres", n=4096, w=256, h=256, samples=16, light_samples=8,
             lens=False, out="linear"),
        # a two-dimensional system of rounded polygons, odd image size
        dict(name="path_polygons", call="path", scene="polygons", n=10000, w=641, h=479, samples=64, light_samples=1,
             lens=False, out="srgb"),
        # bonds or rods with depth of field (thin lens)
        dict(name="path_rods_lens", call="path", scene="cylinders", n=100000, w=853, h=480, samples=32,
             light_samples=1, lens=True, out="srgb"),
        # translucent triangle meshes (instances of a 320-triangle sphere)
        dict(name="path_meshes", call="path", scene="meshes", n=2000, w=1024, h=768, samples=32, light_samples=1,
             lens=False, out="srgb"),
        # the benchmark's large particle scene at its image size and sample count
        dict(name="path_lattice", call="path", scene="lattice", n=1048576, w=1920, h=1080, samples=256,
             light_samples=1, lens=False, out="srgb"),
        # mixed geometry: polyhedra, spherocylinders and meshes at the benchmark's densities
        dict(name="path_mixed", call="path", scene="mixed", n=225000, w=1920, h=1080, samples=32, light_samples=1,
             lens=False, out="srgb"),
        # a movie of a particle trajectory, one frame: every position changes
        dict(name="frame", call="frame", scene="spheres", n=262144, w=1280, h=720, samples=32, out="srgb"),
        # turning a scene in the interactive viewer: its quarter-size image of a full-HD window
        dict(name="orbit", call="orbit", scene="spheres", n=100000, w=480, h=270, out="srgb"),
        # a service that renders thumbnails: requests of 10^3 to 10^5 primitives, 8 samples each
        dict(name="serve", call="serve", scene="requests", requests=16, side=256, samples=8, out="srgb"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    call = rng.choice(["preview", "preview", "path", "path", "path", "path", "frame", "orbit", "serve"])
    if call == "serve":
        return dict(call=call, scene="requests", requests=_log(rng, 2, 24), side=_log(rng, 96, 512),
                    samples=_log(rng, 1, 16), out="srgb")
    if call == "frame":
        return dict(call=call, scene="spheres", n=_log(rng, 200, 400000), w=_log(rng, 160, 1400),
                    h=_log(rng, 120, 800), samples=_log(rng, 4, 48), out="srgb")
    if call == "orbit":
        return dict(call=call, scene=rng.choice(["spheres", "cylinders", "polyhedra"]), n=_log(rng, 200, 300000),
                    w=_log(rng, 160, 640), h=_log(rng, 120, 400), out="srgb")
    scene = rng.choice(["spheres", "spheres", "cylinders", "polyhedra", "meshes", "polygons", "mixed"])
    n = _log(rng, 1, 2500) if scene == "meshes" else _log(rng, 1, 150000)
    if call == "preview":
        return dict(call=call, scene=scene, n=n, w=_log(rng, 96, 1280), h=_log(rng, 64, 720),
                    aa=rng.random() < 0.7, out=rng.choice(["srgb", "linear"]))
    w, h, light = _log(rng, 64, 1920), _log(rng, 48, 1080), rng.choice([1, 1, 1, 2, 5])
    samples = min(_log(rng, 1, 128), max(1, 40_000_000 // (w * h * light)))
    return dict(call=call, scene=scene, n=n, w=w, h=h, samples=samples, light_samples=light,
                lens=rng.random() < 0.25, out=rng.choice(["srgb", "linear"]))


# ------------------------------------------------------------------ inputs

CUBOID = [[x, y, z] for x in (-0.5, 0.5) for y in (-0.5, 0.5) for z in (-0.25, 0.25)]
HEXAGON = [[0.5 * math.cos(k * math.pi / 3), 0.5 * math.sin(k * math.pi / 3)] for k in range(6)]


def _icosphere(radius, subdivisions):
    """Triangle corners of a subdivided icosahedron on a sphere."""
    g = (1 + math.sqrt(5)) / 2
    v = numpy.array([(-1, g, 0), (1, g, 0), (-1, -g, 0), (1, -g, 0), (0, -1, g), (0, 1, g), (0, -1, -g), (0, 1, -g),
                     (g, 0, -1), (g, 0, 1), (-g, 0, -1), (-g, 0, 1)])
    f = [(0, 11, 5), (0, 5, 1), (0, 1, 7), (0, 7, 10), (0, 10, 11), (1, 5, 9), (5, 11, 4), (11, 10, 2), (10, 7, 6),
         (7, 1, 8), (3, 9, 4), (3, 4, 2), (3, 2, 6), (3, 6, 8), (3, 8, 9), (4, 9, 5), (2, 4, 11), (6, 2, 10),
         (8, 6, 7), (9, 8, 1)]
    t = v[numpy.array(f)]
    for _ in range(subdivisions):
        a, b, c = t[:, 0], t[:, 1], t[:, 2]
        ab, bc, ca = a + b, b + c, c + a
        ab, bc, ca = ab / 2, bc / 2, ca / 2
        t = numpy.concatenate([numpy.stack(x, axis=1) for x in ((a, ab, ca), (ab, b, bc), (ca, bc, c), (ab, bc, ca))])
    t = t / numpy.linalg.norm(t, axis=2, keepdims=True)
    return (radius * t.reshape(-1, 3)).astype(numpy.float32)


ICOSPHERE = _icosphere(0.4, 2)


def _side(scene, n):
    """Edge of the box that holds n primitives at the scene's density."""
    if scene == "polygons":
        return max(1.5, math.sqrt(n / 0.9))
    if scene == "lattice":
        return 1.5 * round((n / 4) ** (1 / 3))
    return max(1.5, (n / {"spheres": 0.512, "cylinders": 1.2, "polyhedra": 0.3, "meshes": 0.5, "mixed": 1.3}[scene])
               ** (1 / 3))


def _quaternions(n, rng):
    q = rng.normal(size=(n, 4))
    return (q / numpy.linalg.norm(q, axis=1, keepdims=True)).astype(numpy.float32)


def _sphere_arrays(scene, n, rng):
    side = _side(scene, n)
    if scene == "lattice":
        # face-centred cubic lattice with thermal noise
        cells = round((n / 4) ** (1 / 3))
        g = numpy.stack(numpy.meshgrid(*[numpy.arange(cells, dtype=numpy.float32)] * 3, indexing="ij"), axis=-1)
        basis = numpy.array([[0, 0, 0], [0.5, 0.5, 0], [0.5, 0, 0.5], [0, 0.5, 0.5]], dtype=numpy.float32)
        pos = 1.5 * (g.reshape(-1, 1, 3) + basis).reshape(-1, 3) - side / 2
        pos += numpy.float32(0.05) * rng.standard_normal(pos.shape, dtype=numpy.float32)
        return dict(position=pos.astype(numpy.float32),
                    radius=rng.uniform(0.4, 0.6, len(pos)).astype(numpy.float32),
                    color=rng.uniform(0.05, 0.95, (len(pos), 3)).astype(numpy.float32))
    return dict(position=rng.uniform(-side / 2, side / 2, (n, 3)).astype(numpy.float32),
                radius=rng.uniform(0.4, 0.6, n).astype(numpy.float32),
                color=rng.uniform(0.05, 0.95, (n, 3)).astype(numpy.float32))


def _segments(n, side, rng):
    a = rng.uniform(-side / 2, side / 2, (n, 3))
    d = rng.normal(size=(n, 3))
    d *= rng.uniform(0.3, 1.0, (n, 1)) / numpy.linalg.norm(d, axis=1, keepdims=True)
    return numpy.stack([a, a + d], axis=1).astype(numpy.float32)


# cloudy lights: (direction towards the light in camera space, color, half angle)
LIGHTS = [((0.0, 1.0, 0.0), 0.9, math.pi / 2), ((0.0, -1.0, 0.0), 0.1, math.pi / 2)]
SPHERE_MATERIAL = dict(primitive_color_mix=1.0, roughness=0.3, specular=0.5, metal=0.0)
OUTLINE = 0.05


def _view(scene, side, yaw=0.0):
    """Numbers of the camera: the box from above and aside, or a flat system from the front."""
    if scene == "polygons":
        return dict(position=(0.0, 0.0, 10.0), look_at=(0.0, 0.0, 0.0), up=(0.0, 1.0, 0.0), height=1.05 * side)
    d = numpy.array([math.sin(math.pi / 4 + yaw), 0.8, math.cos(math.pi / 4 + yaw)])
    d /= numpy.linalg.norm(d)
    dist = 2.5 * (side + 1.0)
    return dict(position=tuple(float(x) for x in dist * d), look_at=(0.0, 0.0, 0.0), up=(0.0, 1.0, 0.0),
                focus_distance=dist, focal_length=0.5, height=0.36)


def _camera(scene, side, yaw=0.0, f_stop=math.inf):
    v = _view(scene, side, yaw)
    if scene == "polygons":
        return fresnel.camera.Orthographic(**v)
    return fresnel.camera.Perspective(f_stop=f_stop, **v)


def _material(**k):
    return fresnel.material.Material(**k)


def _build(scene, n, rng, lens=False):
    """The scene a program has set up, and its first geometry."""
    s = fresnel.Scene(_device(), lights=[fresnel.light.Light(direction=d, color=(c, c, c), theta=t)
                                         for d, c, t in LIGHTS])
    side = _side(scene, n)
    first = None
    if scene in ("spheres", "lattice"):
        first = fresnel.geometry.Sphere(s, material=_material(**SPHERE_MATERIAL), outline_width=OUTLINE,
                                        **_sphere_arrays(scene, n, rng))
    mixed = scene == "mixed"
    if scene == "polyhedra" or mixed:
        k = max(1, n * 4 // 45) if mixed else n
        first = fresnel.geometry.ConvexPolyhedron(
            s, fresnel.util.convex_polyhedron_from_vertices(CUBOID),
            position=rng.uniform(-side / 2, side / 2, (k, 3)).astype(numpy.float32),
            orientation=_quaternions(k, rng), color=rng.uniform(0.05, 0.95, (k, 3)).astype(numpy.float32),
            outline_width=0.03, material=_material(primitive_color_mix=1.0, roughness=0.1, metal=0.0))
    if scene == "cylinders" or mixed:
        k = max(1, n * 40 // 45) if mixed else n
        first = fresnel.geometry.Cylinder(s, points=_segments(k, side, rng), radius=0.1, color=(0.8, 0.7, 0.3),
                                          material=_material(color=(0.6, 0.45, 0.07), roughness=0.5, metal=1.0))
    if scene == "meshes" or mixed:
        k = max(1, n // 45) if mixed else n
        first = fresnel.geometry.Mesh(s, ICOSPHERE, color=(0.3, 0.4, 0.9),
                                      position=rng.uniform(-side / 2, side / 2, (k, 3)).astype(numpy.float32),
                                      orientation=_quaternions(k, rng),
                                      material=_material(color=(0.07, 0.13, 0.8), roughness=0.6, metal=0.0,
                                                         spec_trans=0.0 if mixed else 0.3))
    if scene == "polygons":
        first = fresnel.geometry.Polygon(s, HEXAGON, rounding_radius=0.05, outline_width=OUTLINE,
                                         position=rng.uniform(-side / 2, side / 2, (n, 2)).astype(numpy.float32),
                                         angle=rng.uniform(0, 2 * math.pi, n).astype(numpy.float32),
                                         color=rng.uniform(0.05, 0.95, (n, 3)).astype(numpy.float32),
                                         material=_material(primitive_color_mix=1.0, roughness=0.8))
    # a lens wide enough that about a tenth of the box's depth is in focus
    s.camera = _camera(scene, side, f_stop=5.0 / side if lens else math.inf)
    return s, first


_KEPT = {}


def _device():
    """One device and, for the requests, one server, kept for the life of the program."""
    if "device" not in _KEPT:
        _KEPT["device"] = fresnel.Device(mode="gpu", n=1)
    return _KEPT["device"]


def _server():
    if "server" not in _KEPT:
        _KEPT["server"] = serve.Server(_device(), target_paths=32 << 20)
    return _KEPT["server"]


def prepare(case, seed):
    rng = numpy.random.default_rng(seed)
    st = dict(case=case)
    if case["call"] == "serve":
        st["server"] = _server()
        st["requests"] = []
        for k in range(case["requests"]):
            n = int(round(math.exp(rng.uniform(math.log(1e3), math.log(1e5)))))
            scene, _ = _build(["spheres", "cylinders"][int(rng.integers(2))], n, rng)
            st["requests"].append((scene, fresnel.tracer.Path(_device(), w=case["side"], h=case["side"])))
        return st
    st["scene"], st["geometry"] = _build(case["scene"], case["n"], rng, case.get("lens", False))
    w, h = case["w"], case["h"]
    if case["call"] == "preview" and case["out"] == "linear":
        st["tracer"] = fresnel.tracer.Preview(_device(), w, h, case["aa"])
    if case["call"] in ("frame", "orbit") or (case["call"] == "path" and case["w"] * case["h"] > 1000000):
        st["tracer"] = fresnel.tracer.Path(_device(), w, h)
    if case["call"] == "frame":
        pos = st["geometry"].position[:]
        st["positions"] = (pos + rng.normal(0.0, 0.02, pos.shape)).astype(numpy.float32)
    if case["call"] == "orbit":
        side = _side(case["scene"], case["n"])
        yaw = float(rng.uniform(0, math.pi))
        st["poses"] = [_camera(case["scene"], side, yaw + 0.05 * k) for k in range(4)]
    return st


# ------------------------------------------------------------------ the calls


def _image(tracer, out):
    return tracer.linear_output[:] if out == "linear" else tracer.output[:]


def run(st):
    case = st["case"]
    call, out = case["call"], case["out"]
    if call == "preview":
        if out == "srgb":
            return fresnel.preview(st["scene"], w=case["w"], h=case["h"], anti_alias=case["aa"])[:]
        st["tracer"].render(st["scene"])
        return _image(st["tracer"], out)
    if call == "path":
        if "tracer" not in st and out == "srgb":
            return fresnel.pathtrace(st["scene"], w=case["w"], h=case["h"], samples=case["samples"],
                                     light_samples=case["light_samples"])[:]
        tracer = st.get("tracer")
        if tracer is None:
            tracer = fresnel.tracer.Path(_device(), case["w"], case["h"])
        tracer.seed = 20  # the same image each time
        tracer.sample(st["scene"], samples=case["samples"], light_samples=case["light_samples"])
        return _image(tracer, out)
    if call == "frame":
        st["geometry"].position[:] = st["positions"]
        st["tracer"].seed = 20
        st["tracer"].sample(st["scene"], samples=case["samples"])
        return _image(st["tracer"], out)
    if call == "orbit":
        got = []
        tracer = st["tracer"]
        tracer.seed = 20
        for pose in st["poses"]:
            st["scene"].camera = pose
            tracer.reset()
            tracer.render(st["scene"])
            got.append(_image(tracer, out))
            got.append(tracer.histogram()[0])
        return got
    handles = []
    for scene, tracer in st["requests"]:
        tracer.seed = 20
        handles.append(st["server"].submit(scene, tracer, case["samples"]))
    st["server"].run()
    for handle in handles:
        st["server"].release(handle)
    return [_image(tracer, out) for _, tracer in st["requests"]]


# ------------------------------------------------------------------ what a pass cannot do without

# bytes of one primitive as the caller gives it: positions, sizes, orientations, colors
PRIM_BYTES = {"spheres": 28, "lattice": 28, "cylinders": 52, "polyhedra": 40, "meshes": 28, "polygons": 24, "mixed": 50}
# floating point operations of one path: camera ray, search, shading of about 1.4 surface hits
PATH_FLOPS = 170


def work(case):
    pixel = 16 if case["out"] == "linear" else 4
    if case["call"] == "serve":
        paths = case["requests"] * case["side"] ** 2 * case["samples"]
        # 10^3 to 10^5 primitives, log-uniform: 21,500 on average
        return dict(bytes=case["requests"] * (case["side"] ** 2 * pixel + 21500 * 40), flops=paths * PATH_FLOPS)
    pixels = case["w"] * case["h"]
    images = 4 if case["call"] == "orbit" else 1
    per_pixel = images
    if case["call"] == "preview":
        per_pixel = 64 if case["aa"] else 1
    elif case["call"] != "orbit":
        per_pixel = case["samples"] * case.get("light_samples", 1)
    return dict(bytes=images * pixels * pixel + case["n"] * PRIM_BYTES[case["scene"]],
                flops=pixels * per_pixel * PATH_FLOPS)


def tolerance(case):
    # The framework's images are defined to the bit: every ray's random numbers come from its pixel, sample and
    # seed, and each pixel's samples are added in order, so how the work is split does not show.
    return "exact"


# ------------------------------------------------------------------ 64-bit values


def _philox(c2, c3, k0, k1):
    """Philox4x32-10 of the counter (0, 0, c2, c3): the first two words (int64 tensors)."""
    m = 0xFFFFFFFF
    c0 = torch.zeros_like(c2)
    c1 = torch.zeros_like(c2)
    c3 = torch.full_like(c2, c3)
    for _ in range(10):
        # 32 x 32 -> 64 bit products from 16-bit halves of the counter (no 64-bit overflow)
        def product(a, x):
            lo, hi = a * (x & 0xFFFF), a * (x >> 16)
            t = hi + (lo >> 16)
            return t >> 16, ((t & 0xFFFF) << 16) | (lo & 0xFFFF)
        h0, l0 = product(0xD2511F53, c0)
        h1, l1 = product(0xCD9E8D57, c2)
        c0, c1, c2, c3 = h1 ^ c1 ^ k0, l1, h0 ^ c3 ^ k1, l0
        k0 = (k0 + 0x9E3779B9) & m
        k1 = (k1 + 0xBB67AE85) & m
    return c0, c1


def _tent(u):
    r = 2.0 * (u.double() * 2.0 ** -32 + 2.0 ** -33)
    return torch.where(r < 1.0, torch.sqrt(r) - 1.0, 1.0 - torch.sqrt(torch.clamp(2.0 - r, min=0.0)))


def exact(case, seed):
    """Previews of spheres, in 64 bits.

    A path-traced image has no such value: each bounce takes a decision (which surface, which lobe, go on or stop)
    from 32-bit values, and the image is defined by those decisions.
    """
    if case["call"] != "preview" or case["scene"] != "spheres":
        return None
    if case["w"] * case["h"] * (64 if case["aa"] else 1) * case["n"] > 2e10:
        return None
    a = _sphere_arrays("spheres", case["n"], numpy.random.default_rng(seed))
    dev, f8 = "cuda", torch.float64
    centre, radius, color = (torch.from_numpy(a[k]).to(dev, f8) for k in ("position", "radius", "color"))
    view = _view("spheres", _side("spheres", case["n"]))
    W, H = case["w"], case["h"]

    def unit(v):
        return v / numpy.linalg.norm(v)

    p = numpy.array(view["position"], dtype=numpy.float32).astype(numpy.float64)
    focus, focal, height = (float(numpy.float32(view[k])) for k in ("focus_distance", "focal_length", "height"))
    d = unit(numpy.array(view["look_at"]) - p)
    u = unit(numpy.cross(d, view["up"]))
    v = unit(numpy.cross(u, d))
    plane = height / focal * focus
    lights = [(unit(ld[0] * u + ld[1] * v - ld[2] * d), c, t) for ld, c, t in LIGHTS]
    T = {k: torch.tensor(x, device=dev, dtype=f8) for k, x in (("p", p), ("d", d), ("u", u), ("v", v))}
    rough, spec = SPHERE_MATERIAL["roughness"], SPHERE_MATERIAL["specular"]

    def dot(x, y):
        return (x * y).sum(-1, keepdim=True)

    def schlick(x):
        return (1.0 - x) ** 5

    def shade(n, view_dir, base):
        out = torch.zeros_like(base)
        for ld, c, theta in lights:
            l = torch.tensor(ld, device=dev, dtype=f8).expand_as(n)
            r = -view_dir + 2.0 * n * dot(n, view_dir)
            ldotr = dot(l, r)
            axis = torch.linalg.cross(l, r)
            axis = axis / torch.linalg.norm(axis, dim=-1, keepdim=True).clamp_min(1e-300)
            ang = -torch.acos(ldotr.clamp(-1.0, 1.0)) + theta
            s, q = torch.cos(ang / 2), torch.sin(ang / 2) * axis
            turned = (s * s - dot(q, q)) * r + 2 * s * torch.linalg.cross(q, r) + 2 * dot(q, r) * q
            r = torch.where(ldotr < math.cos(theta), turned, r)
            ndotv, ndotl = dot(n, view_dir), dot(n, l)
            h = l + view_dir
            h = h / torch.linalg.norm(h, dim=-1, keepdim=True)
            ldoth = dot(l, h)
            fl, fv, rr = schlick(ndotl), schlick(ndotv), 2 * rough * ldoth ** 2
            diffuse = base / math.pi * ((1 - 0.5 * fl) * (1 - 0.5 * fv) + rr * (fl + fv + fl * fv * (rr - 1)))
            diffuse = torch.where((ndotv > 0) & (ndotl >= 0), diffuse * ndotl, torch.zeros_like(diffuse))
            ndotr = dot(n, r)
            h = r + view_dir
            h = h / torch.linalg.norm(h, dim=-1, keepdim=True)
            rdoth, ndoth = dot(r, h), dot(n, h)
            a2 = rough ** 4
            D = a2 / (math.pi * (1 + (a2 - 1) * ndoth ** 2) ** 2)
            half = min(theta, 0.99 * math.pi / 2)
            wide = min(rough ** 2 + 0.5 * math.tan(half), 1.0)
            D = D * a2 / wide ** 2
            F0 = 0.08 * spec
            F = F0 + (1 - F0) * schlick(rdoth)
            V = 1 / (ndotv + torch.sqrt(a2 + ndotv ** 2 - a2 * ndotv ** 2))
            V = V / (ndotr + torch.sqrt(a2 + ndotr ** 2 - a2 * ndotr ** 2))
            specular = torch.where((ndotv > 0) & (ndotr >= 0), D * F * V * ndotr, torch.zeros_like(ndotr))
            out = out + (diffuse + specular) * math.pi * c
        return out

    rows = max(1, int(1.5e8 // (W * case["n"])))
    image = torch.zeros((H, W, 4), device=dev, dtype=f8)
    rel = centre - T["p"]
    cc = dot(rel, rel).reshape(1, -1) - radius.reshape(1, -1) ** 2
    for sample in range(64 if case["aa"] else 1):
        for j0 in range(0, H, rows):
            j = torch.arange(j0, min(H, j0 + rows), device=dev).reshape(-1, 1).expand(-1, W).reshape(-1)
            i = torch.arange(W, device=dev).repeat(min(H, j0 + rows) - j0)
            x, y = i.double() + 0.5, j.double() + 0.5
            if case["aa"]:
                r = _philox(torch.full_like(i, sample), 0x22AB5871, j * W + i, torch.zeros_like(i))
                x, y = x + _tent(r[0]) * math.sqrt(0.5), y + _tent(r[1]) * math.sqrt(0.5)
            xs, ys = x / H - 0.5 * W / H, -(y / H - 0.5)
            ray = T["d"] * focus + (ys[:, None] * T["v"] + xs[:, None] * T["u"]) * plane
            ray = ray / torch.linalg.norm(ray, dim=-1, keepdim=True)
            b = ray @ rel.T
            det = b * b - cc
            t = b - torch.sqrt(det.clamp_min(0.0))
            t = torch.where((det >= 0) & (t > 1e-4), t, torch.full_like(t, math.inf))
            t, k = t.min(dim=1)
            del b, det
            hit = torch.nonzero(torch.isfinite(t)).reshape(-1)
            if len(hit):
                ray, t, k = ray[hit], t[hit], k[hit]
                at = T["p"] + t[:, None] * ray
                n = at - centre[k]
                n = n / torch.linalg.norm(n, dim=-1, keepdim=True)
                edge = radius[k] - torch.linalg.norm(torch.linalg.cross(rel[k], ray), dim=-1)
                got = shade(n, -ray, color[k])
                got = torch.where((edge >= OUTLINE)[:, None], got, torch.zeros_like(got))
                px = image.view(-1, 4)
                px[j[hit] * W + i[hit]] += torch.cat([got, torch.ones_like(t)[:, None]], dim=1)
    image /= 64 if case["aa"] else 1
    if case["out"] == "linear":
        return image.cpu().numpy()
    c = image[..., :3]
    s = torch.where(c < 0.0031308, 12.92 * c, 1.055 * c.clamp_min(1e-12) ** (1 / 2.4) - 0.055).clamp_max(1.0)
    return (255.0 * torch.cat([s, image[..., 3:]], dim=-1)).cpu().numpy()
