"""Timed workloads of the framework and their plain 64-bit values.

Each case is one call (or one frame) that a program built on althea_amd makes:

- ``resolve``: the deferred resolve of a G-buffer (lights, IBL, SSAO);
- ``frame``: every pass of a rendered frame, from the meshes to the image;
- ``shadow``: the shadow cubes of a set of point lights;
- ``gbuffer``: the G-buffer of a mesh;
- ``precompute``: an environment's IBL state into a handle that is kept;
- ``batch``: the prefiltered cubes of many maps in one run;
- ``labels``: prefiltered radiance at (direction, roughness) queries;
- ``train``: loss and gradients of the learned prefilter on a batch;
- ``infer``: the learned prefilter at queries.

``listed()`` names the representative sizes, ``draw(rng)`` draws others of the
same ranges, ``prepare`` makes what a program has in hand before the call,
``run`` makes the call, ``work`` counts the bytes and operations it cannot do
without and ``exact`` evaluates the same formulas in 64 bits in plain torch.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import althea_amd as aa
from althea_amd import _lib
from althea_amd.batch import PrefilterBatch
from althea_amd.mlp import PrefilterMLP

F64 = torch.float64
CHUNK = 1 << 22  # elements of a 64-bit intermediate


# ------------------------------------------------------------------- cases
def listed() -> list:
    return [
        # A material or probe preview, and the smallest frame an engine asks
        # for: launches and latency.
        dict(name="resolve_160x90", kind="resolve", width=160, height=90, lights=4, fp16=False, ssao=True,
             tonemap=True, env=512, cube=128, mips=5),
        # An FP16 G-buffer and target of a ragged window, SSAO off (a medium
        # quality setting).
        dict(name="resolve_1919x1079_fp16", kind="resolve", width=1919, height=1079, lights=17, fp16=True, ssao=False,
             tonemap=True, env=1024, cube=256, mips=6),
        # The benchmark's 4K frame: 64 lights, SSAO, the 512^2 cube.
        dict(name="resolve_4k", kind="resolve", width=3840, height=2160, lights=64, fp16=False, ssao=True,
             tonemap=False, env=2048, cube=512, mips=6),
        # A whole 1080p frame of a textured scene: glTF G-buffer, shadow
        # cubes, reflections, their convolution and the resolve.
        dict(name="frame_1080p", kind="frame", width=1920, height=1080, lights=32, cells=96, shadow=256, env=1024,
             cube=256, mips=6),
        # The benchmark's shadow pass: 64 lights over 32 768 triangles.
        dict(name="shadow_64x256", kind="shadow", lights=64, size=256, cells=128),
        # A plain mesh into a 1440p G-buffer.
        dict(name="gbuffer_1440p", kind="gbuffer", width=2560, height=1440, cells=128, fp16=False),
        # Scene load with the default description (a 512x256 map).
        dict(name="precompute_128", kind="precompute", env=512, cube=128, mips=5, samples=1024, irradiance=32,
             theta=300, lut=128),
        # Scene load of the 4K benchmark's maps.
        dict(name="precompute_512", kind="precompute", env=2048, cube=512, mips=6, samples=1024, irradiance=32,
             theta=300, lut=128),
        # A library of maps of uneven resolution in one run.
        dict(name="batch_12", kind="batch", maps=12, env=1024, mips=5, samples=1024),
        # Labels of the learned prefilter.
        dict(name="labels_2e18", kind="labels", env=1024, count=1 << 18, samples=1024),
        # One batch of the learned prefilter's training.
        dict(name="train_65536", kind="train", count=65536),
        # Queries of the learned prefilter, an odd number of them.
        dict(name="infer_50001", kind="infer", count=50001),
    ]


def _log(rng, lo: float, hi: float) -> float:
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng) -> dict:
    kind = rng.choice(["resolve", "resolve", "frame", "shadow", "gbuffer", "precompute", "precompute", "batch",
                       "labels", "train", "infer"])
    env = 1 << rng.randint(8, 11)
    if kind in ("resolve", "frame"):
        height = int(_log(rng, 40, 1440 if kind == "resolve" else 900))
        width = max(16, int(height * rng.uniform(0.6, 2.2)))
        cube = 1 << rng.randint(6, 8)
        case = dict(kind=kind, width=width, height=height, lights=int(_log(rng, 1, 65)), env=env, cube=cube,
                    mips=rng.randint(4, 6))
        if kind == "resolve":
            case.update(fp16=rng.random() < 0.4, ssao=rng.random() < 0.7, tonemap=rng.random() < 0.5)
        else:
            case.update(lights=min(case["lights"], 24), cells=rng.randint(20, 96),
                        shadow=rng.choice([64, 96, 128, 256]))
        return case
    if kind == "shadow":
        return dict(kind=kind, lights=int(_log(rng, 1, 49)), size=rng.randint(48, 256), cells=rng.randint(8, 128))
    if kind == "gbuffer":
        height = int(_log(rng, 60, 1440))
        return dict(kind=kind, width=max(16, int(height * rng.uniform(0.6, 1.8))), height=height,
                    cells=rng.randint(4, 128), fp16=rng.random() < 0.4)
    if kind == "precompute":
        return dict(kind=kind, env=env, cube=1 << rng.randint(5, 8), mips=rng.randint(3, 6),
                    samples=int(_log(rng, 100, 1400)), irradiance=rng.choice([8, 9, 16, 24, 32]),
                    theta=rng.choice([64, 150, 200, 300]), lut=rng.choice([32, 50, 64, 128]))
    if kind == "batch":
        return dict(kind=kind, maps=rng.randint(1, 10), env=1 << rng.randint(8, 10), mips=rng.randint(3, 5),
                    samples=int(_log(rng, 64, 1024)))
    if kind == "labels":
        return dict(kind=kind, env=env, count=int(_log(rng, 50, 1 << 17)), samples=int(_log(rng, 64, 2048)))
    if kind == "train":
        return dict(kind=kind, count=int(_log(rng, 100, 65537)))
    return dict(kind=kind, count=int(_log(rng, 20, 400000)))


# ------------------------------------------------------------------ inputs
def _camera(width: int, height: int, lights: int, exposure: float = 0.5):
    """GlobalUniforms of a 60-degree camera at (0, 3.5, 12) looking at the
    origin (column-major; Vulkan depth, y flipped)."""
    eye = np.array([0.0, 3.5, 12.0])
    f = -eye / np.linalg.norm(eye)
    s = np.cross(f, [0.0, 1.0, 0.0])
    s /= np.linalg.norm(s)
    u = np.cross(s, f)
    rot = np.stack([s, u, -f])
    view, iview, proj, iproj = (np.zeros((4, 4)) for _ in range(4))  # [row, column]
    view[:3, :3], view[:3, 3], view[3, 3] = rot, -rot @ eye, 1.0
    iview[:3, :3], iview[:3, 3], iview[3, 3] = rot.T, eye, 1.0
    near, far, th = 0.01, 1000.0, math.tan(math.radians(30.0))
    proj[0, 0], proj[1, 1] = height / (width * th), -1.0 / th
    proj[2, 2], proj[2, 3], proj[3, 2] = far / (near - far), -far * near / (far - near), -1.0
    iproj[0, 0], iproj[1, 1] = 1.0 / proj[0, 0], 1.0 / proj[1, 1]
    iproj[2, 3], iproj[3, 2], iproj[3, 3] = -1.0, 1.0 / proj[2, 3], proj[2, 2] / proj[2, 3]
    g = _lib.GlobalsC()
    for name, m in (("projection", proj), ("inverse_projection", iproj), ("view", view), ("prev_view", view),
                    ("inverse_view", iview), ("prev_inverse_view", iview)):
        getattr(g, name)[:] = [float(x) for x in m.T.ravel()]
    g.light_count = lights
    g.exposure = exposure
    return g


def _env(seed: int, width: int):
    """A high-contrast sky: per-texel log-normal radiance and three suns."""
    return torch.from_numpy(aa.synth.env(seed=seed, width=width, height=width // 2)).cuda()


def _ibl(seed: int, case: dict):
    desc = aa.IBLDesc(prefiltered_size=case["cube"], prefiltered_mips=case["mips"], prefilter_samples=256)
    return aa.ImageBasedLighting.createResources(_env(seed, case["env"]), desc)


def _mesh(seed: int, cells: int):
    pos, idx = aa.synth.heightfield_mesh(seed, n=cells)
    return pos, idx


def _gbuffer_mesh(seed: int, cells: int):
    pos, idx = _mesh(seed, cells)
    nrm, col, mro = aa.synth.mesh_attributes(seed, pos, idx)
    f = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    return aa.GBufferMesh(f(pos), f(idx.view(np.int32)), f(col), f(mro), f(nrm))


def _lights_and_ssao(seed: int, lights: int):
    s = aa.synth.scene(seed=seed, width=4, height=4, lights=lights)
    return s.lights_tensor("cuda"), s.ssao


def _random(seed: int, *shape):
    return torch.rand(shape, generator=torch.Generator("cuda").manual_seed(seed), device="cuda")


def _gltf(seed: int, cells: int):
    """The heightfield as a textured, alpha-tested primitive."""
    pos, idx = _mesh(seed, cells)
    nrm, _, _ = aa.synth.mesh_attributes(seed, pos, idx)
    f = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    rng = np.random.default_rng(seed)
    base = rng.integers(0, 256, (256, 256, 4), dtype=np.uint8)
    base[..., 3] = np.where(rng.uniform(size=(256, 256)) < 0.1, 40, 255)
    bump = np.concatenate([rng.integers(96, 160, (256, 256, 2)), np.full((256, 256, 2), 255)], -1).astype(np.uint8)
    mr = rng.integers(0, 256, (128, 128, 4), dtype=np.uint8)
    tex = [aa.Texture(f(base), mips=9, srgb=True), aa.Texture(f(bump), mips=9), aa.Texture(f(mr), mips=8)]
    uv = ((pos[:, [0, 2]] / 20.0 + 0.5) * 8.0).astype(np.float32)
    axis = lambda k: f(np.tile(np.eye(3, dtype=np.float32)[k], (len(pos), 1)))  # noqa: E731
    prim = aa.GltfPrimitive(f(pos), axis(0), axis(2), f(nrm), [f(uv)], f(idx.view(np.int32)), 0)
    return [prim], [aa.GltfMaterial(0, 1, 2)], tex


class _DeviceArray:
    """A float32 device buffer of an IBL handle as torch takes it; the tensor
    keeps this object, and this object the handle that owns the buffer."""

    def __init__(self, owner, ptr: int, shape: tuple):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=shape, typestr="<f4", data=(ptr, False), version=2)


def _ibl_outputs(ibl):
    """The handle's own maps: environment pyramid, prefiltered cube,
    irradiance cube, BRDF LUT."""
    v = ibl.views()
    of = lambda p, n, c: torch.as_tensor(_DeviceArray(ibl, p, (n, c)), device="cuda")  # noqa: E731
    return [of(v.environment, _lib.lib().althea_env_pyramid_texels(v.env_width, v.env_height), 4),
            of(v.prefiltered, aa.cube_texels(v.prefiltered_size, v.prefiltered_mips), 4),
            of(v.irradiance, 6 * v.irradiance_size ** 2, 4), of(v.brdf_lut, v.brdf_lut_size ** 2, 2)]


def _batch_widths(case: dict) -> list:
    return [case["env"] >> (i % 3) for i in range(case["maps"])]


def _precompute_desc(case: dict):
    return aa.IBLDesc(irradiance_size=case["irradiance"], irradiance_theta_samples=case["theta"],
                      prefiltered_size=case["cube"], prefiltered_mips=case["mips"], prefilter_samples=case["samples"],
                      brdf_lut_size=case["lut"], brdf_lut_samples=1024)


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    s = dict(kind=kind, case=case)
    if kind == "resolve":
        w, h = case["width"], case["height"]
        s["globals"] = _camera(w, h, case["lights"])
        s["lights"], s["ssao"] = _lights_and_ssao(seed, case["lights"])
        if not case["ssao"]:
            s["ssao"] = None
        g = aa.SceneToGBufferPass(w, h).begin(_gbuffer_mesh(seed, 128), s["globals"])
        # Textured materials: albedo and roughness vary from pixel to pixel.
        r = _random(seed, h, w, 8)
        one = torch.ones(h, w, 1, device="cuda")
        albedo = torch.cat([0.05 + 0.9 * r[..., :3], one], -1)
        mro = torch.cat([r[..., 3:4], 0.05 + 0.95 * r[..., 4:5], 0.5 + 0.5 * r[..., 5:6], one], -1)
        dt = torch.float16 if case["fp16"] else torch.float32
        planes = [p.to(dt).contiguous() for p in (g.planes[0], g.planes[1], albedo, mro)]
        s["gbuffer"] = aa.GBufferResources(*planes)
        s["ibl"] = _ibl(seed + 1, case)
        s["out"] = torch.empty((h * w, 4), dtype=dt, device="cuda")
    elif kind == "frame":
        w, h = case["width"], case["height"]
        s["globals"] = _camera(w, h, case["lights"])
        lights, s["ssao"] = _lights_and_ssao(seed, case["lights"])
        s["lights"] = aa.PointLightCollection.from_lights(lights, shadow_size=case["shadow"])
        s["gltf"] = _gltf(seed, case["cells"])
        s["pass"] = aa.SceneToGBufferPass(w, h)
        s["reflection"] = aa.ReflectionBuffer(w, h)
        s["ibl"] = _ibl(seed + 1, case)
        s["out"] = torch.empty((h * w, 4), device="cuda")
    elif kind == "shadow":
        pos, idx = _mesh(seed, case["cells"])
        s["positions"], s["indices"] = torch.from_numpy(pos).cuda(), torch.from_numpy(idx.view(np.int32)).cuda()
        s["lights"] = aa.PointLightCollection.from_lights(_lights_and_ssao(seed, case["lights"])[0],
                                                          shadow_size=case["size"])
    elif kind == "gbuffer":
        s["globals"] = _camera(case["width"], case["height"], 0)
        s["mesh"] = _gbuffer_mesh(seed, case["cells"])
        s["pass"] = aa.SceneToGBufferPass(case["width"], case["height"], fp16=case["fp16"])
    elif kind == "precompute":
        # The handle a program keeps while environments change.
        s["env"] = _env(seed, case["env"])
        s["ibl"] = aa.ImageBasedLighting.createResources(s["env"], _precompute_desc(case))
        s["out"] = _ibl_outputs(s["ibl"])
    elif kind == "batch":
        s["envs"] = [_env(seed + i, w) for i, w in enumerate(_batch_widths(case))]
        s["batch"] = PrefilterBatch(s["envs"], [w // 4 for w in _batch_widths(case)], mips=case["mips"],
                                    samples=case["samples"])
        s["batch"].run()  # captures and instantiates the batch's graph
    elif kind == "labels":
        s["pyramid"] = aa.env_pyramid(_env(seed, case["env"]))
        s["queries"] = torch.from_numpy(aa.synth.dir_rough(seed=seed + 1, n=case["count"])).cuda()
    else:
        s["net"] = PrefilterMLP(seed=seed)
        s["queries"] = torch.from_numpy(aa.synth.dir_rough(seed=seed + 1, n=case["count"])).cuda()
        if kind == "train":
            # Radiance that the queries' directions and roughness determine.
            q = s["queries"]
            t = torch.exp(torch.stack([torch.sin(3.0 * q[:, 0]), q[:, 1] * q[:, 3], q[:, 2], q[:, 0]], 1))
            s["labels"] = t.contiguous()
    return s


def run(s: dict):
    kind = s["kind"]
    if kind == "resolve":
        c = s["case"]
        return aa.DeferredRendering.resolve(s["gbuffer"], s["ibl"], s["lights"], s["globals"], s["ssao"],
                                            tonemap=c["tonemap"], out_fp16=c["fp16"], out=s["out"])
    if kind == "frame":
        prims, mats, texs = s["gltf"]
        g = s["pass"].begin_gltf(prims, mats, texs, s["globals"])
        s["lights"].drawShadowMapsGltf(prims, mats, texs)
        aa.ScreenSpaceReflection.captureReflection(g, s["ibl"], s["lights"], s["globals"], s["reflection"])
        aa.ScreenSpaceReflection.convolveReflectionBuffer(s["reflection"])
        out = aa.DeferredRendering.resolve(g, s["ibl"], s["lights"], s["globals"], s["ssao"], tonemap=True,
                                           out=s["out"], reflection=s["reflection"])
        return [out, s["reflection"].data, *g.planes]
    if kind == "shadow":
        return s["lights"].drawShadowMaps(s["positions"], s["indices"])
    if kind == "gbuffer":
        return list(s["pass"].begin(s["mesh"], s["globals"]).planes)
    if kind == "precompute":
        s["ibl"].precompute(s["env"])
        return s["out"]
    if kind == "batch":
        s["batch"].run()
        return [s["batch"].cube(i) for i in range(s["batch"].count)]
    if kind == "labels":
        w = s["case"]["env"]
        return aa.prefilter_points(s["pyramid"], w, w // 2, s["case"]["samples"], s["queries"])
    if kind == "train":
        return list(s["net"].gradients(s["queries"], s["labels"]))
    return s["net"].infer(s["queries"])


# -------------------------------------------------------------------- work
_LOOKUP = 60      # rotation, two arctangents, four texels and their weights
_LIGHT = 50       # one point light at one pixel
_SSAO = 40        # one SSAO tap
_TEXEL_TEST = 40  # one texel or pixel against one triangle
_MAC = 10176      # multiply-adds of one MLP query


def _kept(samples: int, mips: int) -> list:
    """Share of the samples with N.L > 0 per mip, times the samples (1 at
    roughness 0, where every sample is the mirror direction)."""
    return [1 if m == 0 else samples * 1.0 / (1.0 + (m / (mips - 1)) ** 2) for m in range(mips)]


def _prefilter_flops(size: int, mips: int, samples: int) -> float:
    k = _kept(samples, mips)
    return sum(6 * max(1, size >> m) ** 2 * k[m] * _LOOKUP for m in range(mips))


def work(case: dict) -> dict:
    kind = case["kind"]
    cube = lambda s, m: 16 * sum(6 * max(1, s >> k) ** 2 for k in range(m))  # noqa: E731
    if kind in ("resolve", "frame"):
        px, n = case["width"] * case["height"], case["lights"]
        state = cube(case["cube"], case["mips"]) + 16 * 6 * 32 ** 2 + 8 * 128 ** 2
        if kind == "resolve":
            texel = 8 if case["fp16"] else 16
            return dict(bytes=5 * texel * px + state + 32 * n,
                        flops=px * (n * _LIGHT + 16 * _SSAO * case["ssao"] + 300))
        # The image, the reflection buffer (FP16, 4/3 of a frame) and the
        # planes written, the cubes written; 24 march steps a pixel.
        shadow = 4 * n * 6 * (case["shadow"] + 2) ** 2
        return dict(bytes=px * (16 + 64 + 11) + shadow + state + 100 * case["cells"] ** 2,
                    flops=px * (2 * n * _LIGHT + 16 * _SSAO + 300 + 24 * 40)
                    + n * case["shadow"] ** 2 * _TEXEL_TEST)
    if kind == "shadow":
        tris, texels = 2 * case["cells"] ** 2, 6 * (case["size"] + 2) ** 2
        return dict(bytes=4 * case["lights"] * texels + 18 * tris,
                    flops=case["lights"] * (tris * 60 + texels * _TEXEL_TEST))
    if kind == "gbuffer":
        px, tris = case["width"] * case["height"], 2 * case["cells"] ** 2
        return dict(bytes=px * (32 if case["fp16"] else 64) + 36 * tris, flops=px * (_TEXEL_TEST + 60) + tris * 100)
    if kind == "precompute":
        w, irr = case["env"], 6 * case["irradiance"] ** 2
        return dict(bytes=16 * (w * w // 2) * (1 + 4 / 3) + cube(case["cube"], case["mips"]) + 16 * irr
                    + 8 * case["lut"] ** 2,
                    flops=_prefilter_flops(case["cube"], case["mips"], case["samples"])
                    + irr * case["theta"] * (case["theta"] // 2) * _LOOKUP + case["lut"] ** 2 * 1024 * 30)
    if kind == "batch":
        ws = _batch_widths(case)
        return dict(bytes=sum(16 * (w * w // 2) + cube(w // 4, case["mips"]) for w in ws),
                    flops=sum(_prefilter_flops(w // 4, case["mips"], case["samples"]) for w in ws))
    if kind == "labels":
        return dict(bytes=16 * case["env"] ** 2 * 2 / 3 + 32 * case["count"],
                    flops=case["count"] * case["samples"] * 0.75 * _LOOKUP)
    if kind == "train":  # forward, backward-data and weight gradients
        return dict(bytes=32 * case["count"] + 8 * 10371, flops=3 * 2 * _MAC * case["count"])
    return dict(bytes=32 * case["count"] + 4 * 10371, flops=2 * _MAC * case["count"])


# ------------------------------------------------------- plain 64-bit values
def _unit(v):
    return v / v.norm(dim=-1, keepdim=True)


def _dot(a, b):
    return (a * b).sum(-1)


def _rows(n: int, per_row: int):
    """Ranges of n rows whose intermediates hold about CHUNK elements."""
    step = max(1, CHUNK // max(1, per_row))
    for lo in range(0, n, step):
        yield lo, min(n, lo + step)


def _pyramid64(level0):
    """Box chain of an (h, w, 4) map: list of (h_l, w_l, 4)."""
    levels = [level0.to(F64)]
    count = 1 + int(math.log2(max(level0.shape[:2])))
    while len(levels) < count:
        p = levels[-1]
        h, w = p.shape[:2]
        if h > 1:
            p = 0.5 * (p[0::2] + p[1::2])
        if w > 1:
            p = 0.5 * (p[:, 0::2] + p[:, 1::2])
        levels.append(p)
    return levels


class _Sampler:
    """Trilinear REPEAT lookups of an equirect pyramid at (direction, LOD),
    with the pole branch of the precompute shaders."""

    def __init__(self, levels):
        self.levels = len(levels)
        self.flat = torch.cat([p.reshape(-1, 4)[:, :3] for p in levels])
        dims = [p.shape[:2] for p in levels]
        self.h = torch.tensor([d[0] for d in dims], device="cuda")
        self.w = torch.tensor([d[1] for d in dims], device="cuda")
        size = self.h * self.w
        self.off = torch.cumsum(size, 0) - size

    def _bilinear(self, level, u, v):
        w, h, off = self.w[level], self.h[level], self.off[level]
        x, y = u * w - 0.5, v * h - 0.5
        fx, fy = torch.floor(x), torch.floor(y)
        ax, ay = (x - fx)[..., None], (y - fy)[..., None]
        x0, y0 = fx.long() % w, fy.long() % h
        x1, y1 = (x0 + 1) % w, (y0 + 1) % h
        at = lambda i, j: self.flat[off + j * w + i]  # noqa: E731
        return ((at(x0, y0) * (1 - ax) + at(x1, y0) * ax) * (1 - ay)
                + (at(x0, y1) * (1 - ax) + at(x1, y1) * ax) * ay)

    def __call__(self, d, lod):
        xz = torch.hypot(d[..., 0], d[..., 2])
        off_pole = xz > 0.001
        yaw = torch.where(off_pole, torch.atan2(d[..., 2], d[..., 0]), 0.0)
        pole = torch.where(d[..., 1] > 0, 0.5 * math.pi, -0.5 * math.pi)
        pitch = torch.where(off_pole, torch.atan2(d[..., 1], xz), pole)
        u, v = yaw / (2 * math.pi) + 0.5, 0.5 - pitch / math.pi
        lod = lod.clamp(0, self.levels - 1).expand(u.shape)
        l0 = torch.floor(lod).long()
        l1 = (l0 + 1).clamp(max=self.levels - 1)
        t = (lod - l0)[..., None]
        return self._bilinear(l0, u, v) * (1 - t) + self._bilinear(l1, u, v) * t


def _frame_of(raw):
    n = _unit(raw)
    x, y, z = n.unbind(-1)
    zero = torch.zeros_like(x)
    a = torch.stack([-z, zero, x], -1) / torch.hypot(x, z).clamp_min(1e-300)[..., None]
    b = torch.stack([zero, z, -y], -1) / torch.hypot(y, z).clamp_min(1e-300)[..., None]
    t = torch.where((raw[..., 0].abs() > raw[..., 1].abs())[..., None], a, b)
    return t, torch.cross(n, t, dim=-1), n


def _face_dirs(size: int):
    """(6, size, size, 3) texel-centre directions on the half-texel lattice."""
    c = 2 * torch.arange(size, device="cuda", dtype=F64) + 1 - size
    tc, sc = torch.meshgrid(c, c, indexing="ij")
    m = torch.full_like(sc, float(size))
    faces = [(m, -tc, -sc), (-m, -tc, sc), (sc, m, tc), (sc, -m, -tc), (sc, -tc, m), (-sc, -tc, -m)]
    return torch.stack([torch.stack(f, -1) for f in faces])


def _hammersley(n: int):
    i = torch.arange(n, device="cuda")
    bits = torch.zeros_like(i)
    for k in range(32):
        bits |= ((i >> k) & 1) << (31 - k)
    return i.to(F64) / n, bits.to(F64) / 2 ** 32


def _ggx(rough, samples: int, width: int, height: int):
    """Per sample (and roughness, broadcast): local L and source LOD."""
    x1, x2 = _hammersley(samples)
    a2 = rough * rough
    den = 1 + (a2 - 1) * x2
    c, s = torch.sqrt((1 - x2) / den), torch.sqrt(a2 * x2 / den)
    phi = 2 * math.pi * x1
    lz = 2 * c * c - 1
    L = torch.stack([2 * c * torch.cos(phi) * s, 2 * c * torch.sin(phi) * s, lz], -1)
    D = a2 / (math.pi * (c * c * (a2 - 1) + 1) ** 2)
    pdf = D * c / (4 * c + 1e-5)
    lod = 0.5 * torch.log2(1 / (samples * pdf + 1e-4) / (4 * math.pi / (6.0 * width * height)))
    return L, torch.where(rough == 0, torch.zeros_like(lod), lod), lz.clamp_min(0.0)


def _exact_prefilter(levels, size: int, mips: int, samples: int):
    h, w = levels[0].shape[:2]
    look = _Sampler(levels)
    out = []
    for m in range(mips):
        rough = torch.tensor(m / (mips - 1) if mips > 1 else 0.0, dtype=F64, device="cuda")
        raw = _face_dirs(max(1, size >> m)).reshape(-1, 3)
        if float(rough) == 0.0:
            rgb = torch.cat([look(raw[a:b] / size, torch.zeros((), dtype=F64, device="cuda"))
                             for a, b in _rows(len(raw), 4)])
        else:
            L, lod, weight = _ggx(rough, samples, w, h)
            L, lod, weight = L[weight > 0], lod[weight > 0], weight[weight > 0]
            rgb = torch.empty_like(raw)
            for a, b in _rows(len(raw), len(lod)):
                t, bt, n = _frame_of(raw[a:b])
                d = (t[:, None] * L[None, :, :1] + bt[:, None] * L[None, :, 1:2] + n[:, None] * L[None, :, 2:])
                rgb[a:b] = (look(d, lod[None]) * weight[None, :, None]).sum(1) / weight.sum()
        out.append(torch.cat([rgb, torch.ones_like(rgb[:, :1])], 1))
    return torch.cat(out)


def _exact_irradiance(levels, size: int, theta: int):
    h, w = levels[0].shape[:2]
    phi = int(h * theta / w)
    look = _Sampler(levels)
    lod = torch.tensor(math.log2(w / theta), dtype=F64, device="cuda")
    raw = _face_dirs(size).reshape(-1, 3)
    th = torch.arange(theta, device="cuda", dtype=F64) * (2 * math.pi / theta)
    out = torch.zeros_like(raw)
    for j in range(phi):
        p = 0.5 * math.pi * j / phi
        for a, b in _rows(len(raw), theta):
            t, bt, n = (v[:, None] for v in _frame_of(raw[a:b]))
            d = n * math.cos(p) + (t * torch.cos(th)[:, None] + bt * torch.sin(th)[:, None]) * math.sin(p)
            out[a:b] += look(d, lod).sum(1) * (math.cos(p) * math.sin(p))
    return torch.cat([out * (math.pi / theta / phi), torch.ones_like(out[:, :1])], 1)


def _exact_lut(size: int, samples: int):
    g = (torch.arange(size, device="cuda", dtype=F64) + 0.5) / size
    r, nv = (v.reshape(-1, 1) for v in torch.meshgrid(g, g, indexing="ij"))
    a2 = r ** 4
    k = 0.5 * r * r
    x1, x2 = _hammersley(samples)
    den = 1 + (a2 - 1) * x2
    hz, s = torch.sqrt((1 - x2) / den), torch.sqrt(a2 * x2 / den)
    vdh = torch.sqrt((1 - nv * nv).clamp_min(0)) * torch.cos(2 * math.pi * x1) * s + nv * hz
    ndl = 2 * vdh * hz - nv
    smith = lambda c: c / (c * (1 - k) + k)  # noqa: E731
    vis = torch.where(ndl > 0, smith(nv) * smith(ndl) * vdh / (hz * nv), 0.0)
    fc = (1 - vdh) ** 5
    return torch.stack([((1 - fc) * vis).mean(1), (fc * vis).mean(1)], 1)


def _exact_labels(case: dict, state: dict):
    w, samples = case["env"], case["samples"]
    look = _Sampler(_pyramid64(_split_pyramid(state["pyramid"], w)))
    q = state["queries"].to(F64)
    out = torch.ones(len(q), 4, dtype=F64, device="cuda")
    for a, b in _rows(len(q), samples):
        t, bt, n = (v[:, None] for v in _frame_of(q[a:b, :3]))
        L, lod, weight = _ggx(q[a:b, 3:], samples, w, w // 2)
        d = t * L[..., :1] + bt * L[..., 1:2] + n * L[..., 2:]
        out[a:b, :3] = (look(d, lod) * weight[..., None]).sum(1) / weight.sum(1, keepdim=True)
    return out


def _split_pyramid(flat, width: int):
    return flat[:width * (width // 2)].reshape(width // 2, width, 4)


# The MLP: 3 + 24 + 1 features, three SiLU layers of 64, log radiance.
def _mlp64(params, q):
    f = [q[:, :3]]
    for k in range(4):
        f += [torch.sin(2 ** k * math.pi * q[:, :3]), torch.cos(2 ** k * math.pi * q[:, :3])]
    h = torch.cat(f + [q[:, 3:4]], 1)
    at = 0
    for layer, (n_in, n_out) in enumerate(((28, 64), (64, 64), (64, 64), (64, 3))):
        weight = params[at:at + n_out * n_in].reshape(n_out, n_in)
        bias = params[at + n_out * n_in:at + n_out * n_in + n_out]
        at += n_out * n_in + n_out
        h = h @ weight.T + bias
        if layer < 3:
            h = h * torch.sigmoid(h)
    return h


def _exact_mlp(case: dict, state: dict):
    params = torch.from_numpy(state["net"].get_params()).cuda().to(F64)
    q = state["queries"].to(F64)
    if case["kind"] == "infer":
        y = torch.cat([_mlp64(params, q[a:b]) for a, b in _rows(len(q), 64)])
        return torch.cat([torch.exp(y), torch.ones_like(y[:, :1])], 1)
    params.requires_grad_(True)
    loss = ((_mlp64(params, q) - torch.log(state["labels"][:, :3].to(F64))) ** 2).mean()
    (grad,) = torch.autograd.grad(loss, params)
    return [grad, loss.detach().reshape(1)]


# Seamless cube lookups: faces with the neighbours' texels around them.
def _bordered(cube, size: int):
    """(6, size, size, 3) -> (6, size + 2, size + 2, 3)."""
    ring = [(i, j) for j in range(-1, size + 1) for i in range(-1, size + 1)
            if not (0 <= i < size and 0 <= j < size)]
    lattice = lambda f, i, j: {0: (size, -j, -i), 1: (-size, -j, i), 2: (i, size, j), 3: (i, -size, -j),  # noqa: E731
                               4: (i, -j, size), 5: (-i, -j, -size)}[f]

    def fold(face, i, j):
        p = list(lattice(face, 2 * i + 1 - size, 2 * j + 1 - size))
        over = next(k for k in range(3) if abs(p[k]) == size + 1)
        p[over] = int(math.copysign(size, p[over]))
        p[face // 2] = int(math.copysign(size - 1, p[face // 2]))
        f = 2 * over + (p[over] < 0)
        sc, tc = {0: (-p[2], -p[1]), 1: (p[2], -p[1]), 2: (p[0], p[2]), 3: (p[0], -p[2]), 4: (p[0], -p[1]),
                  5: (-p[0], -p[1])}[f]
        return f, (tc + size - 1) // 2, (sc + size - 1) // 2

    out = torch.zeros(6, size + 2, size + 2, 3, dtype=F64, device="cuda")
    out[:, 1:-1, 1:-1] = cube
    dst, src = [], []
    for f in range(6):
        for i, j in ring:
            ic, jc = min(max(i, 0), size - 1), min(max(j, 0), size - 1)
            if i == ic or j == jc:
                taps = [fold(f, i, j)] * 3
            else:
                taps = [(f, jc, ic), fold(f, i, jc), fold(f, ic, j)]
            dst.append((f, j + 1, i + 1))
            src.append(taps)
    d, t = torch.tensor(dst, device="cuda"), torch.tensor(src, device="cuda")
    out[d[:, 0], d[:, 1], d[:, 2]] = cube[t[..., 0], t[..., 1], t[..., 2]].mean(1)
    return out


def _cube_coords(d):
    x, y, z = d.unbind(-1)
    ax, ay, az = x.abs(), y.abs(), z.abs()
    on_x, on_y = (ax >= ay) & (ax >= az), ay >= az
    face = torch.where(on_x, (x < 0).long(), torch.where(on_y, 2 + (y < 0).long(), 4 + (z < 0).long()))
    sc = torch.where(on_x, torch.where(x >= 0, -z, z), torch.where(on_y, x, torch.where(z >= 0, x, -x)))
    tc = torch.where(on_x, -y, torch.where(on_y, torch.where(y >= 0, z, -z), -y))
    ma = torch.where(on_x, ax, torch.where(on_y, ay, az))
    return face, sc / ma, tc / ma


def _cube_bilinear(mip, d):
    size = mip.shape[1] - 2
    face, pc, pt = _cube_coords(d)
    x, y = (pc + 1) * 0.5 * size - 0.5, (pt + 1) * 0.5 * size - 0.5
    fx, fy = torch.floor(x), torch.floor(y)
    ax, ay = (x - fx)[:, None], (y - fy)[:, None]
    i, j = fx.long() + 1, fy.long() + 1
    return ((mip[face, j, i] * (1 - ax) + mip[face, j, i + 1] * ax) * (1 - ay)
            + (mip[face, j + 1, i] * (1 - ax) + mip[face, j + 1, i + 1] * ax) * ay)


def _matrix(values):
    return torch.tensor(list(values), dtype=F64, device="cuda").reshape(4, 4).T


def _clamped_bilinear(img, x, y):
    h, w = img.shape[:2]
    fx, fy = torch.floor(x), torch.floor(y)
    ax, ay = (x - fx)[:, None], (y - fy)[:, None]
    x0, x1 = fx.long().clamp(0, w - 1), (fx.long() + 1).clamp(0, w - 1)
    y0, y1 = fy.long().clamp(0, h - 1), (fy.long() + 1).clamp(0, h - 1)
    return ((img[y0, x0] * (1 - ax) + img[y0, x1] * ax) * (1 - ay)
            + (img[y1, x0] * (1 - ax) + img[y1, x1] * ax) * ay)


def _view_rays(g, w: int, h: int, px, py):
    ndc = torch.stack([(px + 0.5) / w * 2 - 1, (py + 0.5) / h * 2 - 1, torch.zeros_like(px), torch.ones_like(px)], -1)
    eye = (ndc @ _matrix(g.inverse_projection).T)[:, :3]
    return eye @ _matrix(g.inverse_view)[:3, :3].T


def _ssao64(case, state, pos, depth, P, N, px, py):
    d, g, w, h = state["ssao"], state["globals"], case["width"], case["height"]
    noise = torch.tensor([list(r)[:3] for r in d.noise], dtype=F64, device="cuda")
    r = noise[(px.long() & 3) + 4 * (py.long() & 3)]
    T = _unit(r - N * _dot(r, N)[:, None])
    B = torch.cross(N, T, dim=-1)
    view = _matrix(g.view)
    vp = _matrix(g.projection) @ view
    homog = lambda q: torch.cat([q, torch.ones_like(q[:, :1])], 1)  # noqa: E731
    here = -(homog(P) @ view.T)[:, 2]
    occluded = torch.zeros_like(here)
    for k in range(d.samples):
        kx, ky, kz = list(d.kernel[k])[:3]
        S = P + d.radius * (T * kx + B * ky + N * kz)
        clip = homog(S) @ vp.T
        sd = -(homog(S) @ view.T)[:, 2]
        x = torch.floor((0.5 * clip[:, 0] / clip[:, 3] + 0.5) * w)
        y = torch.floor((0.5 * clip[:, 1] / clip[:, 3] + 0.5) * h)
        ok = (clip[:, 3] > 0) & (x >= 0) & (x < w) & (y >= 0) & (y < h)
        q = depth[torch.where(ok, y * w + x, 0.0).long()]
        t = (d.radius / (here - q).abs()).clamp(0, 1)
        occluded += torch.where(ok & (q <= sd - d.bias), t * t * (3 - 2 * t), 0.0)
    return 1 - occluded / d.samples


def _exact_resolve(case: dict, state: dict):
    w, h, g = case["width"], case["height"], state["globals"]
    pos, nrm, alb, mro = (p.reshape(-1, 4) for p in state["gbuffer"].planes)
    v = state["ibl"].views()
    env = _split_pyramid(state["ibl"].environment_tensor(), v.env_width)[..., :3].to(F64)
    flat = state["ibl"].prefiltered_tensor()[:, :3].to(F64)
    mips, at = [], 0
    for m in range(v.prefiltered_mips):
        s = max(1, v.prefiltered_size >> m)
        mips.append(_bordered(flat[at:at + 6 * s * s].reshape(6, s, s, 3), s))
        at += 6 * s * s
    irr = _bordered(state["ibl"].irradiance_tensor()[:, :3].to(F64).reshape(6, v.irradiance_size, -1, 3),
                    v.irradiance_size)
    lut = state["ibl"].lut_tensor().to(F64).reshape(v.brdf_lut_size, v.brdf_lut_size, 2)
    lights = state["lights"].to(F64)
    depth = None
    if state["ssao"] is not None:
        view = _matrix(g.view)
        depth = -(pos[:, :3].to(F64) @ view[2, :3] + view[2, 3])
        depth = torch.where(pos[:, 3] == 0, math.inf, depth)
    out = torch.ones(w * h, 4, dtype=F64, device="cuda")
    for a, b in _rows(w * h, 4):
        i = torch.arange(a, b, device="cuda")
        px, py = (i % w).to(F64), torch.div(i, w, rounding_mode="floor").to(F64)
        ray = _view_rays(g, w, h, px, py)
        color = torch.zeros(b - a, 3, dtype=F64, device="cuda")
        sky = pos[a:b, 3] == 0
        d = ray[sky]
        u = torch.atan2(d[:, 2], d[:, 0]) / (2 * math.pi) + 0.5
        t = 0.5 - torch.atan2(d[:, 1], torch.hypot(d[:, 0], d[:, 2])) / math.pi
        color[sky] = _clamped_bilinear(env, u * v.env_width - 0.5, t * v.env_height - 0.5)
        at = (~sky).nonzero()[:, 0]
        if len(at):
            P, V = pos[a + at, :3].to(F64), _unit(ray[at])
            N = _unit(nrm[a + at, :3].to(F64))
            base, mat = alb[a + at, :3].to(F64), mro[a + at].to(F64)
            metal, rough, ao = mat[:, 0:1], mat[:, 1:2], mat[:, 2:3]
            R = V - 2 * _dot(N, V)[:, None] * N
            lod = (rough[:, 0] * (len(mips) - 1)).clamp(0, len(mips) - 1)
            l0 = torch.floor(lod).long()
            frac = (lod - l0)[:, None]
            refl = torch.zeros_like(P)
            for m in range(len(mips)):
                for level, weight in ((l0, 1 - frac), ((l0 + 1).clamp(max=len(mips) - 1), frac)):
                    sel = level == m
                    refl[sel] += _cube_bilinear(mips[m], R[sel]) * weight[sel]
            if depth is not None:
                ao = _ssao64(case, state, pos, depth, P, N, px[at], py[at])[:, None]
            nv = (-_dot(N, V)).clamp_min(0)[:, None]
            ab = _clamped_bilinear(lut, nv[:, 0] * v.brdf_lut_size - 0.5, rough[:, 0] * v.brdf_lut_size - 0.5)
            F0 = 0.04 + (base - 0.04) * metal
            dF = torch.maximum(1 - rough, F0) - F0
            kd = base * (1 - metal)
            F = F0 + dF * (1 - nv) ** 5
            c = (_cube_bilinear(irr, N) * (1 - F) * kd + refl * (F * ab[:, :1] + ab[:, 1:])) * ao
            alpha = rough * rough
            k = (alpha + 1) ** 2 / 8
            for light in lights:
                to = light[:3] - P
                d2 = _dot(to, to)[:, None]
                L = to / torch.sqrt(d2)
                nl = _dot(N, L).clamp_min(0)[:, None]
                half = V + L
                nh = (_dot(N, half)[:, None] / half.norm(dim=-1, keepdim=True)).clamp_min(0)
                F = F0 + dF * (1 - nh) ** 5
                D = alpha ** 2 / (math.pi * (nh * nh * (alpha ** 2 - 1) + 1) ** 2)
                G = nv / (nv * (1 - k) + k) * nl / (nl * (1 - k) + k)
                c = c + ((1 - F) * kd / math.pi + D * F * G / (4 * nl * nv + 1e-4)) * light[4:7] * nl / d2
            color[at] = c
        if case["tonemap"]:
            color = 1 - torch.exp(-color * g.exposure)
        out[a:b, :3] = color
    return out


# Rasterization: every (triangle, pixel of its box) pair, nearest hit kept.
def _slots(x0, x1, y0, y1):
    """Pairs (triangle, x, y) of inclusive integer boxes, in ranges."""
    w, h = (x1 - x0 + 1).clamp_min(0), (y1 - y0 + 1).clamp_min(0)
    area = w * h
    order = torch.arange(len(area), device="cuda")[area > 0]
    end = torch.cumsum(area[order], 0)
    lo = 0
    while lo < len(order):
        first = int(end[lo - 1]) if lo else 0
        hi = max(lo + 1, int(torch.searchsorted(end, torch.tensor(first + CHUNK, device="cuda"))))
        t = torch.repeat_interleave(order[lo:hi], area[order[lo:hi]])
        k = torch.arange(len(t), device="cuda") + first - (end - area[order])[lo:hi].repeat_interleave(
            area[order[lo:hi]])
        yield t, x0[t] + k % w[t], y0[t] + torch.div(k, w[t], rounding_mode="floor")
        lo = hi


def _edges(v):
    """Edge functions (b x c, c x a, a x b), plane normal and a . n."""
    a, b, c = v.unbind(1)
    n = torch.cross(b - a, c - a, dim=-1)
    return [torch.cross(b, c, dim=-1), torch.cross(c, a, dim=-1), torch.cross(a, b, dim=-1)], n, _dot(a, n)


def _boxes(corner_x, corner_y, w: int, h: int):
    """Inclusive pixel boxes of projected corners (t, k), one pixel wider;
    corners that project nowhere are NaN."""
    lo = lambda c: torch.nan_to_num(c, nan=math.inf).amin(1).clamp(-3, 1e6)  # noqa: E731
    hi = lambda c: torch.nan_to_num(c, nan=-math.inf).amax(1).clamp(-3, 1e6)  # noqa: E731
    return ((lo(corner_x).floor().long() - 1).clamp_min(0), (hi(corner_x).ceil().long() + 1).clamp_max(w - 1),
            (lo(corner_y).floor().long() - 1).clamp_min(0), (hi(corner_y).ceil().long() + 1).clamp_max(h - 1))


def _exact_shadow(case: dict, state: dict):
    size, near, far = case["size"], 0.01, 1000.0
    tri = state["positions"].to(F64)[state["indices"].long()]
    out = torch.ones(case["lights"], 6, size, size, dtype=F64, device="cuda")
    turn = {2: (1, 1, -1), 3: (1, 1, -1)}  # the reference's face cameras against the Vulkan faces
    axes = [((0, 0, -1), (0, -1, 0), (1, 0, 0)), ((0, 0, 1), (0, -1, 0), (-1, 0, 0)),
            ((1, 0, 0), (0, 0, 1), (0, 1, 0)), ((1, 0, 0), (0, 0, -1), (0, -1, 0)),
            ((1, 0, 0), (0, -1, 0), (0, 0, 1)), ((-1, 0, 0), (0, -1, 0), (0, 0, -1))]
    for li, light in enumerate(state["lights"].lights.to(F64)):
        v = tri - light[:3]
        v = v[_edges(v)[2] < 0]  # front faces
        for face in range(6):
            basis = torch.tensor(axes[face], dtype=F64, device="cuda") * torch.tensor(
                turn.get(face, (-1, 1, 1)), dtype=F64, device="cuda")  # rows: s, t, depth
            q = v @ basis.T
            inside = (q[..., 2] >= 0.5 * near).any(1)
            if not bool(inside.any()):
                continue
            q = q[inside]
            # Corners in front of the plane at near / 2, and the edges' crossings of it.
            nxt = q.roll(-1, 1)
            cross = (q[..., 2] >= 0.5 * near) != (nxt[..., 2] >= 0.5 * near)
            u = (0.5 * near - q[..., 2]) / (nxt[..., 2] - q[..., 2])
            cut = q + u[..., None] * (nxt - q)
            keep = lambda p, m: torch.where(m[..., None], p, math.nan)  # noqa: E731
            corners = torch.cat([keep(q, q[..., 2] >= 0.5 * near), keep(cut, cross)], 1)
            px = (corners[..., 0] / corners[..., 2] + 1) * 0.5 * size - 0.5
            py = (corners[..., 1] / corners[..., 2] + 1) * 0.5 * size - 0.5
            e, n, det = _edges(q)
            flat = out[li, face].view(-1)
            for t, x, y in _slots(*_boxes(px, py, size, size)):
                d = torch.stack([(2 * x + 1) / size - 1, (2 * y + 1) / size - 1, torch.ones_like(x)], -1).to(F64)
                # The face basis may mirror space: the sign of det in it decides "inside".
                sign = torch.sign(det[t])
                hit = (sign * _dot(d, e[0][t]) >= 0) & (sign * _dot(d, e[1][t]) >= 0) & (sign * _dot(d, e[2][t]) >= 0)
                depth = det[t] / _dot(d, n[t])
                hit &= (depth >= near) & (depth <= far)
                value = (depth * d.norm(dim=-1) / far).clamp_max(1.0)
                flat.scatter_reduce_(0, (y * size + x)[hit], value[hit], "amin")
    return out


def _exact_gbuffer(case: dict, state: dict):
    w, h, g, mesh = case["width"], case["height"], state["globals"], state["mesh"]
    idx = mesh.indices.long()
    vertices = mesh.positions.to(F64)[idx]
    eye = _matrix(g.inverse_view)[:3, 3]
    v = vertices - eye
    e, n, det = _edges(v)
    # The whole mesh lies in front of this camera: no near-plane clipping.
    clip = torch.cat([vertices, torch.ones_like(vertices[..., :1])], -1) @ (
        _matrix(g.projection) @ _matrix(g.view)).T
    px = (clip[..., 0] / clip[..., 3] + 1) * 0.5 * w - 0.5
    py = (clip[..., 1] / clip[..., 3] + 1) * 0.5 * h - 0.5
    x0, x1, y0, y1 = _boxes(px, py, w, h)
    x1 = torch.where(det < 0, x1, x0 - 1)
    best = torch.full((w * h,), math.inf, dtype=F64, device="cuda")
    found = []
    for t, x, y in _slots(x0, x1, y0, y1):
        d = _view_rays(g, w, h, x.to(F64), y.to(F64))
        f = torch.stack([_dot(d, e[k][t]) for k in range(3)], -1)
        hit = (f <= 0).all(-1) & (_dot(d, n[t]) < 0)
        ray = (det[t] / _dot(d, n[t]))[hit]
        at = (y * w + x)[hit]
        best.scatter_reduce_(0, at, ray, "amin")
        found.append((at, ray, t[hit], f[hit]))
    planes = [torch.zeros(w * h, 4, dtype=F64, device="cuda") for _ in range(4)]
    for p in planes[1:]:
        p[:, 3] = 1.0
    for at, ray, t, f in found:
        sel = ray == best[at]
        at, t, f = at[sel], t[sel], f[sel]
        bary = f / f.sum(-1, keepdim=True)
        for p, src in zip(planes, (mesh.positions, mesh.normals, mesh.colors, mesh.mro)):
            p[at, :3] = (src.to(F64)[idx[t]] * bary[..., None]).sum(1)
            p[at, 3] = 1.0
    return [p.reshape(h, w, 4) for p in planes]


def exact(case: dict, seed: int):
    """The 64-bit values of run()'s outputs.  None for a whole frame: its
    textured, alpha-tested, marched passes feed decisions (coverage, discards,
    march hits) of one pass into the next, so no value is exact there."""
    kind = case["kind"]
    if kind == "frame":
        return None
    state = prepare(case, seed)
    if kind == "resolve":
        return _exact_resolve(case, state)
    if kind == "shadow":
        return _exact_shadow(case, state)
    if kind == "gbuffer":
        return _exact_gbuffer(case, state)
    if kind == "labels":
        return _exact_labels(case, state)
    if kind in ("train", "infer"):
        return _exact_mlp(case, state)
    if kind == "batch":
        return [_exact_prefilter(_pyramid64(env), w // 4, case["mips"], case["samples"])
                for env, w in zip(state["envs"], _batch_widths(case))]
    levels = _pyramid64(state["env"])
    return [torch.cat([p.reshape(-1, 4) for p in levels]),
            _exact_prefilter(levels, case["cube"], case["mips"], case["samples"]),
            _exact_irradiance(levels, case["irradiance"], case["theta"]), _exact_lut(case["lut"], 1024)]
