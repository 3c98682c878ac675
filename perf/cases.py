"""Workloads of this framework, from single ray batches to whole frames.

Each case stands for a call that a program using the framework makes, through
the Python package or the C ABI underneath it.  Kinds:

query   a batch of rays against a scene already on the GPU: picking, range
        sensors and line-of-sight tests of a simulator (host rays, or rays
        and hits that stay on the GPU)
build   a scene is loaded (every BLAS and the TLAS are built) and answers a
        batch of rays; what a program pays at each scene change
deform  one geometry's vertices move (cloth, soft bodies): refit, then a
        batch of contact rays
step    one step of a simulator: every body has a new pose, one camera image
frame   one image of a scene, with the schedule the renderer has by itself
        or with one that was tuned before and is pinned
envs    one frame of many environments for training agents, targets left on
        the GPU
denoise the U-Net on render targets in GPU memory
noisy   a 1-sample frame and its denoise
train   loss and gradients of a batch of training images
"""
import ctypes as C
import math

import numpy as np
import torch

from kuafu_amd import abi, scenes
from kuafu_amd.api import GpuScene, Renderer, camera_ubo, mat_from_rows, mat_rotate, mat_translate
from kuafu_amd.denoiser import WEIGHTS, Denoiser

DEV = "cuda"


# ------------------------------------------------------------------ cases
def listed():
    return [
        # a lidar or picking query of a small scene: latency of one call
        dict(name="query_4k_spheres", kind="query", scene="spheres", rays=4096, host=True, any=False),
        # a sensor simulation whose rays are made and used on the GPU
        dict(name="query_2m_field_device", kind="query", scene="field", rays=1 << 21, host=False, any=False),
        # loading a scene of 256 distinct meshes, 1.3 M triangles
        dict(name="build_256x5120", kind="build", geoms=256, subdiv=4, same=False, rays=4096),
        # a soft body of 82 k triangles among rigid ones
        dict(name="deform_82k", kind="deform", subdiv=6, bodies=64, rays=16384),
        # a simulator's step: 64 moving bodies, soft lights, a 640 x 360 camera
        dict(name="step_640x360_4spp_soft", kind="step", width=640, height=360, spp=4, depth=6, soft=True),
        # the smallest configured frame
        dict(name="frame_256x256_4spp", kind="frame", scene="spheres", width=256, height=256, spp=4, depth=4,
             tuned=False, graph=False),
        # an infrared camera under a dot projector
        dict(name="frame_720p_32spp_projector", kind="frame", scene="projector", width=1280, height=720, spp=32,
             depth=6, tuned=False, graph=False),
        # the headline frame, schedule tuned before
        dict(name="frame_1080p_16spp", kind="frame", scene="field", width=1920, height=1080, spp=16, depth=8,
             tuned=True, graph=False),
        # 128 environments per frame, replayed as a graph, schedule left alone
        dict(name="envs_128x512x512_8spp", kind="envs", envs=128, size=512, spp=8, depth=6, tuned=False, graph=True),
        # interactive preview: 1 sample per pixel, denoised
        dict(name="noisy_1080p_denoised", kind="noisy", width=1920, height=1080, spp=1, depth=8),
        # the denoise of a batch of environments' images
        dict(name="denoise_32x512x512", kind="denoise", images=32, height=512, width=512),
        # a training batch of the denoiser
        dict(name="train_8x256x256", kind="train", images=8, height=256, width=256),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["query", "query", "build", "deform", "step", "frame", "frame", "envs", "denoise", "noisy",
                       "train"])
    if kind == "query":
        host = rng.random() < 0.5
        return dict(kind=kind, scene=rng.choice(["spheres", "field", "projector"]),
                    rays=log(64, 1 << 19 if host else 1 << 21), host=host, any=host and rng.random() < 0.5)
    if kind == "build":
        subdiv = rng.choice([1, 2, 3, 4, 5])
        return dict(kind=kind, geoms=log(1, min(400, 1310720 // (20 * 4 ** subdiv))), subdiv=subdiv,
                    same=rng.random() < 0.5, rays=log(256, 65536))
    if kind == "deform":
        return dict(kind=kind, subdiv=rng.choice([2, 3, 4, 5, 6]), bodies=log(1, 256), rays=log(256, 65536))
    if kind == "step":
        w = log(96, 1280)
        return dict(kind=kind, width=w, height=max(48, int(w * rng.uniform(0.5, 1.0))), spp=rng.choice([1, 2, 4, 8]),
                    depth=rng.choice([4, 6, 8]), soft=rng.random() < 0.5)
    if kind == "frame":
        w = log(96, 1920)
        scene = rng.choice(["spheres", "field", "projector"])
        return dict(kind=kind, scene=scene, width=w, height=max(48, int(w * rng.uniform(0.5, 0.6))), spp=log(1, 24),
                    depth=rng.choice([3, 4, 6, 8]), tuned=scene in _TUNED and rng.random() < 0.4,
                    graph=rng.random() < 0.4)
    if kind == "envs":
        size = rng.choice([96, 128, 200, 256, 384])
        return dict(kind=kind, envs=log(2, 128), size=size, spp=rng.choice([1, 2, 4, 8]), depth=rng.choice([4, 6]),
                    tuned=rng.random() < 0.5, graph=rng.random() < 0.7)
    if kind == "denoise":
        w = log(64, 1920)
        h = max(48, int(w * rng.uniform(0.5, 1.0)))
        return dict(kind=kind, images=max(1, log(1, max(1, 8388608 // (w * h)))), height=h, width=w)
    if kind == "noisy":
        w = log(160, 1920)
        return dict(kind=kind, width=w, height=max(96, int(w * rng.uniform(0.5, 0.6))), spp=rng.choice([1, 2, 4]),
                    depth=rng.choice([4, 6, 8]))
    return dict(kind=kind, images=rng.choice([1, 2, 3, 4, 6, 8]), height=16 * rng.randint(2, 16),
                width=16 * rng.randint(2, 16))


# ------------------------------------------------------------------ scenes
def _workload(case, seed):
    """The scene of a case and a camera of its size."""
    w, h = case.get("width", 640), case.get("height", 360)
    spp, depth = case.get("spp", 1), case.get("depth", 6)
    kind = case.get("scene", "field")
    if kind == "spheres":
        return scenes.config1(width=w, height=h, spp=spp, path_depth=depth, seed=seed)
    if kind == "projector":
        return scenes.config3(width=w, height=h, spp=spp, path_depth=depth, seed=seed)
    return scenes.config2(width=w, height=h, spp=spp, path_depth=depth, seed=seed)


# Where the rays of a query start and what they are aimed at, per scene.
_RAY_BOX = {"spheres": ((0.0, 2.0, 6.0), 0.5, (0.0, 0.5, 0.0), (3.2, 0.6, 1.0)),
            "projector": ((0.0, -1.8, 1.8), 0.3, (0.0, 0.0, 0.1), (1.5, 1.5, 0.3)),
            "field": ((0.0, -30.0, 6.0), 4.0, (0.0, 0.0, 0.0), (10.0, 10.0, 10.0))}


def _rays(scene, n, seed):
    """n rays from around a sensor to points spread over the scene, (n, 8) float32: origin, tmin, direction, tmax."""
    eye, spread, centre, half = _RAY_BOX[scene]
    rng = np.random.default_rng(seed)
    r = np.empty((n, 8), np.float32)
    r[:, 0:3] = np.asarray(eye) + spread * rng.uniform(-1, 1, (n, 3))
    d = np.asarray(centre) + np.asarray(half) * rng.uniform(-1, 1, (n, 3)) - r[:, 0:3]
    r[:, 4:7] = d / np.linalg.norm(d, axis=1, keepdims=True)
    r[:, 3] = 0.001
    r[:, 7] = 1e4
    return r


def _host_rays(r):
    return np.ascontiguousarray(r).view(abi.RAY_DTYPE).reshape(-1)


def _hits(h):
    """The fields of a hit array; ids as signed integers (-1: no hit)."""
    return {"t": h["t"], "b1": h["b1"], "b2": h["b2"], "inst": h["inst"].view(np.int32), "prim": h["prim"].view(np.int32),
            "back": h["back"].view(np.int32)}


def _meshes(case, seed):
    """Many bodies in a cube, each with a mesh of its own (or all with the same)."""
    rng = np.random.default_rng(seed)
    v0, tris = scenes.icosphere(case["subdiv"])
    s = scenes.SceneData()
    for _ in range(case["geoms"]):
        v = v0
        if not case["same"]:
            v = v0.copy()
            k = rng.normal(size=(3, 3))
            bump = 1.0 + 0.15 * np.sin(v0["pos"] @ k.T * 3.0).prod(axis=1, keepdims=True)
            v["pos"] = v0["pos"] * bump.astype(np.float32)
        g = s.add_geometry(v, tris, scenes.material(diffuse=tuple(rng.uniform(0, 1, 3))))
        s.add_instance(g, mat_from_rows(scenes.random_rotation(rng) * rng.uniform(0.2, 1.5), rng.uniform(-10, 10, 3)))
    return s


def _soft_body(case, seed):
    """A dense ball among rigid ones; two shapes of it."""
    rng = np.random.default_rng(seed)
    v0, tris = scenes.icosphere(case["subdiv"])
    rv, rt = scenes.icosphere(3)
    s = scenes.SceneData()
    g = s.add_geometry(v0, tris, scenes.material())
    s.add_instance(g, mat_from_rows(scenes.random_rotation(rng) * 6.0, (0.0, 0.0, 0.0)))
    for _ in range(case["bodies"]):
        b = s.add_geometry(rv, rt, scenes.material())
        s.add_instance(b, mat_from_rows(scenes.random_rotation(rng) * rng.uniform(0.2, 1.5), rng.uniform(-10, 10, 3)))
    k = rng.normal(size=(3, 3))
    v1 = v0.copy()
    v1["pos"] = v0["pos"] * (1.0 + 0.1 * np.sin(2.0 * v0["pos"] @ k.T).sum(1, keepdims=True)).astype(np.float32)
    return s, v1


def _moved(data, seed):
    """The instances of a scene after a simulator's step: everything but the ground has moved a little."""
    rng = np.random.default_rng(seed + 77)
    inst = data.arrays()["inst"].copy()
    for i in range(1, len(inst)):
        m = inst[i]["transform"].reshape(4, 4)
        step = mat_rotate(rng.uniform(-0.3, 0.3), (0, 0, 1), mat_translate(tuple(rng.uniform(-0.05, 0.05, 3) * (1, 1, 0))))
        moved = (m.astype(np.float64) @ step.astype(np.float64)).astype(np.float32)
        inst[i]["transform"] = moved.ravel()
    return inst


class _Target:
    """A render target in GPU memory, for torch; keeps its renderer."""

    def __init__(self, r, k):
        self.renderer = r
        self.__cuda_array_interface__ = dict(data=(int(r.device_target(k)), False), shape=(r.h_, r.w, 4), typestr="<f4",
                                             version=3)


def _targets(r, which=(0, 1, 2)):
    out = {}
    for k in which:
        t = torch.as_tensor(_Target(r, k), device=DEV)
        t.renderer = r  # the tensor is a view: the renderer owns the memory
        out[("rgba", "albedo", "normal")[k]] = t
    return out


# Schedules that the autotuner picked for these workloads.
_TUNED = {"field": dict(samples_per_batch=16, refill=8, grab=256, tail_bounce=5, grab0=1024, grab_shadow=128),
          "projector": dict(samples_per_batch=32, refill=16, grab=1024, tail_bounce=6, grab0=1024, grab_shadow=0),
          "envs": dict(samples_per_batch=2, refill=16, grab=1024, tail_bounce=5, grab0=1024, grab_shadow=0, tail_pairs=0)}


# ------------------------------------------------------------------ images
def _images(n, h, w, seed):
    """Render targets as a 1-sample frame leaves them: smooth surfaces, noisy radiance with rare bright samples."""
    g = torch.Generator(device=DEV).manual_seed(int(seed))

    def smooth(c, cells):
        low = torch.rand(n, c, cells, cells, generator=g, device=DEV)
        return torch.nn.functional.interpolate(low, size=(h, w), mode="nearest" if cells > 4 else "bilinear")

    albedo = (smooth(3, 12) * 0.3).clamp(0, 1 / math.pi)
    normal = torch.nn.functional.normalize(smooth(3, 9) - 0.5 + 0.2 * (smooth(3, 3) - 0.5), dim=1)
    light = 4.0 * smooth(1, 3) * smooth(1, 4)
    noise = torch.empty(n, 1, h, w, device=DEV).exponential_(1.0, generator=g)
    noise = noise * (1.0 + 40.0 * (torch.rand(n, 1, h, w, generator=g, device=DEV) < 0.002).float())
    clean = albedo * light
    one = torch.ones(n, 1, h, w, device=DEV)

    def rgba(x):
        return torch.cat([x, one], 1).permute(0, 2, 3, 1).reshape(n * h, w, 4).contiguous()

    return rgba(clean * noise), rgba(albedo), rgba(normal), clean.permute(0, 2, 3, 1).contiguous()


# ------------------------------------------------------------------ prepare, run
def prepare(case, seed):
    kind = case["kind"]
    abi.check(abi.lib().kf_init(0))
    s = {"kind": kind, "case": case}
    if kind == "query":
        wl = _workload(case, seed)
        s["scene"] = GpuScene(wl.data)
        r = _rays(case["scene"], case["rays"], seed + 1)
        s["any"] = case["any"]
        if case["host"]:
            s["rays"] = _host_rays(r)
        else:
            s["rays"] = torch.from_numpy(r).to(DEV)
            s["hits"] = torch.empty(case["rays"], 6, dtype=torch.int32, device=DEV)
            torch.cuda.synchronize()
    elif kind == "build":
        s["data"] = _meshes(case, seed)
        s["desc"] = s["data"].desc()
        s["rays"] = _host_rays(_rays("field", case["rays"], seed + 1))
    elif kind == "deform":
        data, s["verts"] = _soft_body(case, seed)
        s["scene"] = GpuScene(data)
        s["rays"] = _host_rays(_rays("field", case["rays"], seed + 1))
    elif kind == "step":
        wl = scenes.config3(width=case["width"], height=case["height"], spp=case["spp"], path_depth=case["depth"],
                            seed=seed, camera="rgb")
        if case["soft"]:
            wl.data.set_directional_light((0.2, 0.3, -1.0), (1, 1, 1), 0.5, 0.1)
            wl.data.add_point_light((0.6, -0.6, 1.6), (1, 1, 1), 3.0, radius=0.2)
        s["wl"], s["scene"] = wl, GpuScene(wl.data)
        s["inst"] = _moved(wl.data, seed)
        s["renderer"] = Renderer(wl.width, wl.height)
        s["targets"] = _targets(s["renderer"], (0,))
    elif kind in ("frame", "noisy"):
        wl = _workload(case, seed)
        s["wl"], s["scene"], s["renderer"] = wl, GpuScene(wl.data), Renderer(wl.width, wl.height)
        s["targets"] = _targets(s["renderer"], (0,))
        if kind == "noisy":
            s["renderer"].set_schedule(1, 8, 64, 3, 256, 64, tail_pairs=0)
            s["denoiser"] = Denoiser()
        elif case["tuned"]:
            s["renderer"].set_schedule(**_TUNED[case["scene"]])
    elif kind == "envs":
        wl = scenes.config5(n_env=case["envs"], size=case["size"], spp=case["spp"], path_depth=case["depth"], seed=seed)
        s["wl"], s["scene"], s["renderer"] = wl, GpuScene(wl.data), Renderer(wl.width, wl.height)
        s["targets"] = _targets(s["renderer"])
        if case["tuned"]:
            s["renderer"].set_schedule(**_TUNED["envs"])
    elif kind == "denoise":
        s["denoiser"] = Denoiser()
        s["rgba"], s["albedo"], s["normal"], _ = _images(case["images"], case["height"], case["width"], seed)
        s["out"] = torch.empty_like(s["rgba"])
        torch.cuda.synchronize()
    elif kind == "train":
        n, h, w = case["images"], case["height"], case["width"]
        s["denoiser"] = Denoiser()
        rgba, albedo, normal, clean = _images(n, h, w, seed)
        s["inputs"] = torch.cat([x.reshape(n, h, w, 4)[..., :3] for x in (rgba, albedo, normal)], -1).cpu().numpy()
        s["targets"] = clean.cpu().numpy()
    else:
        raise ValueError(kind)
    return s


def run(s):
    kind, case = s["kind"], s["case"]
    if kind == "query":
        if s["any"]:
            return s["scene"].trace_any(s["rays"])
        if case["host"]:
            return _hits(s["scene"].trace_closest(s["rays"]))
        abi.check(abi.lib().kf_trace_closest_device(s["scene"].h, s["rays"].data_ptr(), case["rays"],
                                                    s["hits"].data_ptr(), None))
        h = s["hits"]
        f = h.view(torch.float32)
        return {"t": f[:, 0], "inst": h[:, 1], "prim": h[:, 2], "b": f[:, 3:5], "back": h[:, 5]}
    if kind == "build":
        L = abi.lib()
        h = C.c_void_p()
        abi.check(L.kf_scene_create(C.byref(s["desc"]), C.byref(h)))
        hits = np.zeros(len(s["rays"]), abi.HIT_DTYPE)
        abi.check(L.kf_trace_closest(h, abi.ptr(s["rays"]), len(s["rays"]), abi.ptr(hits)))
        L.kf_scene_destroy(h)
        return _hits(hits)
    if kind == "deform":
        s["scene"].update_geometry(0, s["verts"])
        return _hits(s["scene"].trace_closest(s["rays"]))
    if kind == "denoise":
        s["denoiser"].infer_device(s["rgba"].data_ptr(), s["albedo"].data_ptr(), s["normal"].data_ptr(), case["width"],
                                   case["height"], s["out"].data_ptr(), n_images=case["images"])
        return s["out"]
    if kind == "train":
        loss, grads = s["denoiser"].gradients(s["inputs"], s["targets"])
        return {"loss": loss, "grads": grads}
    wl, r = s["wl"], s["renderer"]
    if kind == "step":
        s["scene"].update_instances(s["inst"])
        r.render(s["scene"], wl.cam, wl.pc, seed=wl.seed)
        return {"image": r.download_bgra8(), **s["targets"]}
    if kind == "frame":
        r.render(s["scene"], wl.cam, wl.pc, seed=wl.seed, use_graph=case["graph"])
        image = r.download_gray32f() if case["scene"] == "projector" else r.download_bgra8()
        return {"image": image, **s["targets"]}
    if kind == "noisy":
        r.render(s["scene"], wl.cam, wl.pc, seed=wl.seed, use_graph=True)
        s["denoiser"].apply(r)
        return s["targets"]
    r.render_envs(s["scene"], wl.cam, wl.pc, seed=wl.seed, use_graph=case["graph"])
    return s["targets"]


# ------------------------------------------------------------------ work
_CH = (32, 64, 96, 128, 160)


def _unet_flops(pixels):
    """Multiplies and adds of the network's 19 convolutions, true channel counts."""
    f = 0.0
    for l, c in enumerate(_CH):
        first = 9 if l == 0 else _CH[l - 1]
        f += (first * c + c * c) / 4.0 ** l
    for l in range(4):
        f += ((_CH[l] + _CH[l + 1]) * _CH[l] + _CH[l] * _CH[l]) / 4.0 ** l
    return 18.0 * pixels * (f + _CH[0] * 3)


def _ray_flops(rays, nodes):
    """About 100 operations per four-wide box test and 60 per triangle or instance."""
    return rays * (100.0 * nodes + 60.0 * 4)


# Rays per path (camera, bounce and shadow) and node records per ray, counted on these scenes.
_RAYS = {"spheres": (3.5, 5.0), "projector": (13.9, 8.0), "field": (1.57, 13.0), "envs": (3.3, 5.8)}


def work(case):
    kind = case["kind"]
    if kind == "query":
        n = case["rays"]
        return dict(bytes=n * (32 + (1 if case["any"] else 24)), flops=_ray_flops(n, _RAYS[case["scene"]][1]))
    if kind == "build":
        tris = case["geoms"] * 20 * 4 ** case["subdiv"]
        # vertices and indices in; node boxes and triangle records out
        return dict(bytes=tris * (24 + 16 + 48 + 64) + case["rays"] * 56.0, flops=tris * 100.0)
    if kind == "deform":
        tris = 20 * 4 ** case["subdiv"]
        return dict(bytes=tris * (24 + 12 + 48 + 64) + case["rays"] * 56.0, flops=tris * 60.0 + _ray_flops(case["rays"], 13))
    if kind == "denoise":
        p = case["images"] * case["height"] * case["width"]
        return dict(bytes=p * 64.0, flops=_unet_flops(p))
    if kind == "train":
        p = case["images"] * case["height"] * case["width"]
        return dict(bytes=p * 48.0, flops=3 * _unet_flops(p))
    scene = "envs" if kind == "envs" else "projector" if kind == "step" else case.get("scene", "field")
    pixels = case["envs"] * case["size"] ** 2 if kind == "envs" else case["width"] * case["height"]
    rays, nodes = _RAYS[scene]
    flops = _ray_flops(pixels * case["spp"] * rays, nodes) + (_unet_flops(pixels) if kind == "noisy" else 0.0)
    return dict(bytes=pixels * 52.0, flops=flops)


# ------------------------------------------------------------------ exact
def _mesh_distance(data, inst, rays, verts=None):
    """Distance to the nearest triangle of every ray, in 64 bits (tmax where there is none)."""
    f64 = dict(dtype=torch.float64, device=DEV)
    tri = []
    for k in range(len(inst)):
        g = int(inst[k]["geometry_index"])
        v, ix = data.geoms[g][0], data.geoms[g][1]
        p = torch.tensor((verts[g] if verts and g in verts else v)["pos"].astype(np.float64), **f64)
        m = torch.tensor(inst[k]["transform"].reshape(4, 4).astype(np.float64), **f64)
        tri.append((p @ m[:3, :3] + m[3, :3])[torch.from_numpy(ix.astype(np.int64)).to(DEV)])
    tri = torch.cat(tri)
    r = torch.tensor(rays.astype(np.float64), **f64)
    a, e1, e2 = tri[:, 0], tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0]
    # d . (e1 x e2), and the other determinants, as products of ray and triangle coordinates
    nrm = torch.linalg.cross(e1, e2)
    best = r[:, 7].clone()
    step = max(1, (1 << 27) // len(tri))
    for i in range(0, len(r), step):
        o, d = r[i:i + step, 0:3], r[i:i + step, 4:7]
        od = torch.linalg.cross(o, d)
        det = -(d @ nrm.T)
        # (o - a) x d . e, expanded so that each part is a product of a ray's and a triangle's numbers
        u = (od @ e2.T - d @ torch.linalg.cross(e2, a).T)
        v = -(od @ e1.T - d @ torch.linalg.cross(e1, a).T)
        t = (o @ nrm.T - (a * nrm).sum(1))
        u, v, t = u / det, v / det, t / det
        ok = (u >= -1e-12) & (v >= -1e-12) & (u + v <= 1 + 1e-12) & (t >= r[i:i + step, 3:4]) & (t <= best[i:i + step, None])
        best[i:i + step] = torch.minimum(best[i:i + step], torch.where(ok, t, torch.inf).amin(1))
    return best.cpu().numpy()


def _weights():
    """The network's shipped weights, in 64 bits: per convolution (9, out, in) and the biases."""
    raw = open(WEIGHTS, "rb").read()
    n, at, out = int(np.frombuffer(raw, np.uint32, 1, 8)[0]), 12, []
    for _ in range(n):
        ci, co = (int(x) for x in np.frombuffer(raw, np.uint32, 2, at))
        at += 8
        w = (np.frombuffer(raw, np.uint16, 9 * ci * co, at).astype(np.uint32) << 16).view(np.float32)
        at += 18 * ci * co
        b = np.frombuffer(raw, np.float32, co, at)
        at += 4 * co
        out.append([torch.tensor(w.astype(np.float64).reshape(9, co, ci), device=DEV), torch.tensor(b.astype(np.float64), device=DEV)])
    return out


def _conv(x, w, b):
    n, h, wd, c = x.shape
    p = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
    y = b.expand(n * h * wd, -1)
    for tap in range(9):
        y = y + p[:, tap // 3:tap // 3 + h, tap % 3:tap % 3 + wd].reshape(-1, c) @ w[tap].T
    return y.reshape(n, h, wd, -1)


def _unet(x, P):
    """Output of the network (3 channels) for its input (n, h, w, 32), in 64 bits."""
    k, skips = 0, []
    for l in range(5):
        x = _conv(x, *P[k]).relu()
        x = _conv(x, *P[k + 1]).relu()
        k += 2
        if l < 4:
            skips.append(x)
            x = 0.25 * (x[:, 0::2, 0::2] + x[:, 0::2, 1::2] + x[:, 1::2, 0::2] + x[:, 1::2, 1::2])
    for l in range(3, -1, -1):
        x = torch.cat([skips[l], x.repeat_interleave(2, 1).repeat_interleave(2, 2)], -1)
        x = _conv(x, *P[k]).relu()
        x = _conv(x, *P[k + 1]).relu()
        k += 2
    return _conv(x, *P[k])[..., :3]


def _unet_input(rgb, albedo, normal):
    x = torch.zeros(*rgb.shape[:3], 32, dtype=torch.float64, device=DEV)
    lin = torch.log1p(rgb.double().clamp(0, 1e4))
    x[..., 0:3], x[..., 3:6], x[..., 6:9] = lin, albedo.double() * 3.141592, normal.double()
    return x, lin


def exact(case, seed):
    kind = case["kind"]
    if kind == "query" and not case["any"]:
        wl = _workload(case, seed)
        inst = wl.data.arrays()["inst"]
        tris = sum(len(wl.data.geoms[int(g)][1]) for g in inst["geometry_index"])
        if not case["host"] or tris * case["rays"] > 4e9:
            return None
        t = _mesh_distance(wl.data, inst, _rays(case["scene"], case["rays"], seed + 1))
        return {"t": t, "b1": None, "b2": None, "inst": None, "prim": None, "back": None}
    if kind == "deform":
        data, moved = _soft_body(case, seed)
        tris = len(data.geoms[0][1]) + case["bodies"] * 1280
        if tris * case["rays"] > 4e9:
            return None
        t = _mesh_distance(data, data.arrays()["inst"], _rays("field", case["rays"], seed + 1), {0: moved})
        return {"t": t, "b1": None, "b2": None, "inst": None, "prim": None, "back": None}
    if kind == "denoise":
        n, h, w = case["images"], case["height"], case["width"]
        P, out = _weights(), []
        targets = _images(n, h, w, seed)[:3]
        for i in range(n):
            t = [x[i * h:(i + 1) * h, :, :3].permute(2, 0, 1)[None] for x in targets]
            pad = (0, -w % 16, 0, -h % 16)
            t = [torch.nn.functional.pad(x, pad, mode="replicate").permute(0, 2, 3, 1) for x in t]
            x, lin = _unet_input(*t)
            y = torch.expm1((_unet(x, P) + lin).clamp(max=10.0))[0, :h, :w]
            out.append(torch.cat([y, torch.ones_like(y[..., :1])], -1))
        return torch.cat(out)
    if kind == "train":
        n, h, w = case["images"], case["height"], case["width"]
        rgba, albedo, normal, clean = _images(n, h, w, seed)
        P = _weights()
        for p in P:
            for q in p:
                q.requires_grad_(True)
        x, lin = _unet_input(*(v.reshape(n, h, w, 4)[..., :3] for v in (rgba, albedo, normal)))
        y = _unet(x, P) + lin
        t = clean.double()
        o = torch.expm1(y.clamp(max=10.0))
        loss = (y - torch.log1p(t)).abs().mean() + ((o - t) ** 2 / (t * t + 0.01)).mean()
        loss.backward()
        grads = torch.cat([q.grad.reshape(-1) for p in P for q in p])
        return {"loss": float(loss), "grads": grads.cpu().numpy()}
    return None
