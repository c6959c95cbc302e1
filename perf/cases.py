"""The framework's work as a set of timed cases: what a user's program has it do, through its
public entry points.

Kinds of case:

* ``frame``      one ``MainView.render`` (or ``render_high_accuracy``): ray cast, 8 sample rays,
                 Lyapunov overlay; from the interactive start-up view to 1080p.
* ``batch``      one ``render_batch``: many views of several fields, sizes and steps (escape mode).
* ``surrogate``  one ``render_surrogate`` with the saved weights: RK4 approach, network, RK4
                 fallback, overlay.
* ``train``      ``train_surrogate``: labels, Adam steps, hold-out errors; returns the weights.
* ``flowmap``    ``flowmap`` of host entry states.
* ``infer``      ``surrogate_infer`` of host entry states.
* ``model``      ``update_model`` (the acceleration grid's build) and the first frame after it,
                 as when a user drops a new model on the window.

Frames render on the context's own stream and hand their images over as device tensors
(``device_buffers``), as a program that presents them on the GPU does.
"""
from __future__ import annotations

import functools
import math
import struct

import numpy as np
import torch

import linon_amd as L
from linon_amd import configs, scenes

BENCH = ("swirl", "lens", "hot_air", "warp")
MIRAGES = ("mirage_spherical", "mirage_plane", "mirage_spherical_sigmoid", "mirage_plane_sigmoid")
FLOW_FIELDS = ("swirl", "lens", "hot_air", "warp", "mirage_spherical_sigmoid")
# FP32 operations of the four field evaluations of a step (transcendentals not counted)
FIELD_FLOP = {"swirl": 48, "lens": 64, "hot_air": 217, "warp": 24}
MLP_FLOP = 2 * (198 * 256 + 3 * 256 * 256 + 256 * 7)
F32 = np.float32


# ---------------------------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------------------------
def frame(name, width, height, field, scene, h, adaptive=False, overlay=True, samples=True, weight=1.0, high=False,
          wgsl=False, level=5):
    c = dict(kind="frame", width=width, height=height, field=field, scene=scene, h=h, adaptive=adaptive,
             overlay=overlay, samples=samples, weight=weight, high=high, wgsl=wgsl, level=level)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the interactive default (adaptive h = 0.1, start-up scene and field) in a thumbnail: the
        # smallest frame, where launches and the sample rays' 5000 serial steps count
        frame("startup_96x64", 96, 64, "mirage_spherical_sigmoid", "startup", 0.1, adaptive=True),
        # the repository's CPU-runnable configuration: 256 x 256, Cornell box, swirl, h = 0.01
        frame("swirl_256", 256, 256, "swirl", "cornell", 0.01, overlay=False),
        # the headline workload's heaviest field: 1080p, Cornell box + 20k faces, h = 0.005
        frame("hot_air_1080p", 1920, 1080, "hot_air", "ico", 0.005),
        # an odd window size, the field whose rays are captured by its singularity
        frame("lens_1365x767", 1365, 767, "lens", "ico", 0.005),
        # a field the user typed into the editor (compiled at run time)
        frame("wgsl_hot_air_641x361", 641, 361, "hot_air", "startup", 0.01, wgsl=True),
        # the "Enhance" button on the start-up view: one frame at h = 0.001
        frame("enhance_512x384", 512, 384, "mirage_spherical_sigmoid", "startup", 0.1, adaptive=True, high=True),
        # the batch workload at half its resolutions: views of all fields, sizes and steps
        dict(name="batch_33_half", kind="batch", views=32, scale=2),
        # surrogate + fallback at 1080p, saved weights
        dict(name="surrogate_warp_1080p", kind="surrogate", width=1920, height=1080, field="warp"),
        # surrogate training: the shipped configuration's batch, fewer rays and steps
        dict(name="train_swirl_b65536", kind="train", field="swirl", rays=1 << 20, batch=65536, steps=100, h=0.005,
             coarse_h=0.0),
        # flow map of host states (h = 0.005), an odd number of them
        dict(name="flowmap_hot_air_50001", kind="flowmap", field="hot_air", n=50001, h=0.005),
        # raw network outputs of host states
        dict(name="infer_200k", kind="infer", field="hot_air", n=200_000),
        # a new 20,516-face model and its first frame
        dict(name="model_20k", kind="model", level=5, width=320, height=180),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("frame", "frame", "frame", "frame", "batch", "surrogate", "train", "flowmap", "infer", "model"))
    if kind == "frame":
        w = _log(rng, 48, 1920)
        h = max(32, min(1080, int(w * rng.uniform(0.5, 1.0))))
        style = rng.choice(("interactive", "fixed", "fixed", "wgsl", "enhance"))
        if style == "interactive":
            return frame(None, w, h, rng.choice(MIRAGES + ("rotation",)), "startup", rng.choice((0.1, 0.05)), adaptive=True)
        if style == "enhance":
            w = min(w, 640)
            return frame(None, w, max(32, min(h, w)), rng.choice(MIRAGES), "startup", 0.1, adaptive=True, high=True)
        if style == "wgsl":
            return frame(None, w, h, rng.choice(BENCH), "startup", 0.01, wgsl=True)
        return frame(None, w, h, rng.choice(BENCH + MIRAGES), rng.choice(("ico", "cornell")),
                     rng.choice((0.01, 0.005)), overlay=rng.random() < 0.8, samples=rng.random() < 0.8,
                     weight=rng.choice((1.0, 1.0, 1.0, 0.5)), level=rng.randint(3, 6))
    if kind == "batch":
        return dict(kind="batch", views=rng.randint(3, 40), scale=rng.choice((2, 3, 4, 5, 8)))
    if kind == "surrogate":
        w = _log(rng, 160, 1920)
        return dict(kind="surrogate", width=w, height=max(90, int(w * rng.uniform(0.5, 0.5625))), field=rng.choice(BENCH))
    if kind == "train":
        batch = 64 * _log(rng, 32, 1024)
        field = rng.choice(BENCH)
        return dict(kind="train", field=field, rays=_log(rng, 1 << 16, 1 << 20), batch=batch,
                    steps=rng.randint(5, 100), h=rng.choice((0.005, 0.01)),
                    coarse_h=rng.choice((0.0, configs.SURROGATE_COARSE_H[field])))
    if kind == "flowmap":
        return dict(kind="flowmap", field=rng.choice(FLOW_FIELDS), n=_log(rng, 1, 1 << 19), h=rng.choice((0.005, 0.01)))
    if kind == "infer":
        return dict(kind="infer", field=rng.choice(BENCH), n=_log(rng, 1, 1 << 20))
    return dict(kind="model", level=rng.randint(2, 8), width=_log(rng, 96, 640), height=_log(rng, 64, 360))


# ---------------------------------------------------------------------------------------------
# Inputs and handles
# ---------------------------------------------------------------------------------------------
@functools.lru_cache(maxsize=4)
def _unit_sphere(level):
    return scenes.icosphere_unit(level)


def _ico_scene(level, seed):
    """scenes.benchmark_scene(level, seed) with the unit sphere's subdivision kept."""
    v, f = _unit_sphere(level)
    r = 0.4 + scenes.splitmix_uniform(seed, len(v), -0.05, 0.05)
    return scenes.concat_meshes(scenes.cornell_box_centered(), ((v * r[:, None]).astype(F32), f.astype(np.uint32)))


def _eye(rng, distance=3.0, spread=0.25):
    e = np.array([0.0, 0.0, distance]) + rng.uniform(-spread, spread, 3)
    return tuple(float(x) for x in e)


def _scene(case, seed):
    """(vertices, faces, camera) of a frame: what the user looks at, from where (by the seed)."""
    rng = np.random.default_rng(seed)
    if case["scene"] == "startup":
        v, f, c = scenes.reference_startup_scene()
        cam = L.Camera.arcball_default(np.asarray(c) + rng.uniform(-0.1, 0.1, 3).astype(F32))
        return v, f, cam
    v, f = scenes.cornell_box_centered() if case["scene"] == "cornell" else _ico_scene(case["level"], seed)
    return v, f, L.Camera.look_at(_eye(rng), (0.0, 0.0, 0.0), (0.0, 1.0, 0.0), fov_deg=60.0)


def _settings(case, seed):
    m = np.random.default_rng(seed + 1).uniform(0.3, 0.7, 2)
    return L.Settings.make(field_weight=case.get("weight", 1.0), mouse_pos=(float(m[0]), float(m[1])),
                           overlay_mode=1 if case.get("overlay", True) else 0)


def _integrator(case):
    s = case["samples"]
    return L.Integrator.make(h_initial=case["h"], t_max=5.0, adaptive=case["adaptive"], max_steps=100000,
                             samples_per_ray=100 if s else 0, sample_steps=5000 if s else 0)


def _escape(h, max_steps):
    return L.Integrator.make(h_initial=h, t_max=1e30, adaptive=False, max_steps=max_steps, mode=L.MODE_ESCAPE,
                             escape_radius=2.0, samples_per_ray=0, sample_steps=0, need_mapping=True, clip_exit=True)


class _Buffer:
    """A device pointer of the library as an array interface, for a zero-copy tensor.  Whoever
    holds the tensor holds the view, which owns the memory."""

    def __init__(self, view, ptr, shape, typestr):
        self.view = view
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (ptr, False), "version": 2}


class Images(dict):
    """A view's images as tensors; keeps the view, whose end would free them."""


def _images(view, names, samples=0):
    d = view.device_buffers()
    w, h = d.width, d.height
    at = {"final": (d.final_rgba8, (h, w, 4), "|u1"), "mapping": (d.mapping_rgba32f, (h, w, 4), "<f4"),
          "hit": (d.hit_face_i32, (h, w), "<i4"), "steps": (d.steps_i32, (h, w), "<i4"),
          "lyapunov": (d.lyapunov_f32, (h, w), "<f4"), "samples": (d.ray_samples, (8, samples, 2, 4), "<f4")}
    out = Images({k: torch.as_tensor(_Buffer(view, *at[k]), device="cuda") for k in names})
    out.view = view
    return out


def entry_states(n, seed, radius=2.0, inset=0.005):
    """Entry states of the flow map: on the sphere, pulled inside by up to one step, pointing in."""
    rng = np.random.default_rng(seed)
    p = rng.normal(size=(n, 3))
    p *= (radius - inset * rng.uniform(size=(n, 1))) / np.linalg.norm(p, axis=1, keepdims=True)
    q = rng.normal(size=(n, 3))
    q /= np.linalg.norm(q, axis=1, keepdims=True)
    q[(p * q).sum(1) > 0] *= -1.0
    return np.concatenate([p, q], 1).astype(F32)


def _batch_views(case, seed):
    """The workload's sizes, fields and steps (seed 0), looked at from the seed's eyes."""
    views = configs.batch_views(num_views=case["views"], seed=0, scale=case["scale"])
    for v, other in zip(views, configs.batch_views(num_views=case["views"], seed=seed)):
        v.camera = other.camera
    return views


def _surrogate_view(case, seed):
    rng = np.random.default_rng(seed)
    return L.Camera.look_at(_eye(rng, 3.0, 0.1), (0.0, 0.0, 0.0), (0.0, 1.0, 0.0), fov_deg=60.0)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "frame":
        v, f, cam = _scene(case, seed)
        view = L.MainView(case["width"], case["height"])
        view.update_model(v, f)
        view.update_camera(cam)
        view.update_settings(_settings(case, seed))
        view.set_integrator(_integrator(case))
        if case["wgsl"]:
            view.reload_shader(configs.FIELD_WGSL[case["field"]])
        else:
            view.set_field(case["field"])
        render = view.render_high_accuracy if case["high"] else view.render
        names = ("final", "mapping", "hit", "steps", "lyapunov") + (("samples",) if case["samples"] else ())
        return {"view": view, "render": render, "out": _images(view, names, 100)}
    if kind == "batch":
        # (a batch's images have no device accessor: the program reads them back, and the read-back
        # belongs to the pass)
        view = L.MainView(64, 64)
        view.update_model(*_ico_scene(5, seed))
        view.set_integrator(configs.batch_integrator(max_steps=8000))
        views = _batch_views(case, seed)
        view.set_batch(views)
        # the launch shape the autotuner picks for this workload at full size
        view.set_batch_tuning(waves_per_cu=24, waves_per_block=2, compact_every=256, refill_min=48)
        return {"view": view, "views": len(views)}
    if kind == "surrogate":
        view = L.MainView(case["width"], case["height"])
        view.update_model(np.zeros((0, 3), F32), np.zeros((0, 3), np.uint32))
        view.update_camera(_surrogate_view(case, seed))
        view.update_settings(L.Settings.make(overlay_mode=1))
        view.load_surrogate(configs.saved_surrogate(case["field"]))
        return {"view": view, "out": _images(view, ("mapping", "lyapunov"))}
    if kind == "train":
        cfg = L.SurrogateConfig.make(case["field"], train_rays=case["rays"], batch=case["batch"], steps=case["steps"],
                                     h=case["h"], max_steps=int(20 / case["h"]), coarse_h=case["coarse_h"],
                                     seed=seed % (1 << 31))
        return {"view": L.MainView(64, 64), "cfg": cfg}
    if kind == "flowmap":
        return {"states": entry_states(case["n"], seed), "field": case["field"],
                "integrator": _escape(case["h"], int(20 / case["h"]))}
    if kind == "infer":
        view = L.MainView(64, 64)
        view.load_surrogate(configs.saved_surrogate(case["field"]))
        return {"view": view, "states": entry_states(case["n"], seed)}
    if kind == "model":
        rng = np.random.default_rng(seed)
        view = L.MainView(case["width"], case["height"])
        view.update_camera(L.Camera.look_at(_eye(rng), (0.0, 0.0, 0.0), (0.0, 1.0, 0.0), fov_deg=60.0))
        view.update_settings(L.Settings.make(overlay_mode=0))
        view.set_integrator(L.Integrator.make(h_initial=0.01, adaptive=False, samples_per_ray=0, sample_steps=0))
        view.set_field("swirl")
        return {"view": view, "mesh": _ico_scene(case["level"], seed), "out": _images(view, ("final", "mapping", "hit"))}
    raise ValueError(kind)


# ---------------------------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------------------------
def _weights(blob):
    """The five layers' weights and biases of a saved surrogate (the tail of the blob)."""
    shapes = [s for k in (224, 256, 256, 256) for s in ((k, 256), (256,))] + [(256, 7), (7,)]
    flat = np.frombuffer(blob, F32, offset=len(blob) - 4 * sum(int(np.prod(s)) for s in shapes))
    out = []
    for s in shapes:
        n = int(np.prod(s))
        out.append(flat[:n].reshape(s))
        flat = flat[n:]
    return out


def run(state):
    view = state.get("view")
    if "render" in state:
        state["render"]()
        return state["out"]
    if "views" in state:
        view.render_batch()
        frames = [view.read_batch_view(i) for i in range(state["views"])]
        return {"rgba": np.concatenate([f.final.reshape(-1) for f in frames]),
                "mapping": np.concatenate([f.mapping.reshape(-1) for f in frames]),
                "hit": np.concatenate([f.hit_faces.reshape(-1) for f in frames]),
                "steps": np.concatenate([f.steps.reshape(-1) for f in frames])}
    if "cfg" in state:
        stats = view.train_surrogate(state["cfg"])
        keep = ("train_loss", "holdout_err_q50", "holdout_err_q99", "holdout_frac_within_tol")
        return {"stats": np.array([stats[k] for k in keep], F32), "weights": _weights(view.save_surrogate())}
    if "integrator" in state:
        exits, steps = L.flowmap(state["field"], state["integrator"], state["states"])
        return {"exits": exits, "steps": steps}
    if "states" in state:
        return view.surrogate_infer(state["states"])
    if "mesh" in state:
        view.update_model(*state["mesh"])
        view.render()
        return state["out"]
    view.render_surrogate()
    return state["out"]


# ---------------------------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------------------------
def _steps_of(h, t_max=5.0):
    """Iterations of `for (; t <= t_max; t += h)` with t and h in FP32."""
    t, n, h = F32(0.0), 0, F32(h)
    while t <= F32(t_max):
        t = F32(t + h)
        n += 1
    return n


def _step_flop(field):
    return 56 + FIELD_FLOP.get(field, 217 if field.startswith("mirage") else 40)


def work(case):
    kind = case["kind"]
    if kind == "frame":
        px, n = case["width"] * case["height"], _steps_of(0.001 if case["high"] else case["h"])
        faces = 36 + (20 * 4 ** case["level"] if case["scene"] == "ico" else 0)
        serial = 8 * 5000 if case["samples"] else 0
        return {"bytes": 40 * px + 48 * faces, "flops": (px * n + serial) * _step_flop(case["field"])}
    if kind == "batch":
        # a ray's way: about a unit to the sphere and on average two thirds of its diameter through it
        views = _batch_views(case, 0)
        names = {v: k for k, v in L.FIELDS.items()}
        px = sum(v.width * v.height for v in views)
        return {"bytes": 28 * px, "flops": sum(v.width * v.height * (3.0 / v.h_initial) * _step_flop(names[v.field]) for v in views)}
    if kind == "surrogate":
        # the approach (about a unit at h = 0.005), the network for about four rays of five
        px = case["width"] * case["height"]
        return {"bytes": 24 * px, "flops": px * (200 * _step_flop(case["field"]) + 0.8 * MLP_FLOP)}
    if kind == "train":
        labels = case["rays"] * (2.7 / case["h"]) * _step_flop(case["field"])
        return {"bytes": 48 * case["rays"], "flops": labels + 3 * MLP_FLOP * case["batch"] * case["steps"]}
    if kind == "flowmap":
        return {"bytes": 52 * case["n"], "flops": case["n"] * (2.7 / case["h"]) * _step_flop(case["field"])}
    if kind == "infer":
        return {"bytes": 52 * case["n"], "flops": MLP_FLOP * case["n"]}
    faces, px = 36 + 20 * 4 ** case["level"], case["width"] * case["height"]
    cells = (128 if faces <= 65536 else 256) ** 3
    return {"bytes": 66 * faces + 5 * cells + 24 * px, "flops": px * _steps_of(0.01) * _step_flop("swirl")}


# ---------------------------------------------------------------------------------------------
# The same results in 64 bits (plain torch)
# ---------------------------------------------------------------------------------------------
def _dot(a, b):
    return (a * b).sum(-1, keepdim=True)


def _unit(a):
    return a / _dot(a, a).sqrt()


def _refract(t_in, t_out, v, n):
    def index(t):
        return 0.0000104 * 101325.0 * (1.0 + 101325.0 * (60.1 - 0.972 * t) * 1e-10) / (1.0 + 0.00366 * t)
    cosi = _dot(v, n).clamp(max=1.0)
    n = torch.where(cosi < 0, n, -n)
    cosi = cosi.abs()
    eta = index(t_in) / index(t_out)
    k = 1.0 - eta * eta * (1.0 - cosi * cosi)
    return torch.where(k < 0, v - 2.0 * _dot(n, v) * n, eta * v + (eta * cosi - k.clamp(min=0).sqrt()) * n)


def _field64(name):
    def swirl(pp, p, v0, v, t):
        a = 0.5 * _dot(p, p).sqrt()
        s, c = a.sin(), a.cos()
        x, y, z = v0[..., 0:1], v0[..., 1:2], v0[..., 2:3]
        return torch.cat((c * x + s * z, y.expand_as(s), c * z - s * x), -1)

    def warp(pp, p, v0, v, t):
        y = 4.0 * p
        return v0 + 0.3 * torch.cat((y[..., 1:2].sin(), torch.zeros_like(y[..., :1]), y[..., 0:1].sin()), -1)

    def hot_air(pp, p, v0, v, t):
        c = torch.tensor([0.0, -0.5, 0.0], dtype=p.dtype, device=p.device)

        def temp(q):
            d = q - c
            return 20.0 + 80.0 * torch.sigmoid(8.0 * (0.5 - _dot(d, d).sqrt()))
        return _refract(temp(pp), temp(p), v, _unit(p - c))

    def rotation(pp, p, v0, v, t):
        s, c = math.sin(math.pi * t), math.cos(math.pi * t)
        x, y = v0[..., 0:1], v0[..., 1:2]
        return _unit(v0 + torch.cat((c * x - s * y, s * x + c * y, torch.zeros_like(x)), -1))

    def mirage(pp, p, v0, v, t):
        spherical, sig = "spherical" in name, "sigmoid" in name
        src, far = (200.0, 0.25) if spherical else (30.0, 0.01)
        c = torch.tensor([-0.5, 0.5, -0.5], dtype=p.dtype, device=p.device)

        def temp(q):
            d = _dot(q - c, q - c).sqrt() if spherical else (q[..., 1:2] - 0.1).abs()
            x = d / far
            part = (torch.sigmoid(x * 12.0 - 6.0) if sig else x).clamp(max=1.0)
            return part * 15.0 + (1.0 - part) * src
        n = _unit(p - c) if spherical else torch.tensor([0.0, 1.0, 0.0], dtype=p.dtype, device=p.device).expand_as(p)
        return _refract(temp(pp), temp(p), v, n)

    return mirage if name.startswith("mirage") else {"swirl": swirl, "warp": warp, "hot_air": hot_air, "rotation": rotation}[name]


def _step64(f, p, d, v0, t, h, w=1.0):
    k1 = f(p, p, v0, d, t)
    k2 = f(p, p + 0.5 * h * k1, v0, k1, t + 0.5 * h)
    k3 = f(p, p + 0.5 * h * k2, v0, k2, t + 0.5 * h)
    k4 = f(p, p + h * k3, v0, k3, t + h)
    return (1.0 - w) * d + w * (k1 + 2.0 * k2 + 2.0 * k3 + k4) / 6.0


def _rays64(cam, w, h, u, v, device):
    """Camera rays through the normalised positions (u, v) of a w x h image."""
    def vec(a):
        return torch.tensor([a[0], a[1], a[2]], dtype=torch.float64, device=device)
    vd, up = vec(cam.view_direction), vec(cam.up)
    fov = cam.view_direction[3]
    vh = float(F32(2.0 * 0.035 * math.tan(fov * math.pi / 360.0))) if fov > 0 else 0.025
    vw = w / h * vh
    hor = torch.linalg.cross(up, -vd)
    ver = torch.linalg.cross(-vd, hor)
    d = (u * vw - 0.5 * vw)[..., None] * _unit(hor) + (v * vh - 0.5 * vh)[..., None] * _unit(ver) + 0.035 * vd
    return vec(cam.origin).expand_as(d), _unit(d)


def _pixels64(cam, w, h):
    gx = torch.arange(w, dtype=torch.float64, device="cuda") / (w - 1.0)
    gy = torch.arange(h, dtype=torch.float64, device="cuda").flip(0) / (h - 1.0)  # texel row 0 is the top
    return _rays64(cam, w, h, gx[None, :].expand(h, w), gy[:, None].expand(h, w), "cuda")


def _lyapunov64(p):
    """The overlay's exponent (central differences of the end points, delta 1); -1 at the border."""
    gx, gy = 0.5 * (p[1:-1, 2:] - p[1:-1, :-2]), 0.5 * (p[2:, 1:-1] - p[:-2, 1:-1])
    a, b, c = _dot(gx, gx), _dot(gx, gy), _dot(gy, gy)
    tr, det = a + c, a * c - b * b
    lam = (0.5 * (tr + (tr * tr - 4.0 * det).clamp(min=0).sqrt())).sqrt()[..., 0]
    out = torch.full(p.shape[:2], -1.0, dtype=p.dtype, device=p.device)
    out[2:-2, 2:-2] = lam[1:-1, 1:-1]
    return out


def _samples64(case, cam, settings, f):
    """The 8 sample rays around the mouse: 100 records of 5000 steps at h = 0.001 (on the CPU)."""
    ox = torch.tensor([-1, 0, 1, 1, 1, 0, -1, -1], dtype=torch.float64)
    oy = torch.tensor([-1, -1, -1, 0, 1, 1, 1, 0], dtype=torch.float64)
    rgb = torch.tensor([[1, 0, 0], [.5, .5, 0], [0, 1, 0], [.5, 1, 0], [1, 1, 0], [.5, .5, .5], [0, 0, 1], [.5, 0, .5]],
                       dtype=torch.float64)
    p, d = _rays64(cam, case["width"], case["height"], settings.mouse_pos[0] + 0.01 * ox,
                   settings.mouse_pos[1] + 0.01 * oy, "cpu")
    v0, h = d, float(F32(0.001))
    out = torch.empty(8, 100, 2, 4, dtype=torch.float64)
    out[:, :, 0, 3], out[:, :, 1, :3], out[:, :, 1, 3] = 1.0, rgb[:, None, :], 0.5
    for i in range(5000):
        if i % 50 == 0:
            out[:, i // 50, 0, :3] = p
        d = _step64(f, p, d, v0, i * h, h, case["weight"])
        p = p + h * d
    return out


def _escape64(f, p, v0, h, max_steps, r=2.0):
    """Escape-mode flow map, exits clipped to the sphere: end points and final directions."""
    shape, p, v0 = p.shape, p.reshape(-1, 3).clone(), v0.reshape(-1, 3)
    end, out_d = p.clone(), v0.clone()
    at = torch.arange(len(p), device=p.device)
    d, v, t = v0.clone(), v0, 0.0
    for i in range(max_steps):
        d = _step64(f, p, d, v, t, h)
        q, t = p + h * d, t + h
        left = ((_dot(q, q) > r * r) & (_dot(q, d) > 0))[:, 0]
        if bool(left.any()):
            a, b, c = _dot(h * d, h * d), _dot(p, h * d), _dot(p, p) - r * r
            u = ((-b + (b * b - a * c).clamp(min=0).sqrt()) / a).clamp(0, 1)
            x = torch.where(c <= 0, p + u * h * d, q)
            end[at[left]], out_d[at[left]] = x[left], d[left]
            keep = ~left
            at, q, d, v = at[keep], q[keep], d[keep], v[keep]
            if not len(at):
                break
        p = q
    if len(at):
        end[at], out_d[at] = p, d
    return end.reshape(shape), out_d.reshape(shape)


def exact(case, seed):
    kind = case["kind"]
    if kind == "frame":
        # adaptive steps are decided at rounding level and rays that the lens captures by the last
        # bit; the images, hit faces and step counts are whole numbers
        if case["adaptive"] or case["field"] == "lens":
            return None
        _, _, cam = _scene(case, seed)
        f, n, h = _field64(case["field"]), _steps_of(case["h"]), float(F32(case["h"]))
        p, d = _pixels64(cam, case["width"], case["height"])
        v0 = d
        for i in range(n):
            d = _step64(f, p, d, v0, i * h, h, case["weight"])
            p = p + h * d
        out = {"final": None, "hit": None, "steps": None,
               "mapping": torch.cat((p, torch.ones_like(p[..., :1])), -1),
               "lyapunov": _lyapunov64(p) if case["overlay"] else torch.full(p.shape[:2], -1.0, dtype=p.dtype)}
        if case["samples"]:
            out["samples"] = _samples64(case, cam, _settings(case, seed), f)
        return out
    if kind == "surrogate":
        # the RK4 frame that the surrogate stands for
        if case["field"] == "lens":
            return None
        p, d = _pixels64(_surrogate_view(case, seed), case["width"], case["height"])
        p, _ = _escape64(_field64(case["field"]), p, d, float(F32(0.005)), 4000)
        return {"mapping": torch.cat((p, torch.ones_like(p[..., :1])), -1), "lyapunov": None}
    if kind == "flowmap":
        if case["field"] == "lens":
            return None
        s = torch.from_numpy(entry_states(case["n"], seed)).double().cuda()
        p, d = _escape64(_field64(case["field"]), s[:, :3], s[:, 3:], float(F32(case["h"])), int(20 / case["h"]))
        return {"exits": torch.cat((p, d), -1), "steps": None}
    if kind == "infer":
        blob = configs.saved_surrogate(case["field"]).read_bytes()
        w = [torch.from_numpy(x.copy()).double().cuda() for x in _weights(blob)]
        # the header: magic 8, two words, the layers' sizes, the 16 Fourier frequencies
        freqs = torch.tensor(struct.unpack_from("<16f", blob, 56), dtype=torch.float64, device="cuda")
        s = torch.from_numpy(entry_states(case["n"], seed)).double().cuda()
        x = torch.cat((s[:, :3] / 2.0, s[:, 3:]), -1)
        out = []
        for part in x.split(1 << 17):
            a = freqs[None, :, None] * part[:, None, :]
            z = torch.cat((part, torch.stack((a.sin(), a.cos()), -1).reshape(len(part), -1)), -1)
            z = torch.nn.functional.pad(z, (0, 224 - z.shape[1]))
            for l in range(4):
                z = torch.nn.functional.silu(z @ w[2 * l] + w[2 * l + 1])
            out.append(z @ w[8] + w[9])
        return torch.cat(out)
    if kind == "model":
        f, h = _field64("swirl"), float(F32(0.01))
        rng = np.random.default_rng(seed)
        cam = L.Camera.look_at(_eye(rng), (0.0, 0.0, 0.0), (0.0, 1.0, 0.0), fov_deg=60.0)
        p, d = _pixels64(cam, case["width"], case["height"])
        v0 = d
        for i in range(_steps_of(0.01)):
            d = _step64(f, p, d, v0, i * h, h)
            p = p + h * d
        return {"final": None, "hit": None, "mapping": torch.cat((p, torch.ones_like(p[..., :1])), -1)}
    # a batch's rays end on the mesh (faces tested at every step: too long here); training's
    # weights after many Adam steps follow the rounding of the first
    return None
