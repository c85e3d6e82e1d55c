"""The calls whose speed is tracked, over the sizes that renders really use.

The framework is used in three ways: its renderers (plain path tracing, HairMSNN, neural radiance caching, each
a whole image from a scene description), the appearance optimisation (a differentiable render with its backward
pass), and the batched device entry points that other renderers call (hair BSDF streams, ray queries, the
radiance-cache network). Every case is one such call with the inputs already in hand.
"""
from __future__ import annotations

import copy
import ctypes as C
import math
import os
import struct
import tempfile

import numpy as np
import torch

import hairmsnn_amd as hm
from hairmsnn_amd import diff
from hairmsnn_amd._lib import HairParams, check, load

DEV = "cuda"
WEIGHTS = 5 * 64 * 64 + 3 * 64
ALPHA = float(np.float32(np.float32(3.14159) * np.float32(2.0)) / np.float32(180.0))  # two degrees of scale tilt
PRECISIONS = {"fp16": 0, "bf16": 1, "fp8": 2}


# ---- cases -------------------------------------------------------------------

def listed() -> list[dict]:
    return [
        # a renderer shading one small tile through the BSDF stream: latency of a call
        {"name": "bsdf_eval_1k", "op": "bsdf_eval", "n": 1021, "beta_m": 0.3, "beta_n": 0.3},
        # importance sampling for a wavefront of four million hair hits (a 2K frame's paths)
        {"name": "bsdf_sample_4m", "op": "bsdf_sample", "n": 4_000_037, "beta_m": 0.3, "beta_n": 0.3},
        # the radiance cache queried at every pixel of a 1024 x 1024 frame
        {"name": "mlp_infer_fp16_1m", "op": "mlp_infer", "precision": "fp16", "n": 1 << 20},
        # the eight-bit cache queried for a half-size frame of ragged size
        {"name": "mlp_infer_fp8_300k", "op": "mlp_infer", "precision": "fp8", "n": 300_001},
        # weight gradient of one training batch of the radiance cache, the default 65,536 records
        {"name": "mlp_grad_fp16_64k", "op": "mlp_grad", "precision": "fp16", "n": 65_536, "loss": 0},
        # a million closest-hit queries of another program against a mid-size groom
        {"name": "rays_closest_1m", "op": "rays", "n": 1_000_003, "strands": 20_000, "segments": 32, "any_hit": False},
        # the small hair ball at its own 256 x 256 x 16 spp: a preview render
        {"name": "pt_ball_256", "op": "pt", "scene": "ball", "strands": 2000, "segments": 16, "width": 256,
         "height": 256, "spp": 16},
        # the headline scene: 3.2 million segments at 1024 x 1024
        {"name": "pt_curly_1024", "op": "pt", "scene": "curly", "strands": 50_000, "segments": 64, "width": 1024,
         "height": 1024, "spp": 16},
        # a groom read from a .hair file, traced as round cubic curves, odd height
        {"name": "pt_curves_640", "op": "pt", "scene": "curves", "strands": 10_000, "segments": 24, "width": 640,
         "height": 363, "spp": 8},
        # the whole HairMSNN render of the headline scene: warm-up training, then frames
        {"name": "msnn_curly_1024", "op": "msnn", "scene": "curly", "strands": 50_000, "segments": 64, "width": 1024,
         "height": 1024, "spp": 16, "BETA": 1, "records": 65_536, "warmup": 64},
        # the neural-radiance-caching renderer on a mid-size frame
        {"name": "nrc_curly_512", "op": "nrc", "scene": "curly", "strands": 20_000, "segments": 64, "width": 512,
         "height": 512, "spp": 8, "records": 65_536},
        # one step of appearance optimisation: image, per-strand absorption and roughness gradients
        {"name": "adjoint_curly_512", "op": "adjoint", "scene": "curly", "strands": 50_000, "segments": 64,
         "width": 512, "height": 512, "spp": 16},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _frame(rng, lo: int, hi: int) -> dict:
    # scene files need width x height to be a multiple of 128; heights are odd or even as they come
    return {"width": 128 * rng.randint(max(1, lo // 128), hi // 128), "height": rng.randint(lo, hi)}


def draw(rng) -> dict:
    op = rng.choice(["bsdf_eval", "bsdf_sample", "mlp_infer", "mlp_grad", "rays", "pt", "pt", "msnn", "nrc", "adjoint"])
    if op in ("bsdf_eval", "bsdf_sample"):
        return {"op": op, "n": _log_int(rng, 200, 4_000_000), "beta_m": round(rng.uniform(0.12, 0.6), 3),
                "beta_n": round(rng.uniform(0.12, 0.6), 3)}
    if op == "mlp_infer":
        return {"op": op, "precision": rng.choice(["fp16", "bf16", "fp8"]), "n": _log_int(rng, 500, 1 << 20)}
    if op == "mlp_grad":
        return {"op": op, "precision": rng.choice(["fp16", "bf16"]), "n": _log_int(rng, 130, 65_536), "loss": 0}
    if op == "rays":
        return {"op": op, "n": _log_int(rng, 1000, 1_000_000), "strands": _log_int(rng, 100, 20_000),
                "segments": rng.randint(5, 40), "any_hit": rng.random() < 0.5}
    scene = rng.choice(["ball", "curly", "curves"]) if op == "pt" else "curly"
    strands = _log_int(rng, 200, 10_000 if scene != "curly" else 50_000)
    segments = rng.randint(8, 24 if scene != "curly" else 64)
    case = {"op": op, "scene": scene, "strands": strands, "segments": segments, "spp": rng.randint(2, 16)}
    if op == "pt":
        return {**case, **_frame(rng, 128, 640 if scene == "curves" else 1024)}
    if op == "msnn":
        return {**case, **_frame(rng, 256, 1024), "BETA": rng.choice([1, 2, 5]), "records": 128 * rng.randint(16, 512),
                "warmup": rng.randint(8, 64)}
    if op == "nrc":
        return {**case, **_frame(rng, 128, 512), "spp": rng.randint(2, 8), "records": 128 * rng.randint(16, 512)}
    return {**case, **_frame(rng, 128, 512)}


# ---- inputs ------------------------------------------------------------------

def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(seed)


def _sphere(n: int, g: torch.Generator) -> torch.Tensor:
    v = torch.randn(n, 3, generator=g, device=DEV, dtype=torch.float64)
    return v / v.norm(dim=1, keepdim=True).clamp_min(1e-12)


def _uniform(shape, lo: float, hi: float, g: torch.Generator) -> torch.Tensor:
    return torch.rand(shape, generator=g, device=DEV, dtype=torch.float64) * (hi - lo) + lo


def _bsdf_inputs(case: dict, seed: int):
    """Queries as a renderer makes them in the hair frame: wo.y = 0, wi anywhere, |h| < 1; and four uniforms each."""
    n, g = case["n"], _gen(seed)
    so = _uniform((n,), -0.995, 0.995, g)
    wo = torch.stack([so, torch.zeros_like(so), (1 - so * so).sqrt()], 1)
    q = torch.cat([wo, _sphere(n, g), _uniform((n, 1), -0.999, 0.999, g), _uniform((n, 3), 0.01, 1.0, g)], 1)
    return q.float().contiguous(), torch.rand(n, 4, generator=g, device=DEV)


def _hair_params(case: dict) -> HairParams:
    p = HairParams()
    p.beta_m, p.beta_n, p.alpha = case["beta_m"], case["beta_n"], ALPHA
    for i in range(4):
        p.gain[i] = 1.0
    return p


def _mlp_inputs(case: dict, seed: int):
    """Hit records (position over scene scale, view direction, tangent, absorption), targets and network weights."""
    n, g = case["n"], _gen(seed)
    rec = torch.cat([_uniform((n, 3), -0.5, 0.5, g), _sphere(n, g), _sphere(n, g), _uniform((n, 3), 0.01, 0.5, g)], 1)
    target = _uniform((n, 3), 0.1, 2.0, g).float().contiguous()
    hidden = _uniform((5 * 4096,), -1.0, 1.0, g) * math.sqrt(6.0 / 128.0)
    out = _uniform((3 * 64,), -1.0, 1.0, g) * math.sqrt(6.0 / 67.0)
    return rec.float().contiguous(), target, torch.cat([hidden, out]).float()


def _strands(case: dict, seed: int) -> np.ndarray:
    """Helical strands rooted on the unit sphere, strands x (segments + 1) x 3."""
    rng = np.random.default_rng(seed)
    n, s = case["strands"], case["segments"]
    nrm = rng.normal(size=(n, 3))
    nrm /= np.linalg.norm(nrm, axis=1, keepdims=True)
    e1 = np.cross(nrm, np.where(np.abs(nrm[:, :1]) < 0.9, [[1.0, 0.0, 0.0]], [[0.0, 1.0, 0.0]]))
    e1 /= np.linalg.norm(e1, axis=1, keepdims=True)
    e2 = np.cross(nrm, e1)
    k = np.arange(s + 1)[None, :, None]
    phase = rng.uniform(0, 2 * np.pi, (n, 1, 1))
    ang = phase + 2 * np.pi * k / 12
    rise = 0.45 * k / s
    p = (nrm[:, None] * (1 + rise) + 0.03 * ((np.cos(ang) - np.cos(phase)) * e1[:, None]
                                            + (np.sin(ang) - np.sin(phase)) * e2[:, None]))
    return p.astype(np.float32)


def _write_hair(path: str, pts: np.ndarray, thickness: float) -> None:
    """A .hair file with a fixed number of segments per strand (header, then the point array)."""
    n, m, _ = pts.shape
    head = b"HAIR" + struct.pack("<IIIIff3f", n, n * m, 2, m - 1, thickness, 0.0, 1.0, 1.0, 1.0)
    with open(path, "wb") as f:
        f.write(head + b"\0" * (128 - len(head)))
        f.write(np.ascontiguousarray(pts, np.float32).tobytes())


def _scene(case: dict, seed: int) -> hm.Scene:
    """The scene description a user's file would hold, with this seed's strands and environment."""
    kind = case["scene"]
    hair = {"type": 1, "alpha": 2.0, "beta_m": 0.3, "beta_n": 0.3, "sigma_a": [0.06, 0.1, 0.2]}
    cfg = {
        "camera": {"from": [0.0, -4.5, 0.0], "to": [0.0, 0.0, 0.0], "up": [0.0, 0.0, 1.0], "cos_fovy": 0.66},
        "hair": hair,
        "integrator": {"ENV_PDF": True, "MIS": True, "width": case["width"], "height": case["height"],
                       "spp": case["spp"], "path_v1": 1, "path_v2": 40, "image_output": "out.exr",
                       "stats_output": "out.json"},
        "lights": {"directional": [{"from": [3, 3, 3], "emit": [1, 1, 1]}]},
    }
    if kind == "ball":
        hair["procedural"] = {"kind": "ball", "strands": case["strands"], "segments": case["segments"],
                              "segment_length": 0.05, "radius": 0.005, "curl_sigma": 0.05, "root_sphere_radius": 1.0,
                              "seed": seed}
        cfg["camera"]["from"] = [0.0, -6.0, 0.0]
        cfg["lights"]["environment"] = {"constant": [0.5, 0.5, 0.5], "resolution": [64, 32], "scale": 1.0}
    else:
        hair["procedural"] = {"kind": "curly", "strands": case["strands"], "segments": case["segments"],
                              "helix_radius": 0.02, "helix_pitch": 0.1, "segments_per_turn": 16, "radius": 0.005,
                              "root_sphere_radius": 1.0, "seed": seed}
        cfg["surface"] = {"sphere": {"center": [0.0, 0.0, 0.0], "radius": 1.0, "albedo": [0.0, 0.0, 0.0],
                                     "alpha": 1.0}}
        cfg["lights"]["environment"] = {
            "procedural": {"width": 1024, "height": 512, "mu": 0.0, "sigma": 1.5, "seed": seed,
                           "hotspots": [{"theta": 0.6, "phi": 0.8, "width": 0.05, "color": [200.0, 180.0, 160.0]},
                                        {"theta": 1.2, "phi": 2.5, "width": 0.08, "color": [60.0, 80.0, 100.0]},
                                        {"theta": 0.9, "phi": 4.4, "width": 0.12, "color": [30.0, 30.0, 30.0]}]},
            "scale": 1.0}
    if "records" in case:
        cfg["tcnn"] = {"config": "tcnn.json", "init_train": True}
        cfg["hairmsnn"] = {"train_records": case["records"], "warmup_steps": case.get("warmup", 0),
                           "learning_rate": 0.01, "loss": "RelativeL2Luminance", "precision": "fp16",
                           "seed": seed % 1000 + 1}
        cfg["nrc"] = {"train_records": case["records"]}
    if kind != "curves":
        return hm.Scene(json_text=cfg)
    with tempfile.TemporaryDirectory() as d:
        path = os.path.join(d, "groom.hair")
        _write_hair(path, _strands(case, seed), 0.025)
        del hair["procedural"]
        hair["geometry"] = path
        return hm.Scene(json_text=cfg)


def _ray_inputs(case: dict, seed: int, pts: np.ndarray) -> torch.Tensor:
    """A third camera-like rays from outside, the rest secondary rays from next to the hair, as n x 8 floats."""
    n, g = case["n"], _gen(seed)
    k = n // 3
    o = _sphere(k, g) * 4.0
    d = _sphere(k, g) * _uniform((k, 1), 0.0, 1.45, g) - o
    p = torch.from_numpy(pts.reshape(-1, 3)).to(DEV).double()
    at = torch.randint(0, p.shape[0], (n - k,), generator=g, device=DEV)
    o = torch.cat([o, p[at] + _sphere(n - k, g) * 0.012])
    d = torch.cat([d / d.norm(dim=1, keepdim=True), _sphere(n - k, g)])
    rays = torch.zeros(n, 8, device=DEV)
    rays[:, 0:3], rays[:, 4:7] = o.float(), d.float()
    return rays


RAY_RADIUS = np.float32(0.2) * np.float32(0.025)  # the radius of a strand of that thickness


def _ray_scene(pts: np.ndarray) -> hm.Scene:
    with tempfile.TemporaryDirectory() as d:
        path = os.path.join(d, "groom.hair")
        _write_hair(path, pts, 0.025)
        return hm.Scene(json_text={
            "camera": {"from": [0.0, -4.5, 0.0], "to": [0.0, 0.0, 0.0], "up": [0.0, 0.0, 1.0], "cos_fovy": 0.66},
            "hair": {"geometry": path, "primitive": "linear", "tessellation": 1},
            "integrator": {"ENV_PDF": False, "MIS": False, "width": 128, "height": 128, "spp": 1, "path_v1": 1,
                           "path_v2": 1, "image_output": "out.exr", "stats_output": "out.json"},
            "lights": {"directional": [{"from": [3, 3, 3], "emit": [1, 1, 1]}]}})


class _Mlp:
    """A network handle, destroyed with the state that holds it."""

    def __init__(self, precision: str, weights: torch.Tensor):
        self.lib = load()
        self.h = C.c_void_p()
        check(self.lib.hmsnn_mlp_create(PRECISIONS[precision], 1, C.byref(self.h)))
        w = weights.cpu().numpy()
        check(self.lib.hmsnn_mlp_set_weights(self.h, C.c_void_p(w.ctypes.data), w.size))

    def __del__(self):
        if self.h:
            self.lib.hmsnn_mlp_destroy(self.h)
            self.h = None


def _p(t: torch.Tensor) -> C.c_void_p:
    return C.c_void_p(t.data_ptr())


def prepare(case: dict, seed: int) -> dict:
    case = copy.copy(case)
    op, s = case["op"], {"case": case, "lib": load()}
    if op in ("bsdf_eval", "bsdf_sample"):
        n = case["n"]
        s["params"] = _hair_params(case)
        s["q"], s["u"] = _bsdf_inputs(case, seed)
        s["f"], s["pdf"] = torch.empty(n, 3, device=DEV), torch.empty(n, device=DEV)
        if op == "bsdf_sample":
            s["wi"], s["lobe"] = torch.empty(n, 3, device=DEV), torch.empty(n, device=DEV, dtype=torch.int32)
    elif op in ("mlp_infer", "mlp_grad"):
        s["rec"], s["target"], w = _mlp_inputs(case, seed)
        s["mlp"] = _Mlp(case["precision"], w)
        s["out"] = torch.empty(case["n"], 3, device=DEV) if op == "mlp_infer" else torch.empty(WEIGHTS, device=DEV)
    elif op == "rays":
        pts = _strands(case, seed)
        s["scene"] = _ray_scene(pts)
        s["rays"] = _ray_inputs(case, seed, pts)
        n = case["n"]
        s["prim"] = torch.empty(n, device=DEV, dtype=torch.int32)
        s["t"], s["u"] = torch.empty(n, device=DEV), torch.empty(n, device=DEV)
    else:
        s["scene"] = _scene(case, seed)
        if op == "adjoint":
            rng = np.random.default_rng(seed)
            s["sigma"] = torch.from_numpy(rng.uniform(0.05, 0.3, (case["strands"], 3)).astype(np.float32))
            s["grad"] = torch.from_numpy(rng.normal(size=(case["height"], case["width"], 3)).astype(np.float32))
    torch.cuda.synchronize()
    return s


# ---- one pass ------------------------------------------------------------------

def run(s: dict):
    case, lib = s["case"], s["lib"]
    op = case["op"]
    if op == "bsdf_eval":
        check(lib.hmsnn_hair_bsdf_eval_dev(C.byref(s["params"]), _p(s["q"]), case["n"], _p(s["f"]), _p(s["pdf"]), None))
        return {"f": s["f"], "pdf": s["pdf"]}
    if op == "bsdf_sample":
        check(lib.hmsnn_hair_bsdf_sample_dev(C.byref(s["params"]), _p(s["q"]), _p(s["u"]), case["n"], _p(s["wi"]),
                                             _p(s["f"]), _p(s["pdf"]), _p(s["lobe"]), None))
        return {"wi": s["wi"], "f": s["f"], "pdf": s["pdf"], "lobe": s["lobe"]}
    if op == "mlp_infer":
        check(lib.hmsnn_mlp_forward_dev(s["mlp"].h, _p(s["rec"]), case["n"], _p(s["out"]), None))
        return s["out"]
    if op == "mlp_grad":
        check(lib.hmsnn_mlp_backward_dev(s["mlp"].h, _p(s["rec"]), _p(s["target"]), case["n"], case["loss"],
                                         _p(s["out"]), None, None))
        return s["out"]
    if op == "rays":
        any_hit = case["any_hit"]
        check(lib.hmsnn_trace_rays_dev(s["scene"].h, _p(s["rays"]), case["n"], int(any_hit), _p(s["prim"]),
                                       None if any_hit else _p(s["t"]), None if any_hit else _p(s["u"])))
        return {"prim": s["prim"]} if any_hit else {"prim": s["prim"], "t": s["t"], "u": s["u"]}
    if op == "pt":
        return s["scene"].render_path_tracing(case["spp"])
    if op == "msnn":
        return s["scene"].render_hair_msnn(case["BETA"], case["spp"])
    if op == "nrc":
        return s["scene"].render_nrc(case["spp"])
    sigma = s["sigma"].clone().requires_grad_(True)
    params = torch.tensor([0.3, 0.3, ALPHA], dtype=torch.float64, requires_grad=True)
    img = diff.render_hair(s["scene"], sigma, params, case["spp"])
    img.backward(s["grad"])
    return {"image": img.detach(), "sigma": sigma.grad, "params": params.grad}


# ---- what a pass cannot do without ----------------------------------------------

MLP_FLOPS = 2 * WEIGHTS
TREE_BOX_FLOPS, SEGMENT_FLOPS, VERTEX_FLOPS = 14, 80, 900


def _ray_flops(rays: float, prims: int) -> float:
    """A ray descends one four-wide tree of the primitives once and tests one of them."""
    levels = math.ceil(math.log(max(2, prims), 4))
    return rays * (levels * 4 * TREE_BOX_FLOPS + SEGMENT_FLOPS)


def work(case: dict) -> dict:
    op, n = case["op"], case.get("n", 0)
    if op == "bsdf_eval":
        return {"bytes": 56.0 * n, "flops": 250.0 * n}
    if op == "bsdf_sample":
        return {"bytes": 88.0 * n, "flops": 320.0 * n}
    if op == "mlp_infer":
        return {"bytes": 60.0 * n + 2 * WEIGHTS, "flops": float(MLP_FLOPS) * n}
    if op == "mlp_grad":
        return {"bytes": 60.0 * n + 6 * WEIGHTS, "flops": 3.0 * MLP_FLOPS * n}
    prims = case["strands"] * case["segments"]
    if op == "rays":
        return {"bytes": 32.0 * prims + (36.0 if case["any_hit"] else 44.0) * n, "flops": _ray_flops(n, prims)}
    px = case["width"] * case["height"]
    geometry = (80.0 if case["scene"] == "curves" else 32.0) * prims + 16.0 * 1024 * 512
    # about half the pixels see hair; a path that does has some eight vertices with one continuation and one or
    # two light rays each, a truncated one two
    paths = px * case["spp"]
    vertices = paths * 0.5 * (2.0 if op == "msnn" else 8.0)
    flops = _ray_flops(2.5 * vertices + paths, prims) + VERTEX_FLOPS * vertices
    nbytes = geometry + 16.0 * px
    if op in ("msnn", "nrc"):
        steps = case["spp"] + case.get("warmup", 0)
        flops += MLP_FLOPS * paths + 3.0 * MLP_FLOPS * case["records"] * steps
        flops += (_ray_flops(2.5 * 8, prims) + 8 * VERTEX_FLOPS) * case["records"] * steps if op == "msnn" else 0.0
    if op == "adjoint":
        flops *= 2.0
        nbytes += 16.0 * px + 24.0 * case["strands"]
    return {"bytes": nbytes, "flops": flops}


def tolerance(case: dict):
    """About four times the distance from the 64-bit result, or from the same call with its sums in another order."""
    op = case["op"]
    if op == "bsdf_eval":
        return {"rel": 5e-6, "max": 2e-3}
    if op == "bsdf_sample":  # a draw beside a lobe's edge takes the other lobe
        return {"rel": 1.5e-3, "max": 0.9, "differ": 1e-5}
    if op == "mlp_infer":
        return {"rel": {"fp16": 4e-4, "bf16": 4e-3, "fp8": 3e-2}[case["precision"]], "max": 0.5}
    if op == "mlp_grad":
        return {"rel": {"fp16": 4e-3, "bf16": 3e-2}[case["precision"]], "max": 0.5}
    if op == "rays":
        return {"rel": 1e-6, "max": 1e-3, "differ": 1e-5}
    if op == "msnn":  # the trained cache's share of the image, after other sums in every training step
        return {"rel": 2.5e-3, "max": 0.1}
    if op == "nrc":  # cache values as the fp16 inference gives them
        return {"rel": 4e-4, "max": 0.1}
    return {"rel": 1e-5, "max": 1e-3}  # the same paths, their 32-bit sums in another order


# ---- the same in 64 bits ----------------------------------------------------------

PI = float(np.float32(3.1415926))


def _consts(case: dict) -> dict:
    bm, bn, alpha = (float(np.float32(x)) for x in (case["beta_m"], case["beta_n"], ALPHA))
    v0 = (0.726 * bm + 0.812 * bm * bm + 3.7 * bm ** 20) ** 2
    s = 0.626657069 * (0.265 * bn + 1.194 * bn * bn + 5.372 * bn ** 22)
    lo, hi = 1 / (1 + math.exp(PI / s)), 1 / (1 + math.exp(-PI / s))
    sk = [math.sin(alpha)]
    ck = [math.sqrt(max(0.0, 1 - sk[0] ** 2))]
    for i in range(2):
        sk, ck = sk + [2 * ck[i] * sk[i]], ck + [ck[i] ** 2 - sk[i] ** 2]
    return {"v": [v0, 0.25 * v0, 4 * v0, 4 * v0], "s": s, "lo": lo, "span": hi - lo,
            "tilt": [(-sk[1], ck[1]), (sk[0], ck[0]), (sk[2], ck[2]), (0.0, 1.0)], "f0": (0.55 / 2.55) ** 2}


def _root(x: torch.Tensor) -> torch.Tensor:
    return x.clamp_min(0.0).sqrt()


def _i0(x: torch.Tensor) -> torch.Tensor:
    out, term = torch.ones_like(x), torch.ones_like(x)
    for i in range(1, 10):
        term = term * (x * x) / (4.0 * i * i)
        out = out + term
    return out


def _longitudinal(v: float, ci, co, si, so):
    a, b = ci * co / v, si * so / v
    if v > 0.1:
        return torch.exp(-b) * _i0(a) / (math.sinh(1 / v) * 2 * v)
    big = a - b - 1 / v + 0.5 * (-math.log(2 * PI) - torch.log(a) + 1 / (8 * a))
    small = torch.log(_i0(a)) - b - 1 / v
    return torch.exp(torch.where(a > 12.0, big, small) + float(np.float32(0.6931)) + math.log(1 / (2 * v)))


def _hair_prepare(c: dict, q: torch.Tensor) -> dict:
    wo, h, sigma = q[:, 0:3], q[:, 6], q[:, 7:10]
    eta = float(np.float32(1.55))
    so = wo[:, 0]
    co = _root(1 - so * so)
    st = so / eta
    sin_gt = h * co / _root(eta * eta - so * so)
    trans = torch.exp(-sigma * (2 * _root(1 - sin_gt ** 2) / _root(1 - st * st))[:, None])
    fr = (c["f0"] + (1 - c["f0"]) * (1 - co * _root(1 - h * h)) ** 5)[:, None]
    ap = [fr.expand_as(trans), (1 - fr) ** 2 * trans, (1 - fr) ** 2 * fr * trans * trans]
    ap.append(ap[2] * fr * trans / (1 - fr * trans))
    mean = torch.stack([x.mean(1) for x in ap])
    return {"so": so, "co": co, "phi": torch.atan2(wo[:, 2], wo[:, 1]), "go": torch.asin(h),
            "gt": torch.asin(sin_gt.clamp(-1, 1)), "ap": ap, "prob": mean / mean.sum(0)}


def _centre(p: int, w: dict) -> torch.Tensor:
    return 2.0 * p * w["gt"] - 2.0 * w["go"] + p * PI


def _hair_eval(c: dict, w: dict, wi: torch.Tensor):
    si = wi[:, 0]
    ci = _root(1 - si * si)
    phi = torch.atan2(wi[:, 2], wi[:, 1]) - w["phi"]
    f, pdf = torch.zeros_like(wi), torch.zeros_like(si)
    for p in range(4):
        ts, tc = c["tilt"][p]
        m = _longitudinal(c["v"][p], ci, (w["co"] * tc - w["so"] * ts).abs(), si, w["so"] * tc + w["co"] * ts)
        if p < 3:
            d = phi - _centre(p, w)
            d = d - 2 * PI * torch.round(d / (2 * PI))
            e = torch.exp(-d.abs() / c["s"])
            m = m * e / (c["s"] * (1 + e) ** 2 * c["span"])
        else:
            m = m / (2 * PI)
        f = f + m[:, None] * w["ap"][p]
        pdf = pdf + m * w["prob"][p]
    return f, pdf


def _hair_sample(c: dict, w: dict, u: torch.Tensor):
    cum = w["prob"].cumsum(0)
    lobe = (u[:, 0] >= cum[:3]).sum(0)
    pick = lambda v: torch.tensor(v, device=u.device, dtype=u.dtype)[lobe]  # noqa: E731
    ts, tc = pick([t[0] for t in c["tilt"]]), pick([t[1] for t in c["tilt"]])
    so, co = w["so"] * tc + w["co"] * ts, w["co"] * tc - w["so"] * ts
    v = pick(c["v"][:3] + [c["s"]])  # the residual lobe is sampled with the logistic scale
    e = u[:, 1].clamp_min(float(np.float32(1e-5)))
    cos_t = 1 + v * torch.log(e + (1 - e) * torch.exp(-2 / v))
    si = -cos_t * so + _root(1 - cos_t ** 2) * torch.cos(2 * PI * u[:, 2]) * co
    x = (-c["s"] * torch.log(1 / (u[:, 3] * c["span"] + c["lo"]) - 1)).clamp(-PI, PI)
    centre = torch.stack([_centre(p, w) for p in range(3)] + [torch.zeros_like(x)]).gather(0, lobe[None])[0]
    phi = w["phi"] + torch.where(lobe < 3, centre + x, 2 * PI * u[:, 3])
    ci = _root(1 - si * si)
    wi = torch.stack([si, ci * torch.cos(phi), ci * torch.sin(phi)], 1)
    return wi / wi.norm(dim=1, keepdim=True), lobe


def _encode(rec: torch.Tensor) -> torch.Tensor:
    cols = []
    for k in range(3):
        for j in range(6):
            a = rec[:, k] * (math.pi * 2 ** j)
            cols += [torch.sin(a), torch.cos(a)]
    for k in (3, 6):
        cols += [torch.acos(rec[:, k + 2].clamp(-1, 1)) / math.pi,
                 torch.atan2(rec[:, k + 1], rec[:, k]) / (2 * math.pi) + 0.5]
    cols += [rec[:, 9], rec[:, 10], rec[:, 11], torch.ones_like(rec[:, 0])]
    return torch.cat([torch.stack(cols, 1), torch.zeros(rec.shape[0], 20, device=rec.device, dtype=rec.dtype)], 1)


def _network(rec: torch.Tensor, w: torch.Tensor):
    """Every layer's input and the three outputs."""
    h = [_encode(rec)]
    for k in range(5):
        h.append((h[-1] @ w[4096 * k:4096 * (k + 1)].view(64, 64).T).clamp_min(0.0))
    return h, torch.exp(h[-1] @ w[5 * 4096:].view(3, 64).T)


def _network_grad(rec, target, w):
    """Weight gradient of the mean luminance-relative squared error; the weight of an error and the floor of the
    exponential's slope (1e-2) are as the training step defines them."""
    h, y = _network(rec, w)
    lum = y @ torch.tensor([0.212671, 0.715160, 0.072169], device=y.device, dtype=y.dtype)
    dz = 2 * (y - target) / (lum * lum + 0.01)[:, None] * y.clamp_min(1e-2) / y.numel()
    grads = [(dz.T @ h[5]).reshape(-1)]
    d = dz @ w[5 * 4096:].view(3, 64)
    for k in range(4, -1, -1):
        d = d * (h[k + 1] > 0)
        grads.insert(0, (d.T @ h[k]).reshape(-1))
        d = d @ w[4096 * k:4096 * (k + 1)].view(64, 64)
    return torch.cat(grads)


def _segment_hits(o, d, p0, p1, r):
    """Nearest root of every ray with every open cylinder: t (inf on a miss) and u, rays x segments."""
    a = p1 - p0
    w = o[:, None] - p0
    aa, da, wa = (a * a).sum(-1), d @ a.T, (w * a).sum(-1)
    qa = (d * d).sum(-1)[:, None] * aa - da * da
    qb = (w * d[:, None]).sum(-1) * aa - da * wa
    qc = (w * w).sum(-1) * aa - wa * wa - r * r * aa
    disc = qb * qb - qa * qc
    best, at = torch.full_like(disc, math.inf), torch.zeros_like(disc)
    for sign in (-1.0, 1.0):
        t = (-qb + sign * _root(disc)) / qa
        u = (wa + t * da) / aa
        ok = (disc >= 0) & (qa > 0) & (t > 0) & (u >= 0) & (u <= 1) & (t < best)
        best, at = torch.where(ok, t, best), torch.where(ok, u, at)
    return best, at


def exact(case: dict, seed: int):
    op = case["op"]
    if op in ("bsdf_eval", "bsdf_sample"):
        q, u = _bsdf_inputs(case, seed)
        c, q = _consts(case), q.double()
        w = _hair_prepare(c, q)
        if op == "bsdf_eval":
            f, pdf = _hair_eval(c, w, q[:, 3:6])
            return {"f": f, "pdf": pdf}
        wi, lobe = _hair_sample(c, w, u.double())
        f, pdf = _hair_eval(c, w, wi)
        return {"wi": wi, "f": f, "pdf": pdf, "lobe": lobe}
    if op == "mlp_infer":
        rec, _, w = _mlp_inputs(case, seed)
        return _network(rec.double(), w.double())[1]
    if op == "mlp_grad":
        rec, target, w = _mlp_inputs(case, seed)
        return _network_grad(rec.double(), target.double(), w.double())
    if op == "rays":
        n, prims = case["n"], case["strands"] * case["segments"]
        if n * prims > 5e9:
            return None  # every ray against every segment would take minutes
        pts = _strands(case, seed)
        rays = _ray_inputs(case, seed, pts).double()
        seg = torch.from_numpy(pts).to(DEV).double()
        p0, p1 = seg[:, :-1].reshape(-1, 3), seg[:, 1:].reshape(-1, 3)
        t, u = torch.empty(n, device=DEV, dtype=torch.float64), torch.empty(n, device=DEV, dtype=torch.float64)
        prim = torch.empty(n, device=DEV, dtype=torch.int64)
        step = max(1, int(2e7 // prims))
        for b in range(0, n, step):
            bt, bu = _segment_hits(rays[b:b + step, 0:3], rays[b:b + step, 4:7], p0, p1, float(RAY_RADIUS))
            t[b:b + step], prim[b:b + step] = bt.min(1)
            u[b:b + step] = bu.gather(1, prim[b:b + step, None])[:, 0]
        miss = torch.isinf(t)
        if case["any_hit"]:
            return {"prim": (~miss).long()}
        prim[miss], u[miss] = -1, 0.0
        return {"prim": prim, "t": t, "u": u}
    return None  # a path's decisions turn on the last bit of 32-bit draws; no 64-bit render has the same paths
