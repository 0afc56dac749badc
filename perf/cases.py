"""Timed workloads of the compound-eye renderer, through its public C ABI.

Four scenes, all with fixed geometry:

  lab      100 x 100-vertex heightfield, 19,602 triangles, vertex colours
  natural  the reference's shipped outdoor scene: 24,200 textured triangles
  field    bee-scale heightfield and stems, 2,189,058 triangles
  large    heightfield, stems and rocks, 16,316,418 triangles

A program loads its scene, eye and sampler network once and then renders pose
after pose, so `prepare` loads those (once per process and scene) and makes the
poses and the random-stream seed from the seed; `run` is the call itself, with
what the caller reads back.

Work is counted per ray as what any tracer has to do for it: drawing and
turning the ray, one walk down a 4-wide tree of the scene's depth, two triangle
tests and the shading.
"""
from __future__ import annotations

import gzip
import importlib.util
import math
import pathlib
import sys
import tempfile
from ctypes import c_void_p

import numpy as np
import torch

ROOT = pathlib.Path(__file__).resolve().parents[1]


def _package():
    if "compound_ray_amd" not in sys.modules:
        pkg = ROOT / "compound-ray_amd"
        spec = importlib.util.spec_from_file_location("compound_ray_amd", pkg / "__init__.py",
                                                      submodule_search_locations=[str(pkg)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["compound_ray_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["compound_ray_amd"]


cra = _package()
from compound_ray_amd import eyerenderer as er  # noqa: E402
from compound_ray_amd import scenes  # noqa: E402

TRIANGLES = {"lab": 19602, "natural": 24200, "field": 2189058, "large": 16316418}
EXTENT = {"lab": 10.0, "field": 40.0, "large": 80.0}
MLP_WIDTHS = (16, 64, 64, 64, 1)


def listed():
    return [
        # The smallest call: one sample per ommatidium, a fast preview or the
        # inner loop of a closed-loop agent; launches and waiting dominate.
        {"name": "frame-1k-1spp", "kind": "frame", "scene": "lab", "omm": 1000, "spp": 1},
        # The reference's speed test at an ordinary and at its largest rate:
        # the 1,000-ommatidium equidistant eye over its own textured scene.
        {"name": "frame-1k-100spp", "kind": "frame", "scene": "natural", "omm": 1000, "spp": 100},
        {"name": "frame-1k-3200spp", "kind": "frame", "scene": "natural", "omm": 1000, "spp": 3200},
        # Both eyes of a bee, frame by frame, at the plain uniform rate.
        {"name": "frame-bee-128spp", "kind": "frame", "scene": "field", "omm": 5500, "spp": 128},
        # A regular camera's preview of the same scene, odd window size.
        {"name": "camera-panorama", "kind": "camera", "scene": "field", "camera": "panoramic", "width": 641,
         "height": 361},
        # A few poses of a small eye at a small odd rate: one step of several
        # agents, colours to host memory.
        {"name": "batch-small", "kind": "batch", "scene": "lab", "omm": 733, "spp": 15, "poses": 17, "to": "host"},
        # The bee's left eye at many poses, uniform at the rate of 1 % error,
        # colours to host memory (data sets of views along a route).
        {"name": "batch-bee-63spp", "kind": "batch", "scene": "field", "omm": 5500, "spp": 63, "poses": 203,
         "to": "host"},
        # Thousands of poses with uneven per-ommatidium rates, colours left on
        # the device for a consumer there: the largest call.
        {"name": "batch-uneven", "kind": "batch", "scene": "lab", "omm": 5000, "spp": 0, "poses": 4096,
         "to": "device"},
        # Learned adaptive sampling of the bee's eye along a route.
        {"name": "adaptive-bee", "kind": "adaptive", "scene": "field", "omm": 5500, "poses": 256},
        # Learned adaptive sampling of 256 different eyes merged into one list
        # (2,149,386 ommatidia) over the largest scene.
        {"name": "adaptive-large", "kind": "adaptive", "scene": "large", "omm": 0, "poses": 1},
        # Closest hits of free rays (line-of-sight and distance queries).
        {"name": "rays", "kind": "rays", "scene": "field", "rays": 300007},
        # One epoch of the sampler network's training (forward, backward, Adam).
        {"name": "sampler-train", "kind": "train", "rows": 100003, "batch": 4096},
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["frame"] * 5 + ["batch"] * 4 + ["camera", "adaptive", "rays", "train"])
    if kind == "frame":
        scene = rng.choice(["lab", "natural", "field"])
        omm = log_int(300, 8000)
        spp = log_int(1, 3200)
        most = 12_000_000 if scene == "field" else 40_000_000
        return {"kind": kind, "scene": scene, "omm": omm, "spp": max(1, min(spp, most // omm))}
    if kind == "batch":
        scene = rng.choice(["lab", "field"])
        omm = log_int(300, 8000)
        poses = log_int(2, 2048)
        most = 90_000_000 if scene == "field" else 400_000_000
        poses = max(1, min(poses, 6_000_000 // omm))
        spp = 0 if rng.random() < 0.35 else max(1, min(log_int(4, 256), most // (omm * poses)))
        if spp == 0:
            poses = max(1, min(poses, most // (omm * 100)))
        return {"kind": kind, "scene": scene, "omm": omm, "spp": spp, "poses": poses,
                "to": rng.choice(["host", "device"])}
    if kind == "camera":
        return {"kind": kind, "scene": rng.choice(["lab", "field"]),
                "camera": rng.choice(["perspective", "orthographic", "panoramic"]),
                "width": log_int(60, 1500), "height": log_int(40, 1000)}
    if kind == "adaptive":
        omm = log_int(700, 8000)
        return {"kind": kind, "scene": rng.choice(["lab", "field"]), "omm": omm,
                "poses": max(1, min(log_int(4, 400), 1_500_000 // omm))}
    if kind == "rays":
        return {"kind": kind, "scene": rng.choice(["lab", "field"]), "rays": log_int(500, 1_000_000)}
    return {"kind": kind, "rows": log_int(5000, 200_000), "batch": rng.choice([512, 1000, 4096, 8192])}


# ------------------------------------------------------------- scenes and eyes

_scenes = {}      # name -> generated scene, kept for the process
_bound = {}       # what the library holds now: scene, eye, counts, network
_weights = {}     # trained sampler networks by case scene


def _scene(name):
    if name not in _scenes:
        _scenes[name] = {"lab": scenes.config1_scene, "field": scenes.config2_scene,
                         "large": scenes.config5_scene}[name]()
    return _scenes[name]


def _eye_rows(case):
    """The (n, 8) ommatidia of a case's eyes, one array per eye."""
    n = case["omm"]
    if case["scene"] == "natural":
        if n == 1000:
            text = gzip.decompress((ROOT / "tests" / "golden" / "equidistant_eye.eye.gz").read_bytes()).decode()
            return [np.asarray([[float(t) for t in ln.split()] for ln in text.splitlines() if ln.strip()], np.float32)]
        return [scenes.fibonacci_eye(n, 0.001, 3.0 * scenes.DEG)]
    if case["scene"] == "lab":
        return [scenes.fibonacci_eye(n, 0.001, 2.0 * scenes.DEG)]
    if case["scene"] == "field":
        return list(scenes.config2_eyes(n=n))
    scene = _scene("large")
    eyes = scenes.config5_eyes()
    poses = scenes.batch_poses(scene, len(eyes), seed=902, extent=EXTENT["large"])
    return [np.concatenate([scenes.world_ommatidia(e, scenes.pose_matrix12(p)) for e, p in zip(eyes, poses)])]


def _load(lib, name):
    """Loads a scene with two compound eyes and the three regular cameras."""
    if _bound.get("scene") == name:
        return
    _bound.clear()
    with tempfile.TemporaryDirectory() as tmp:
        d = pathlib.Path(tmp)
        if name == "natural":
            golden = ROOT / "tests" / "golden"
            path = d / "natural-standin-sky.gltf"
            path.write_bytes(gzip.decompress((golden / "natural_standin_sky.gltf.gz").read_bytes()))
            eye = gzip.decompress((golden / "standin_eye.eye.gz").read_bytes())
            (d / "eyes").mkdir()
            for where in (d, d / "eyes"):
                (where / "1000-horizontallyAcute-variableDegree.eye").write_bytes(eye)
        else:
            scene = _scene(name)
            rows = scenes.fibonacci_eye(16, 0.001, 0.03)
            scene.eyes = [scenes.Eye("left", rows), scenes.Eye("right", rows)]
            scene.cameras = [scenes.Camera("perspective", "perspective", yfov=1.2),
                             scenes.Camera("orthographic", "orthographic", xmag=3.0, ymag=2.0),
                             scenes.Camera("panoramic", "panoramic")]
            path = scenes.write_gltf(d, name, scene)
        lib.loadGlTFscene(str(path).encode())
        if er.last_error(lib):
            raise RuntimeError(er.last_error(lib))
    er.gotoFirstCompoundEye(lib)
    _bound.update(scene=name, first=int(lib.getCurrentCameraIndex()), home=er.pose_np(lib)[:3].copy())


def _poses(case, count, seed):
    """(count, 6) positions and rotations over the scene's ground."""
    name = case["scene"]
    if name == "natural":
        rng = np.random.default_rng([seed, 7])
        p = np.zeros((count, 6), np.float32)
        p[:, 0:3] = _bound["home"] + rng.uniform([-4.0, 0.0, -4.0], [4.0, 1.5, 4.0], (count, 3))
        p[:, 4] = rng.uniform(0.0, 2.0 * math.pi, count)
        return p
    if name == "large":   # the eyes are placed already; the swarm moves a little as a whole
        rng = np.random.default_rng([seed, 8])
        p = np.zeros((count, 6), np.float32)
        p[:, 0:3] = rng.uniform(-0.02, 0.02, (count, 3))
        return p
    return scenes.batch_poses(_scene(name), count, seed=[seed, 9], extent=EXTENT[name])


def _counts(case):
    return scenes.log_uniform_counts(case["omm"], 8, 256, 4) if case["spp"] == 0 else None


def _bind(lib, case):
    """Gives the library the case's scene, eyes and rates (once per case)."""
    key = repr(sorted((k, v) for k, v in case.items() if k != "name"))
    if _bound.get("case") == key:
        return
    _load(lib, case["scene"])
    lib.setSampleRecording(False)
    if case["kind"] == "camera":
        lib.gotoCameraByName(case["camera"].encode())
        er.setRenderSize(lib, case["width"], case["height"])
    elif case["kind"] != "rays":
        for k, rows in enumerate(_eye_rows(case)):
            lib.gotoCamera(_bound["first"] + k)
            er.set_ommatidia_np(lib, rows)
            er.set_sample_counts(lib, None)
            lib.setCurrentEyeShaderName(b"single_dimension_fast")
            if case.get("spp"):
                lib.setCurrentEyeSamplesPerOmmatidium(case["spp"])
        lib.gotoCamera(_bound["first"])
        if case["kind"] == "batch" and case["spp"] == 0:
            er.set_sample_counts(lib, _counts(case))
        if case["kind"] == "frame":
            er.setRenderSize(lib, case["omm"], 1)
    if case["kind"] == "adaptive":
        name = case["scene"]
        if name not in _weights:
            _weights[name] = _train_offline(*_training_rows(lib, case))
        w = _weights[name]
        if lib.mlpSetParams(w.ctypes.data_as(c_void_p), w.size) != 0:
            raise RuntimeError(er.last_error(lib))
        lib.setAdaptiveSampler(0)
        lib.setAdaptiveLabelError(0.01)
    _bound["case"] = key


# ------------------------------------------------------- the sampler's network

def _layers(params):
    """(W, b) per layer of a flat parameter vector: W1, b1, W2, b2, ..."""
    out, at = [], 0
    for i, o in zip(MLP_WIDTHS[:-1], MLP_WIDTHS[1:]):
        out.append((params[at:at + i * o].reshape(i, o), params[at + i * o:at + i * o + o]))
        at += i * o + o
    return out


def _initial_params(seed):
    rng = np.random.default_rng([seed, 11])
    flat = []
    for i, o in zip(MLP_WIDTHS[:-1], MLP_WIDTHS[1:]):
        flat += [rng.normal(0.0, math.sqrt(2.0 / i), i * o), np.zeros(o)]
    return np.concatenate(flat).astype(np.float32)


def _training_rows(lib, case):
    """Pilot features and sample-count labels of held-out poses of the eye."""
    held = dict(case, poses=8 if case["scene"] != "large" else 1)
    poses = _poses(held, held["poses"], 12345)
    n = lib.getCurrentEyeOmmatidialCount()
    mask = (np.random.default_rng(13).random((len(poses), n)) < 20000.0 / (len(poses) * n)).astype(np.uint8)
    lib.setRandomSeed(42)
    lib.setCurrentEyeFrameIndex(1000)
    return er.training_set_np(lib, poses, unit_mask=mask, pilot=8, label_spp=512, error_target=0.01)


def _train_offline(features, labels):
    """The sampler network fitted on the CPU, in float32 torch: what a program
    loads from its own file."""
    x, t = torch.from_numpy(features), torch.from_numpy(labels)
    p = torch.from_numpy(_initial_params(5)).requires_grad_(True)
    opt = torch.optim.Adam([p], lr=2e-3)
    order = torch.Generator().manual_seed(6)
    for _ in range(8):
        for rows in torch.randperm(len(x), generator=order).split(1024):
            h = x[rows]
            pairs = _layers(p)
            for k, (w, b) in enumerate(pairs):
                h = h @ w + b
                h = torch.relu(h) if k + 1 < len(pairs) else h
            loss = (h[:, 0] - t[rows]).square().mean()
            opt.zero_grad()
            loss.backward()
            opt.step()
    return np.ascontiguousarray(p.detach().numpy())


# ------------------------------------------------------------ prepare and run

def prepare(case, seed):
    lib = cra.load_library()
    lib.setVerbosity(False)
    s = {"case": case, "lib": lib, "seed": int(seed) & 0xFFFFFFFF}
    kind = case["kind"]
    if kind == "train":
        rng = np.random.default_rng([seed, 3])
        x = rng.normal(0.0, 1.0, (case["rows"], 16)).astype(np.float32)
        x[:, 3:] = np.abs(x[:, 3:]) * 0.3
        s["x"] = x
        s["t"] = np.clip(3.0 + 8.0 * x[:, 7] + x[:, 0] + rng.normal(0.0, 0.5, case["rows"]), 0.0, 12.0).astype(
            np.float32)
        s["w"] = _initial_params(seed)
        s["out"] = {"params": np.empty(s["w"].size, np.float32), "loss": np.empty(1, np.float32)}
        return s
    _bind(lib, case)
    if kind == "rays":
        rng = np.random.default_rng([seed, 5])
        n = case["rays"]
        origin = scenes.batch_poses(_scene(case["scene"]), 64, seed=[seed, 6], extent=EXTENT[case["scene"]])[:, 0:3]
        d = rng.normal(0.0, 1.0, (n, 3))
        d[:, 1] *= 0.4
        d /= np.linalg.norm(d, axis=1, keepdims=True)
        rays = np.zeros((n, 8), np.float32)
        rays[:, 0:3] = origin[rng.integers(0, 64, n)]
        rays[:, 4:7] = d
        rays[:, 7] = 1e16
        s["rays"] = rays
        s["out"] = {"ids": np.empty(n, np.int32), "tbb": np.empty((n, 3), np.float32)}
        return s
    s["poses"] = _poses(case if kind != "camera" else dict(case, poses=1), case.get("poses", 1), seed)
    units = case.get("poses", 1) * (lib.getCurrentEyeOmmatidialCount() if kind != "camera" else 0)
    if kind == "batch" and case["to"] == "device":
        # poses as 12 floats each, resident; one ordinary frame uploads the eye
        rows = np.empty((len(s["poses"]), 12), np.float32)
        for k, p in enumerate(s["poses"]):
            lib.setCameraPose(*[float(v) for v in p])
            lib.getCameraPose(rows[k])
        s["dev_poses"] = torch.from_numpy(rows).cuda()
        s["out"] = {"colours": torch.empty((len(rows), units // len(rows), 4), device="cuda")}
        if not _bound.get("resident") == _bound["case"]:
            lib.renderFrame()
            _bound["resident"] = _bound["case"]
    elif kind == "batch":
        s["out"] = {"rgb": np.empty((units, 3), np.float32)}
    elif kind == "adaptive":
        s["out"] = {"rgb": np.empty((units, 3), np.float32), "counts": np.empty(units, np.uint32),
                    "samples": np.empty(1, np.uint64)}
    elif kind == "frame":
        eyes = 2 if case["scene"] == "field" else 1
        s["out"] = {"colours": [np.empty((case["omm"], 3), np.float32) for _ in range(eyes)]}
    return s


def _checked(lib, value):
    if value < 0:
        raise RuntimeError(er.last_error(lib))
    return value


def _ptr(a):
    return a.ctypes.data_as(c_void_p)


def run(s):
    case, lib = s["case"], s["lib"]
    kind = case["kind"]
    if kind == "train":
        out, x = s["out"], s["x"]
        lib.mlpSetParams(_ptr(s["w"]), s["w"].size)
        _checked(lib, lib.mlpTrain(_ptr(x), _ptr(s["t"]), x.shape[0], 1, case["batch"], 1e-3, 9, _ptr(out["loss"])))
        _checked(lib, lib.mlpGetParams(_ptr(out["params"]), out["params"].size))
        return out
    if kind == "rays":
        out = s["out"]
        _checked(lib, lib.traceRays(s["rays"], s["rays"].shape[0], out["ids"], out["tbb"]))
        return out
    if kind == "camera":
        lib.setCameraPose(*s["poses"][0].tolist())
        _checked(lib, lib.renderFrame())
        return {"frame": lib.getFramePointer()}
    lib.setRandomSeed(s["seed"])
    if kind == "frame":
        frames = []
        for k, colours in enumerate(s["out"]["colours"]):
            lib.gotoCamera(_bound["first"] + k)
            lib.setCurrentEyeFrameIndex(0)
            lib.setCameraPose(*s["poses"][0].tolist())
            _checked(lib, lib.renderFrame())
            lib.getOmmatidialColours(colours, colours.shape[0])
            frames.append(lib.getFramePointer())
        # one frame buffer serves all eyes: the last eye's frame is in it
        return {"colours": s["out"]["colours"], "frame": frames[-1]}
    lib.setCurrentEyeFrameIndex(0)
    out = s["out"]
    if kind == "adaptive":
        p = s["poses"]
        _checked(lib, lib.renderPoseBatchAdaptive(_ptr(p), p.shape[0], 0.01, 1024, 0.85, _ptr(out["rgb"]),
                                                  _ptr(out["counts"]), _ptr(out["samples"])))
        return {"rgb": out["rgb"], "counts": out["counts"].view(np.int32), "samples": int(out["samples"][0])}
    if case["to"] == "device":
        _checked(lib, lib.renderPoseBatchInto(s["dev_poses"].data_ptr(), s["dev_poses"].shape[0],
                                              out["colours"].data_ptr(), None))
        return out
    _checked(lib, lib.renderPoseBatch(s["poses"], s["poses"].shape[0], _ptr(out["rgb"])))
    return out


# ------------------------------------------------------------------------ work

def work(case):
    kind = case["kind"]
    if kind == "train":
        muls = sum(i * o for i, o in zip(MLP_WIDTHS[:-1], MLP_WIDTHS[1:]))
        steps = -(-case["rows"] // case["batch"])
        return {"bytes": case["rows"] * 17 * 4.0 + steps * muls * 7 * 4.0, "flops": 6.0 * muls * case["rows"]}
    depth = math.ceil(math.log(TRIANGLES[case["scene"]] / 3.0, 4))
    per_ray = 250.0 + depth * 4 * 18.0 + 2 * 60.0
    if kind == "rays":
        rays, units, io = case["rays"], case["rays"], 32 + 16
    elif kind == "camera":
        rays = units = case["width"] * case["height"]
        io = 4
    else:
        omm = case["omm"] or 2149386
        units = omm * case.get("poses", 1) * (2 if kind == "frame" and case["scene"] == "field" else 1)
        if kind == "adaptive":   # the pilot's 8 samples and about as many again
            rays, io = units * 18, 16
        elif case["spp"] == 0:
            rays, io = int(_counts(case).sum()) * case["poses"], 16
        else:
            rays, io = units * case["spp"], 16
    # a triangle is 36 bytes of corners and 36 of colours; no more of them are needed than there are rays
    touched = 72.0 * min(rays, TRIANGLES[case["scene"]])
    return {"bytes": units * float(io) + min(units, case.get("omm") or units) * 32.0 + touched,
            "flops": rays * per_ray}


# ------------------------------------------------------------ 64-bit reference

def exact(case, seed):
    """The lab scene's colours, traced against every triangle in float64 with
    the same random draws; the other scenes have too many triangles (or a
    texture) for that, and a training epoch draws its own row order."""
    if case["kind"] not in ("frame", "batch") or case["scene"] != "lab" or case["spp"] == 0:
        return None
    poses = _poses(case, case.get("poses", 1), seed)
    if len(poses) * case["omm"] * case["spp"] * TRIANGLES["lab"] > 5e9:
        return None
    rows = _eye_rows(case)[0]
    colours = np.concatenate([_exact_colours(rows, p, k, case["spp"], seed) for k, p in enumerate(poses)])
    if case["kind"] == "frame":
        return {"colours": [colours], "frame": None}
    if case["to"] == "device":
        n = np.full((colours.shape[0], 1), float(case["spp"]))
        return {"colours": np.concatenate([colours, n], axis=1).reshape(len(poses), case["omm"], 4)}
    return {"rgb": colours}


def _philox(counter, key):
    """Philox4x32-10 of (n, 4) uint32 counters."""
    mask = np.uint64(0xFFFFFFFF)
    c = [counter[:, k].astype(np.uint64) for k in range(4)]
    k0, k1 = key
    for _ in range(10):
        p0 = c[0] * np.uint64(0xD2511F53)
        p1 = c[2] * np.uint64(0xCD9E8D57)
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), p1 & mask,
             (p0 >> np.uint64(32)) ^ c[3] ^ np.uint64(k1), p0 & mask]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return np.stack(c, axis=1)


def _turned(p, angle, k):
    c, s = np.cos(angle)[:, None], np.sin(angle)[:, None]
    return c * p + s * np.cross(k, p) + (1.0 - c) * np.sum(k * p, axis=1, keepdims=True) * k


def _exact_colours(rows, pose, pose_index, spp, seed):
    omm = rows.astype(np.float64)
    n = len(omm)
    ids = np.repeat(np.arange(n), spp)
    counter = np.zeros((n * spp, 4), np.uint32)
    counter[:, 0] = ids
    counter[:, 1] = np.tile(np.arange(spp), n)
    counter[:, 3] = pose_index
    r = _philox(counter, (int(seed) & 0xFFFFFFFF, 0)) >> np.uint64(8)
    unit = 2.0 ** -24
    normal = np.sqrt(-2.0 * np.log((r[:, 0] + np.uint64(1)) * unit)) * np.cos(2.0 * math.pi * (r[:, 1] * unit))
    spin = (r[:, 2] + np.uint64(1)) * unit * math.pi
    o = omm[ids]
    axis = o[:, 3:6]
    perp = np.cross(np.array([0.0, 1.0, 0.0]), axis)
    flat = perp.sum(axis=1) == 0.0
    perp[flat] = (0.0, 0.0, 1.0)
    perp[~flat] /= np.linalg.norm(perp[~flat], axis=1, keepdims=True)
    d = _turned(_turned(axis, normal * o[:, 6] / 2.35482004503094938, perp), spin, axis)
    start = o[:, 0:3] - axis / np.linalg.norm(axis, axis=1, keepdims=True) * o[:, 7:8]
    world = scenes.pose_matrix12(pose)
    turn = np.stack([world[3:6], world[6:9], world[9:12]], axis=1)
    start, d = start @ turn.T + world[0:3], d @ turn.T
    where = "cuda" if torch.cuda.is_available() else "cpu"
    mesh = _scene("lab").meshes[0]
    corner = torch.from_numpy(mesh.pos[mesh.idx].astype(np.float64)).to(where)
    paint = torch.from_numpy(mesh.col[mesh.idx][:, :, :3].astype(np.float64)).to(where)
    v0, e1, e2 = corner[:, 0], corner[:, 1] - corner[:, 0], corner[:, 2] - corner[:, 0]
    start, d = torch.from_numpy(start).to(where), torch.from_numpy(d).to(where)
    near = torch.from_numpy(o[:, 7]).to(where)
    out = []
    for at in range(0, len(d), 1024):
        dd, oo = d[at:at + 1024, None, :], start[at:at + 1024, None, :]
        p = torch.linalg.cross(dd.expand(-1, len(v0), -1), e2[None].expand(dd.shape[0], -1, -1))
        det = (e1[None] * p).sum(-1)
        tv = oo - v0[None]
        u = (tv * p).sum(-1) / det
        q = torch.linalg.cross(tv, e1[None].expand(dd.shape[0], -1, -1))
        v = (dd * q).sum(-1) / det
        t = (e2[None] * q).sum(-1) / det
        good = (u >= 0) & (v >= 0) & (u + v <= 1) & (t >= near[at:at + 1024, None])
        t = torch.where(good, t, torch.full_like(t, math.inf))
        best, which = t.min(dim=1)
        at_ray = torch.arange(len(which), device=where)
        b1, b2 = u[at_ray, which][:, None], v[at_ray, which][:, None]
        c = paint[which]
        seen = ((1.0 - b1 - b2) * c[:, 0] + b1 * c[:, 1] + b2 * c[:, 2]).clamp_min(0.0) ** 2.2
        up = torch.nn.functional.normalize(d[at:at + 1024], dim=1)[:, 1:2].clamp(-1.0, 1.0)
        mix = (torch.asin(up) * 2.0 / math.pi).clamp_min(0.0)
        low = torch.tensor([143.0, 179.0, 203.0], dtype=torch.float64, device=where) / 255.0 * 0.8
        high = torch.tensor([1.0, 31.0, 117.0], dtype=torch.float64, device=where) / 255.0
        out.append(torch.where(torch.isfinite(best)[:, None], seen, low * (1.0 - mix) + high * mix))
    return torch.cat(out).reshape(n, spp, 3).mean(dim=1).cpu().numpy()
