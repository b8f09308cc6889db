"""Performance cases of the tracer, the observation post-pass, point queries and scene loading.

Each case is one pass through the package's public entry points with the sizes that its
users meet: the drop-in ``torch_sdf.cast_rays`` from one small environment up, the
multi-scene tracer with explicit rays or rays from poses, the post-pass in the policy's and
the reference's output formats, spawn-check point queries, and a scene rotation (upload,
conversion, first trace). The scenes, sensor layouts and step limits are those of the
benchmark (``navi_amd/workloads.py``) and of ``bench_sdfdag``, with generic odd sizes
beside them. A scene stands for a compiled asset, the same in every state of a case; rays,
poses, distances and points come from the seed.
"""

from __future__ import annotations

import concurrent.futures
import functools
import math

import numpy as np
import torch

from navi_amd import scenes as S
from navi_amd import torch_sdf
from navi_amd.multiscene import ResidentScenes

DEVICE = "cuda"
CLEARANCE = 0.15  # the observation's collision clearance
# mean march steps per ray of the scene families (the tracer's own step counts at 30 m)
MEAN_STEPS = {"box_room": 20.0, "cluttered": 27.0, "rooms": 64.0, "corpus": 45.0}
# of one march step: the sample point (3 fma), the box test (6) and the distance added
STEP_FLOPS = 13.0


def listed():
    return [
        # one environment with a small sensor in a small room: latency of one call
        _dropin("room_one_env", "box_room", 1, 64, 1, 64, 16, 64),
        # the default actor count of a trainer on a workstation, full sensor
        _dropin("cluttered_four_envs", "cluttered", 2, 128, 4, 256, 48, 128),
        # a caller that keeps direction validation on and asks for step counts, on a
        # sensor whose bins divide by nothing
        _dropin("ragged_validated", "rooms", 9, 256, 7, 101, 37, 200, validate=True, steps=True),
        # a mid-size batch on one scene, rays declared in sensor order
        _dropin("rooms_64_envs", "rooms", 3, 512, 64, 256, 48, 256, tiled=True),
        # the whole multi-scene batch with explicit rays
        _multi("corpus_explicit", 16, 1024, 1024, 256, 48, 256, rays="explicit"),
        # the trainer's step on it: rays from poses, policy depth, move checks
        _multi("corpus_step", 16, 1024, 1024, 256, 48, 256, observe="policy"),
        # one of eight shards of that batch with bfloat16 distances
        _multi("corpus_shard_bf16", 16, 1024, 128, 256, 48, 256, dtype="bfloat16"),
        # bench_sdfdag's default: four actors, the reference's observation tensors
        _multi("four_actors_step", 1, 1024, 4, 256, 48, 256, observe="reference"),
        # the reference's observation tensors for a full batch, two frames
        _observe("observe_reference", 1024, 256, 48, "reference"),
        # policy depth at the largest sensor of the reference's resolution tables
        _observe("observe_policy_wide", 256, 512, 96, "policy"),
        # spawn candidates of a full batch of actors
        {"name": "spawn_points", "kind": "points", "scenes": 16, "resolution": 1024, "points": 65536},
        # a scene rotation: words from the host, record layout, the first trace
        {"name": "scene_rotation", "kind": "load", "family": "cluttered", "scene": 100, "resolution": 1024,
         "envs": 4, "az": 256, "el": 48, "max_steps": 256},
    ]


def draw(rng):
    kind = rng.choice(["dropin", "dropin", "dropin", "multi", "multi", "multi", "observe", "observe", "points", "load"])
    if kind in ("dropin", "load"):
        family = rng.choice(["box_room", "cluttered", "rooms"])
        resolution = rng.choice([64, 128, 256] if family == "box_room" else [128, 256, 512])
        scene = rng.randrange(1, 5)
    if kind == "dropin":
        az, el = _sensor(rng)
        envs = _log_int(rng, 1, min(96, 1_500_000 // (az * el)))
        return _dropin(None, family, scene, resolution, envs, az, el, rng.choice([64, 128, 200, 256]),
                       max_distance=rng.choice([10.0, 20.0, 30.0, 50.0]), tiled=rng.random() < 0.5,
                       validate=rng.random() < 0.25, steps=rng.random() < 0.25)
    if kind == "multi":
        az, el = _sensor(rng)
        scenes, resolution = rng.choice([(1, 512), (2, 256), (5, 512), (8, 256), (3, 1024), (16, 1024)])
        envs = _log_int(rng, 1, min(1024, 6_000_000 // (az * el)))
        observe = rng.choice(["none", "none", "policy", "reference"])
        return _multi(None, scenes, resolution, envs, az, el, rng.choice([128, 256]),
                      rays=rng.choice(["poses", "poses", "explicit"]), observe=observe,
                      dtype=rng.choice(["float32", "float32", "bfloat16"]) if observe == "none" else "float32")
    if kind == "observe":
        az, el = _sensor(rng)
        return _observe(None, _log_int(rng, 1, min(1024, 12_000_000 // (az * el))), az, el,
                        rng.choice(["policy", "reference", "both"]))
    if kind == "points":
        return {"kind": "points", "scenes": rng.choice([1, 5]), "resolution": 512, "points": _log_int(rng, 64, 1 << 20)}
    return {"kind": "load", "family": family, "scene": scene, "resolution": resolution, "envs": rng.randrange(1, 9),
            "az": 256, "el": 48, "max_steps": 256}


def _sensor(rng):
    """Azimuth and elevation bins: the named sensors half of the time, any size otherwise."""
    if rng.random() < 0.5:
        return rng.choice([(64, 16), (128, 24), (256, 48), (384, 72), (512, 96)])
    return _log_int(rng, 24, 400), _log_int(rng, 9, 90)


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(max(lo, hi)))))))


def _named(name, case):
    return {"name": name, **case} if name else case


def _dropin(name, family, scene, resolution, envs, az, el, max_steps, max_distance=30.0, tiled=False,
            validate=False, steps=False):
    return _named(name, {"kind": "dropin", "family": family, "scene": scene, "resolution": resolution, "envs": envs,
                         "az": az, "el": el, "max_steps": max_steps, "max_distance": max_distance, "tiled": tiled,
                         "validate": validate, "steps": steps})


def _multi(name, scenes, resolution, envs, az, el, max_steps, rays="poses", observe="none", dtype="float32"):
    return _named(name, {"kind": "multi", "scenes": scenes, "resolution": resolution, "envs": envs, "az": az,
                         "el": el, "max_steps": max_steps, "max_distance": 30.0, "rays": rays, "observe": observe,
                         "dtype": dtype})


def _observe(name, envs, az, el, outputs):
    return _named(name, {"kind": "observe", "envs": envs, "az": az, "el": el, "outputs": outputs,
                         "max_distance": 30.0})


# ---- scenes ----


@functools.lru_cache(maxsize=None)
def _scene(family, seed, resolution, threads=8):
    """A compiled scene (the asset a user has on disk)."""
    scene = getattr(S, family)(seed=seed, resolution=resolution)
    scene.compile(threads=threads)
    return scene


@functools.lru_cache(maxsize=None)
def _corpus(count, resolution):
    """The first ``count`` of the benchmark's scenes: cluttered volumes and room grids in turn."""
    seeds = [(S.corpus_scene(s, resolution).name, s) for s in range(100, 100 + count)]
    with concurrent.futures.ThreadPoolExecutor(max_workers=4) as pool:
        return list(pool.map(lambda fs: _scene(fs[0], fs[1], resolution, 4), seeds))


def _triple(scene):
    return scene.words, scene.bbox_min_list, scene.bbox_max


def _poses(scenes, envs, rng):
    """Scene ids, free positions and yaws of ``envs`` envs spread over ``scenes``."""
    ids = rng.integers(0, len(scenes), envs).astype(np.int32)
    pos = np.empty((envs, 3), np.float32)
    for s, scene in enumerate(scenes):
        at = np.flatnonzero(ids == s)
        if at.size:
            pos[at] = scene.free_origins(rng, at.size)
    yaw = rng.uniform(0.0, 2.0 * math.pi, envs).astype(np.float32)
    to = lambda a: torch.from_numpy(a).to(DEVICE)  # noqa: E731
    return to(ids), to(pos), to(np.stack((np.cos(yaw), np.sin(yaw)), 1))


def _local(case):
    return torch.from_numpy(S.canonical_directions(case["az"], case["el"])).to(DEVICE)


def _rays(local, pos, rot):
    """World rays ``[E, R, 3]`` of the poses, as the reference builds them."""
    c, s = rot[:, :1], rot[:, 1:]
    x, y, z = local[:, 0], local[:, 1], local[:, 2]
    dirs = torch.stack((x * c + z * s, y.expand(pos.shape[0], -1), -x * s + z * c), dim=2).contiguous()
    return pos[:, None, :].expand_as(dirs).contiguous(), dirs


def _outputs(envs, rays, dtype=torch.float32):
    return (torch.empty((envs, rays), device=DEVICE, dtype=dtype),
            torch.empty((envs, rays), device=DEVICE, dtype=torch.int32))


# ---- inputs ----


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def _prepare_dropin(case, seed):
    scene = _scene(case["family"], case["scene"], case["resolution"])
    _, pos, rot = _poses([scene], case["envs"], np.random.default_rng(seed))
    origins, dirs = _rays(_local(case), pos, rot)
    out_d, out_s = _outputs(*origins.shape[:2])
    state = {"case": case, "origins": origins, "dirs": dirs, "d": out_d, "s": out_s, "extra": {},
             "lo": scene.bbox_min_list, "hi": scene.bbox_max}
    if case.get("tiled"):
        state["extra"]["elevation_bins"] = case["el"]
    if case.get("steps"):
        state["extra"]["out_steps"] = torch.empty_like(out_s)
    if case["kind"] == "load":
        state["words"] = scene.words.view(np.int64)
    else:
        state["dag"] = torch.from_numpy(scene.words.view(np.int64)).to(DEVICE)
        torch_sdf.prepare(state["dag"], state["lo"], state["hi"])
    return state


def _prepare_multi(case, seed):
    scenes = _corpus(case["scenes"], case["resolution"])
    rng = np.random.default_rng(seed)
    ids, pos, rot = _poses(scenes, case["envs"], rng)
    local = _local(case)
    E, R, az, el = case["envs"], int(local.shape[0]), case["az"], case["el"]
    out_d, out_s = _outputs(E, R, getattr(torch, case["dtype"]))
    state = {"case": case, "res": ResidentScenes([_triple(s) for s in scenes], DEVICE, keep_words=False), "ids": ids,
             "pos": pos, "rot": rot, "local": local, "d": out_d, "s": out_s}
    if case["rays"] == "explicit":
        state["origins"], state["dirs"] = _rays(local, pos, rot)
    if case["observe"] != "none":
        state.update(_observe_outputs(case["observe"], E, az, el))
    if case["observe"] == "policy":
        jitter = rng.uniform(-0.3, 0.3, (E, 4, 3)).astype(np.float32)
        state["points"] = (pos[:, None, :] + torch.from_numpy(jitter).to(DEVICE)).reshape(-1, 3).contiguous()
        state["point_ids"] = ids.repeat_interleave(4).contiguous()
        state.update(_point_outputs(4 * E))
    # a running program is past the launches in which the scenes' costs are measured
    for _ in range(2):
        _trace(state)
        torch.cuda.synchronize()
    return state


def _observe_outputs(kind, envs, az, el):
    out = {"stats": torch.empty((envs, 5), device=DEVICE),
           "collision": torch.empty((envs,), device=DEVICE, dtype=torch.int32)}
    if kind in ("policy", "both"):
        out["depth16"] = torch.empty((envs, 1, el, az), device=DEVICE, dtype=torch.float16)
    if kind in ("reference", "both"):
        out["obs"] = torch.empty((envs, 3, az, el), device=DEVICE)
        out["prev"] = torch.zeros((envs, az, el), device=DEVICE)
        out["delta"] = torch.empty((envs, az, el), device=DEVICE)
    return out


def _point_outputs(n):
    return {"pd": torch.empty((n,), device=DEVICE),
            "ps": torch.empty((n,), device=DEVICE, dtype=torch.int32),
            "pk": torch.empty((n,), device=DEVICE, dtype=torch.int32)}


def _frames(case, seed):
    """Two frames of traced distances and semantics: most rays hit within a few metres (the
    nearest 0.1 to 0.5 m away), some run past the range, a few leave the scene."""
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(int(seed))
    shape = (2, case["envs"], case["az"] * case["el"])
    u = torch.rand(shape, generator=gen, device=DEVICE)
    v = torch.rand(shape, generator=gen, device=DEVICE)
    near = 0.1 + 0.4 * torch.rand((1, case["envs"], 1), generator=gen, device=DEVICE)
    hit = (near - 4.0 * torch.log1p(-u * 0.9995)).clamp_(max=29.5)
    d = torch.where(v < 0.90, hit, torch.where(v < 0.98, 30.0 + 0.5 * u, 1000.0 + 30.0 * u))
    sem = torch.where(v < 0.90, (1 + 7 * u).to(torch.int32), torch.zeros((), device=DEVICE, dtype=torch.int32))
    return d.contiguous(), sem.contiguous()


def _prepare_observe(case, seed):
    d, sem = _frames(case, seed)
    res = ResidentScenes([_triple(_scene("box_room", 1, 64))], DEVICE, keep_words=False)
    return {"case": case, "res": res, "frames": d, "sems": sem,
            **_observe_outputs(case["outputs"], case["envs"], case["az"], case["el"])}


def _prepare_points(case, seed):
    scenes = _corpus(case["scenes"], case["resolution"])
    rng = np.random.default_rng(seed)
    ids = rng.integers(0, len(scenes), case["points"]).astype(np.int32)
    lo = np.array([s.bbox_min_list for s in scenes])[ids]
    hi = np.array([s.bbox_max for s in scenes])[ids]
    pts = rng.uniform(lo, hi).astype(np.float32)
    return {"case": case, "res": ResidentScenes([_triple(s) for s in scenes], DEVICE, keep_words=False),
            "points": torch.from_numpy(pts).to(DEVICE), "point_ids": torch.from_numpy(ids).to(DEVICE),
            **_point_outputs(case["points"])}


_PREPARE = {"dropin": _prepare_dropin, "load": _prepare_dropin, "multi": _prepare_multi, "observe": _prepare_observe,
            "points": _prepare_points}


# ---- one pass ----


def run(state):
    return _RUN[state["case"]["kind"]](state)


def _cast(state, dag):
    case = state["case"]
    torch_sdf.cast_rays(dag, state["origins"], state["dirs"], state["d"], state["s"], case["max_steps"],
                        case.get("max_distance", 30.0), state["lo"], state["hi"], case["resolution"],
                        not case.get("validate", False), **state["extra"])
    out = {"d": state["d"], "s": state["s"]}
    if case.get("steps"):
        out["steps"] = state["extra"]["out_steps"]
    return out


def _run_dropin(state):
    return _cast(state, state["dag"])


def _run_load(state):
    dag = torch.from_numpy(state["words"]).to(DEVICE)
    torch_sdf.prepare(dag, state["lo"], state["hi"])
    return _cast(state, dag)


def _trace(state):
    case = state["case"]
    if case["rays"] == "explicit":
        state["res"].cast_rays(state["ids"], state["origins"], state["dirs"], state["d"], state["s"],
                               case["max_steps"], case["max_distance"], elevation_bins=case["el"])
    else:
        state["res"].cast_rays_poses(state["ids"], state["local"], state["pos"], state["rot"], state["d"], state["s"],
                                     case["max_steps"], case["max_distance"], elevation_bins=case["el"])


def _post(state, distances, semantics):
    case = state["case"]
    extra = {}
    if "depth16" in state:
        extra["out_depth_f16"] = state["depth16"]
    if "obs" in state:
        extra.update(semantics=semantics, out_obs=state["obs"], prev_depth=state["prev"], out_delta=state["delta"])
    if "points" in state:
        extra.update(points=state["points"], point_scene=state["point_ids"], point_distances=state["pd"],
                     point_semantics=state["ps"], point_kind=state["pk"])
    state["res"].observe(distances, case["az"], case["el"], case["max_distance"], out_stats=state["stats"],
                         out_collision=state["collision"], collision_clearance=CLEARANCE, **extra)


_RETURNED = ("stats", "collision", "depth16", "obs", "prev", "delta", "pd", "ps", "pk")


def _run_multi(state):
    _trace(state)
    if state["case"]["observe"] != "none":
        _post(state, state["d"], state["s"])
    return {"d": state["d"], "s": state["s"], **{k: state[k] for k in _RETURNED if k in state}}


def _run_observe(state):
    # two consecutive frames: the second one's delta is against the first one's depth
    for k in range(2):
        _post(state, state["frames"][k], state["sems"][k])
    return {k: state[k] for k in _RETURNED if k in state}


def _run_points(state):
    state["res"].point_query(state["points"], state["pd"], state["ps"], point_scene=state["point_ids"],
                             out_kind=state["pk"])
    return {k: state[k] for k in ("pd", "ps", "pk")}


_RUN = {"dropin": _run_dropin, "load": _run_load, "multi": _run_multi, "observe": _run_observe, "points": _run_points}


# ---- what a pass cannot do without ----


def work(case):
    kind = case["kind"]
    if kind == "points":
        return {"bytes": case["points"] * (12 + 4 + 12), "flops": case["points"] * 9.0 * 10}
    rays = case["envs"] * case["az"] * case["el"]
    if kind == "observe":
        return {"bytes": 2 * rays * _observe_bytes(case["outputs"]), "flops": 2 * rays * 20.0}
    family = case.get("family", "corpus")
    flops = rays * MEAN_STEPS[family] * STEP_FLOPS
    if kind in ("dropin", "load"):
        b = rays * (24 + 8 + (4 if case.get("steps") else 0))
        if kind == "load":
            # a word of the DAG is read once (its size grows with the surface, 4.3 M words at 1024^3)
            b += 8 * 4_300_000 * (case["resolution"] / 1024) ** 2
        return {"bytes": b, "flops": flops}
    b = rays * ((2 if case["dtype"] != "float32" else 4) + 4 + (24 if case["rays"] == "explicit" else 0))
    if case["observe"] != "none":
        b += rays * (_observe_bytes(case["observe"]) - 4) + (case["envs"] * 4 * 28 if case["observe"] == "policy" else 0)
        flops += rays * 20.0
    return {"bytes": b, "flops": flops}


def _observe_bytes(outputs):
    # distance read; the policy's depth written; semantic and previous depth read, three
    # planes, delta and previous depth written
    return 4 + (2 if outputs in ("policy", "both") else 0) + (28 if outputs in ("reference", "both") else 0)


def tolerance(case):
    # a march is a fixed sequence of binary32 operations: another order of steps is
    # another result, so distances, semantics and step counts agree in every bit
    if case["kind"] in ("dropin", "load", "points") or case["kind"] == "multi" and case["observe"] == "none":
        return "exact"
    outputs = case["observe"] if case["kind"] == "multi" else case["outputs"]
    if outputs == "reference":
        # float32 log1p within an ulp or two, and a difference of two of them
        return {"rel": 1e-6, "max": 4e-6}
    # binary16 depth: rounding ties of one unit in the last place
    return {"rel": 5e-5, "max": 1.2e-3}


def exact(case, seed):
    """The post-pass in 64 bits. A trace or a point query has no such value: its result is
    defined by the binary32 march, and a march in 64 bits takes other steps at cell faces."""
    if case["kind"] != "observe":
        return None
    d, sem = _frames(case, seed)
    E, az, el = case["envs"], case["az"], case["el"]
    top = case["max_distance"]
    x = d[1].double()
    c = x.clamp(0.0, top)
    log_top = math.log1p(top)
    q = [(f.double().clamp(0.0, top).log1p() / log_top).clamp(0.0, 1.0) for f in d]
    n = az * el
    fwd = max(1, az // 6)
    band = (c >= 1.5) & (c <= 30.0)
    grid = band.view(E, az, el)
    stats = torch.stack((c.amin(1), (c >= top - 1e-3).double().sum(1) / n, (c <= 2.0).double().sum(1) / n,
                         band.double().sum(1) / n,
                         (grid[:, :fwd].double().sum((1, 2)) + grid[:, az - fwd:].double().sum((1, 2))) / (2 * fwd * el)),
                        dim=1)
    out = {"stats": stats, "collision": (c.amin(1) < CLEARANCE).to(torch.int32)}
    if case["outputs"] in ("policy", "both"):
        out["depth16"] = q[1].view(E, 1, az, el).transpose(2, 3).contiguous()
    if case["outputs"] in ("reference", "both"):
        out["obs"] = torch.stack((q[1], sem[1].double(), torch.ones_like(x)), dim=1).view(E, 3, az, el)
        out["prev"] = q[1].view(E, az, el)
        out["delta"] = (q[1] - q[0]).view(E, az, el)
    return out
