"""The work a user of this framework has it do, as cases that can be timed and compared.

A case is a dict of plain values; `kind` says which path it takes:

  scan       a simulator's simulate(): one sensor model cast from n poses into a kept bundle
  fleet      BatchSimulatorHip: sensors of several models, each with its own poses
  particles  pose_range_loss forward and backward: loss and 6-DoF gradient per particle
  rcc        BatchedRCC: one outer correction iteration of many pose hypotheses
  register   correspondence statistics of scans already at hand, then Umeyama
  noise      range noise on a buffer of ranges
  closest    closest points of a batch of queries
  rebuild    a new mesh from host arrays: BVH build, then one scan of it
  refit      moved vertices: refit of a kept map, then one scan of it

Meshes are the repository's synthetic scenes (a map file on disk, as it were: the same for
every seed); poses, directions, queries, ranges, clouds and motions come from the seed.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from rmagine_amd import adjoint, icp, noise, scenes, simulation
from rmagine_amd import math as rmath
from rmagine_amd import types as T

DEV = "cuda"
ALL = "hits,ranges,points,normals,face_ids,geom_ids,object_ids"
CELL = 0.1  # terrain grid spacing in metres


def listed():
    return [
        # one lidar revolution in a room, everything asked for: a localisation node's call
        # per scan, where the launch and the host path are most of the time
        {"name": "scan_one", "kind": "scan", "scene": "room", "model": "vlp16", "w": 900, "h": 16, "poses": 1,
         "attrs": ALL},
        # the same sensor from 100 places at once: the small batch of a particle filter
        {"name": "scan_room", "kind": "scan", "scene": "room", "model": "vlp16", "w": 900, "h": 16, "poses": 100,
         "attrs": ALL},
        # the headline: 1,000 high-resolution lidars on 2.1M triangles, all attributes
        {"name": "scan_terrain", "kind": "scan", "scene": "terrain", "grid": 1024, "model": "sphere", "w": 1024,
         "h": 128, "poses": 1000, "attrs": ALL},
        # a lidar whose beams start off-centre (per-ray origins), ranges and points only
        {"name": "scan_beams", "kind": "scan", "scene": "terrain", "grid": 1024, "model": "ondn", "w": 1024,
         "h": 128, "poses": 250, "attrs": "hits,ranges,points"},
        # lidars, depth cameras and scattered ray lists of a fleet in one persistent launch
        {"name": "fleet_mixed", "kind": "fleet", "sensors": 30, "poses": 16},
        # gradient-based localisation: loss and gradient of 2,000 particles
        {"name": "particles", "kind": "particles", "scene": "fine_room", "w": 900, "h": 16, "n": 2000},
        # global localisation: one correction iteration of 256 hypotheses
        {"name": "rcc_hypotheses", "kind": "rcc", "rays": 32768, "n": 256, "inner": 5},
        # registration of one high-resolution scan against its simulated counterpart
        {"name": "register_scan", "kind": "register", "stat": "p2l", "seg": 131072, "n": 1, "ids": False},
        # noise on the ranges of 250 simulated scans
        {"name": "noise_ranges", "kind": "noise", "model": "rel_gaussian", "n": 32_768_000},
        # a point cloud of a million points matched to the map, in no particular order
        {"name": "closest_points", "kind": "closest", "scene": "terrain", "grid": 1024, "n": 1_048_576,
         "max_distance": 0.0},
        # a map that changed (mapping, a new file): from host arrays to the first scan
        {"name": "map_rebuild", "kind": "rebuild", "scene": "terrain", "grid": 1024},
        # a deforming map: every vertex moved, refit, one scan
        {"name": "map_refit", "kind": "refit", "scene": "terrain", "grid": 1024},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_scene(rng):
    scene = rng.choice(("room", "fine_room", "objects", "terrain"))
    return {"scene": scene, **({"grid": _log(rng, 64, 1024)} if scene == "terrain" else {})}


ATTR_SETS = (ALL, "ranges", "hits,ranges", "hits,ranges,points", "hits,points,normals", "ranges,normals,face_ids")


def draw(rng):
    kind = rng.choice(("scan", "scan", "scan", "fleet", "particles", "rcc", "register", "register", "noise", "closest",
                       "closest", "rebuild", "refit"))
    if kind == "scan":
        model = rng.choice(("vlp16", "sphere", "camera", "o1dn", "ondn"))
        c = {"kind": kind, **_draw_scene(rng), "model": model}
        if model == "vlp16":
            c["w"], c["h"] = 900, 16
        elif model == "camera":
            c["w"], c["h"] = _log(rng, 80, 640), _log(rng, 60, 480)
        elif model == "o1dn":
            c["w"], c["h"] = _log(rng, 1000, 50_000), 1
        else:
            c["w"], c["h"] = _log(rng, 256, 2048), _log(rng, 16, 128)
        # scattered rays cost several times a coherent one
        most = (8_000_000 if model == "o1dn" else 32_000_000) // (c["w"] * c["h"])
        return {**c, "poses": _log(rng, 1, max(1, min(1000, most))), "attrs": rng.choice(ATTR_SETS)}
    if kind == "fleet":
        return {"kind": kind, "sensors": rng.randint(3, 30), "poses": _log(rng, 1, 16)}
    if kind == "particles":
        return {"kind": kind, "scene": rng.choice(("room", "fine_room")), "w": _log(rng, 180, 900),
                "h": rng.choice((1, 8, 16)), "n": _log(rng, 1, 8000)}
    if kind == "rcc":
        rays = _log(rng, 1000, 50_000)
        return {"kind": kind, "rays": rays, "n": _log(rng, 1, max(1, min(500, 8_000_000 // rays))),
                "inner": rng.randint(1, 6)}
    if kind == "register":
        n = rng.choice((1, 1, _log(rng, 2, 1000)))
        return {"kind": kind, "stat": rng.choice(("p2l", "p2p")), "seg": _log(rng, 500, min(2_000_000, 16_000_000 // n)),
                "n": n, "ids": rng.random() < 0.25}
    if kind == "noise":
        return {"kind": kind, "model": rng.choice(("gaussian", "rel_gaussian", "uniform_dust")),
                "n": _log(rng, 1000, 100_000_000)}
    if kind == "closest":
        return {"kind": kind, **_draw_scene(rng), "n": _log(rng, 100, 1_500_000),
                "max_distance": rng.choice((0.0, 0.0, round(rng.uniform(0.2, 5.0), 2)))}
    return {"kind": kind, "scene": "terrain", "grid": _log(rng, 64, 1024)}


# ---- scenes and models ---------------------------------------------------------------------


@functools.lru_cache(maxsize=None)
def _mesh(scene, grid=0):
    """(vertices, faces, what poses are placed by) of a scene, host arrays."""
    if scene == "terrain":
        h = scenes.terrain_heights(grid)
        return (*scenes.heightfield_mesh(h, CELL), h)
    if scene == "objects":
        return (*scenes.objects_mesh(), None)
    V, F, boxes = scenes.room_with_boxes()
    if scene == "fine_room":
        V, F, _, _ = scenes.fine_room_workload(n_particles=1)
    return V, F, boxes


def _mesh_of(case):
    return _mesh(case["scene"], case.get("grid", 0))


def _map_of(case):
    V, F, _ = _mesh_of(case)
    return simulation.HipMap(V, F, device=DEV)


def _terrain_points(rng, n, heights, share=0.8):
    half = (heights.shape[0] - 1) / 2.0 * CELL * share
    x, y = rng.uniform(-half, half, n), rng.uniform(-half, half, n)
    return x, y, scenes.terrain_height_at(heights, CELL, x, y)


def _poses(case, n, seed):
    """(n, 8) float32 host poses inside the scene, yaw only (objects: any rotation)."""
    rng = np.random.default_rng(seed)
    info = _mesh_of(case)[2]
    if case["scene"] in ("room", "fine_room"):
        return scenes.poses_in_room(n, info, seed=seed)
    if case["scene"] == "objects":
        q = rng.normal(size=(n, 4))
        return T.make_transforms(rng.uniform(-80.0, 80.0, size=(n, 3)), q / np.linalg.norm(q, axis=1, keepdims=True))
    x, y, z = _terrain_points(rng, n, info)
    yaw = 0.5 * rng.uniform(-math.pi, math.pi, n)
    q = np.stack([np.zeros(n), np.zeros(n), np.sin(yaw), np.cos(yaw)], 1)
    return T.make_transforms(np.stack([x, y, z + 1.5], 1), q)


def _sphere(w, h, phi_deg):
    """h rows over +-phi_deg, w columns over the full turn, 0.1-100 m."""
    return T.SphericalModel(
        phi=T.DiscreteInterval(T.f32(-phi_deg * T.DEG_TO_RAD), T.f32(2.0 * phi_deg / max(1, h - 1) * T.DEG_TO_RAD), h),
        theta=T.DiscreteInterval(T.f32(-math.pi), T.f32(2.0 * math.pi / w), w), range=T.Interval(0.1, 100.0))


def _model(name, w, h, seed):
    if name == "vlp16":
        return scenes.vlp16_workload_model()
    if name == "sphere":
        return _sphere(w, h, 22.5)
    if name == "camera":  # 90 degrees across
        return T.PinholeModel(width=w, height=h, range=T.Interval(0.1, 100.0), f=(w / 2.0, w / 2.0),
                              c=((w - 1) / 2.0, (h - 1) / 2.0))
    if name == "o1dn":
        dirs = scenes.random_unit_dirs(w * h, np.random.default_rng(seed + 1))
        return T.O1DnModel(w, h, T.Interval(0.1, 100.0), (0.0, 0.0, 0.0), dirs)
    # a scanner's grid whose beams start 15.8 mm off the centre along their azimuth
    phi = np.deg2rad(np.linspace(-22.5, 22.5, h))[:, None]
    th = (-math.pi + np.arange(w) * 2.0 * math.pi / w)[None, :]
    one = np.ones((h, w))
    dirs = np.stack([np.cos(phi) * np.cos(th), np.cos(phi) * np.sin(th), np.sin(phi) * one], -1)
    origs = 0.0158 * np.stack([np.cos(th) * one, np.sin(th) * one, 0.0 * one], -1)
    return T.OnDnModel(w, h, T.Interval(0.1, 100.0), origs.reshape(-1, 3).astype(np.float32),
                       dirs.reshape(-1, 3).astype(np.float32))


def _device(a):
    return torch.as_tensor(np.ascontiguousarray(a), device=DEV)


def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _bundle(model, n, attrs):
    return simulation.resize_memory_bundle(simulation.Bundle(), model.getWidth(), model.getHeight(), n,
                                           tuple(attrs.split(",")), device=DEV)


def _results(bundle):
    return {k: getattr(bundle, k) for k in bundle.enabled()}


# ---- preparation ------------------------------------------------------------------------------


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def _prepare_scan(case, seed):
    model = _model(case["model"], case["w"], case["h"], seed)
    sim = simulation.simulator_for(model, _map_of(case), device=DEV)
    return {"run": _run_scan, "sim": sim, "Tbm": _device(_poses(case, case["poses"], seed)),
            "bundle": _bundle(model, case["poses"], case["attrs"])}


def _run_scan(s):
    return _results(s["sim"].simulate(s["Tbm"], s["bundle"]))


def _fleet_sizes(case):
    """(model name, w, h) of every sensor of a fleet: 40 % lidars, 30 % depth cameras, 30 % lists."""
    rng = np.random.default_rng(case["sensors"])
    out = []
    for i in range(case["sensors"]):
        if i % 10 in (0, 3, 6, 9):
            out.append(("vlp16", 900, 16))
        elif i % 10 in (1, 4, 7):
            out.append(("camera", 640, 480))
        else:
            out.append(("o1dn", int(rng.integers(1000, 50_001)), 1))
    return out


def _prepare_fleet(case, seed):
    place = {"scene": "objects"}
    entries = [{"model": _model(name, w, h, seed + i), "Tbm": _device(_poses(place, case["poses"], seed * 1000 + i)),
                "attrs": ("hits", "ranges")} for i, (name, w, h) in enumerate(_fleet_sizes(case))]
    return {"run": _run_fleet, "batch": simulation.BatchSimulatorHip(_map_of(place), entries, device=DEV)}


def _run_fleet(s):
    return [_results(b) for b in s["batch"].simulate()]


def _particle_inputs(case, seed):
    """(model, true pose, start poses, (n, 6) pose perturbations), host arrays."""
    rng = np.random.default_rng(seed)
    true = _poses(case, 1, seed)
    T0 = np.repeat(true, case["n"], 0)
    T0[:, 4:6] += rng.normal(scale=0.2, size=(case["n"], 2)).astype(np.float32)
    xi = rng.normal(scale=0.01, size=(case["n"], 6))
    xi[:, 5] += rng.normal(scale=math.radians(3.0), size=case["n"])
    return _sphere(case["w"], case["h"], 15.0), true, T0, xi


def _prepare_particles(case, seed):
    model, true, T0, xi = _particle_inputs(case, seed)
    sim = simulation.simulator_for(model, _map_of(case), device=DEV)
    scan = sim.simulate(_device(true), attrs=("hits", "ranges"))
    target = scan.ranges + 0.01 * torch.randn(scan.ranges.shape, generator=_generator(seed), device=DEV)
    return {"run": _run_particles, "sim": sim, "T0": _device(T0), "xi": _device(xi).requires_grad_(),
            "target": target.contiguous(), "mask": scan.hits}


def _run_particles(s):
    loss = adjoint.pose_range_loss(s["xi"], s["T0"], s["sim"], s["target"], s["mask"])
    (grad,) = torch.autograd.grad(loss.sum(), s["xi"])
    return {"loss": loss.detach(), "grad": grad}


def _prepare_rcc(case, seed):
    rng = np.random.default_rng(seed)
    model = _model("o1dn", case["rays"], 1, seed)
    hm = _map_of({"scene": "objects"})
    sim = simulation.simulator_for(model, hm, device=DEV)
    true = T.make_transforms([[0.0, 0.0, 0.0]], [[0.0, 0.0, 0.0, 1.0]])
    scan = sim.simulate(_device(true), attrs=("hits", "points"))
    hyp = np.repeat(true, case["n"], 0)
    hyp[:, 4:7] += rng.normal(scale=0.2, size=(case["n"], 3)).astype(np.float32)
    a = 0.5 * rng.normal(scale=math.radians(2.0), size=case["n"])
    hyp[:, 2], hyp[:, 3] = np.sin(a), np.cos(a)
    hyp = _device(hyp)
    rcc = icp.BatchedRCC(hm, model, scan.points, scan.hits, hyp, n_inner=case["inner"], max_dist=0.5, device=DEV)
    return {"run": _run_rcc, "rcc": rcc, "hyp": hyp}


def _run_rcc(s):
    rcc = s["rcc"]
    rcc.Tbm.copy_(s["hyp"])
    rcc.run(1, graph=True)
    return {"Tbm": rcc.Tbm, "stats": rcc.stats, "system": rcc.grad}


def _register_inputs(case, seed):
    """A scan of a 20 m room per segment: model points on its walls with their normals, the
    dataset the same points moved by a small rigid motion plus noise, a tenth masked out."""
    g = _generator(seed)
    n, count = case["n"], case["n"] * case["seg"]
    m = (torch.rand((count, 3), generator=g, device=DEV) - 0.5) * 20.0
    axis = torch.randint(0, 3, (count, 1), generator=g, device=DEV)
    side = torch.randint(0, 2, (count, 1), generator=g, device=DEV).float() * 2.0 - 1.0
    m.scatter_(1, axis, 10.0 * side)
    nrm = torch.zeros_like(m).scatter_(1, axis, -side)
    d = m + 0.05 + 0.01 * torch.randn((count, 3), generator=g, device=DEV)
    d[:, 0] += 0.02 * m[:, 1]
    d[:, 1] -= 0.02 * m[:, 0]
    pre = torch.randn((n, 8), generator=g, device=DEV) * 0.01
    pre[:, 3], pre[:, 7] = 1.0, 0.0
    pre[:, :4] /= pre[:, :4].norm(dim=1, keepdim=True)
    dmask, mmask = ((torch.rand(count, generator=g, device=DEV) > 0.05).to(torch.uint8) for _ in range(2))
    ids = torch.randint(0, 4, (count,), generator=g, device=DEV, dtype=torch.int32) if case["ids"] else None
    return {"pre": pre.contiguous(), "d": d, "m": m, "nrm": nrm, "dmask": dmask, "mmask": mmask, "ids": ids}


GATE, MODEL_ID = 1.0, 2


def _prepare_register(case, seed):
    i = _register_inputs(case, seed)
    return {"run": _run_register, "stat": rmath.statistics_p2l if case["stat"] == "p2l" else rmath.statistics_p2p,
            "pre": i["pre"], "n": case["n"], "dataset": rmath.PointCloudView(i["d"], mask=i["dmask"]),
            "model": rmath.PointCloudView(i["m"], mask=i["mmask"], normals=i["nrm"], ids=i["ids"]),
            "params": rmath.UmeyamaReductionConstraints(max_dist=GATE, model_id=MODEL_ID if case["ids"] else 0)}


def _run_register(s):
    stats = s["stat"](s["pre"], s["dataset"], s["model"], s["params"], n_segments=s["n"])
    return {"stats": stats, "T": rmath.umeyama_transform(stats)[0]}


NOISE = {"gaussian": (noise.GaussianNoiseHip, (0.0, 0.01)), "rel_gaussian": (noise.RelGaussianNoiseHip, (0.0, 0.002, 1.0)),
         "uniform_dust": (noise.UniformDustNoiseHip, (0.001, 0.5))}
MAX_RANGE = 100.0


def _noise_ranges(case, seed):
    """Ranges of a scan in 0.1-100 m, a tenth of them misses (range.max + 1)."""
    g = _generator(seed)
    r = 0.1 + 99.9 * torch.rand(case["n"], generator=g, device=DEV)
    return torch.where(torch.rand(case["n"], generator=g, device=DEV) < 0.1, torch.full_like(r, MAX_RANGE + 1.0), r)


def _prepare_noise(case, seed):
    cls, prm = NOISE[case["model"]]
    return {"run": _run_noise, "noise": cls(*prm, options=noise.Options(seed=seed, max_range=MAX_RANGE)),
            "ranges": _noise_ranges(case, seed)}


def _run_noise(s):
    return s["noise"].apply(s["ranges"])


def _queries(case, seed):
    """Points near the scene's surfaces (terrain: within 2 m of them), in random order."""
    rng = np.random.default_rng(seed)
    n, info = case["n"], _mesh_of(case)[2]
    if case["scene"] == "terrain":
        x, y, z = _terrain_points(rng, n, info, 1.0)
        q = np.stack([x, y, z + rng.uniform(-2.0, 2.0, n)], 1)
    elif case["scene"] == "objects":
        q = rng.uniform(-100.0, 100.0, size=(n, 3))
    else:
        q = rng.uniform((-10.0, -10.0, 0.0), (10.0, 10.0, 4.0), size=(n, 3))
    return q.astype(np.float32)


def _prepare_closest(case, seed):
    return {"run": _run_closest, "map": _map_of(case), "q": _device(_queries(case, seed)),
            "within": {"max_distance": case["max_distance"]} if case["max_distance"] else {}}


def _run_closest(s):
    return s["map"].closest_points(s["q"], **s["within"])


def _moved(case, seed):
    """The scene's vertices moved by up to 0.2 m along z in slow waves."""
    V = _mesh_of(case)[0].copy()
    p = np.random.default_rng(seed).uniform(0.0, 2.0 * math.pi, 2).astype(np.float32)
    V[:, 2] += 0.1 * (np.sin(0.7 * V[:, 0] + p[0]) + np.cos(0.9 * V[:, 1] + p[1]))
    return V


def _scanner(case, seed, hm):
    model = scenes.ouster_workload_model()
    pose = _poses(case, 1, seed)
    pose[:, 6] += 0.5
    return {"sim": simulation.simulator_for(model, hm, device=DEV), "Tbm": _device(pose), "bundle": _bundle(model, 1, ALL)}


def _prepare_rebuild(case, seed):
    return {"run": _run_rebuild, "V": _moved(case, seed), "F": _mesh_of(case)[1], **_scanner(case, seed, None)}


def _run_rebuild(s):
    s["sim"].setMap(simulation.HipMap(s["V"], s["F"], device=DEV))
    return _run_scan(s)


def _prepare_refit(case, seed):
    hm = _map_of(case)
    return {"run": _run_refit, "map": hm, "V": _device(_moved(case, seed)), **_scanner(case, seed, hm)}


def _run_refit(s):
    s["map"].refit(s["V"])
    return _run_scan(s)


_PREPARE = {"scan": _prepare_scan, "fleet": _prepare_fleet, "particles": _prepare_particles, "rcc": _prepare_rcc,
            "register": _prepare_register, "noise": _prepare_noise, "closest": _prepare_closest,
            "rebuild": _prepare_rebuild, "refit": _prepare_refit}


def run(state):
    return state["run"](state)


# ---- the work a pass cannot do without ----------------------------------------------------------

_ATTR_BYTES = {"hits": 1, "ranges": 4, "points": 12, "normals": 12, "face_ids": 4, "geom_ids": 4, "object_ids": 4}
_RAY_FLOPS = 150  # the ray set-up and one triangle test; how much of the tree it takes depends on the scene


def _scan_work(w, h, poses, attrs, model):
    rays = w * h * poses
    lists = {"o1dn": 12, "ondn": 24}.get(model, 0) * w * h
    return {"bytes": rays * sum(_ATTR_BYTES[a] for a in attrs.split(",")) + lists + 32 * poses, "flops": _RAY_FLOPS * rays}


def work(case):
    """Inputs read once, outputs written once.  Of a map a ray cast has to read no known part:
    it is left out except where it is itself the input (rebuild, refit)."""
    kind = case["kind"]
    if kind == "scan":
        return _scan_work(case["w"], case["h"], case["poses"], case["attrs"], case["model"])
    if kind == "fleet":
        parts = [_scan_work(w, h, case["poses"], "hits,ranges", m) for m, w, h in _fleet_sizes(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    if kind == "particles":
        rays = case["w"] * case["h"]
        return {"bytes": 5 * rays + (32 + 48 + 8 + 48) * case["n"], "flops": (_RAY_FLOPS + 60) * rays * case["n"]}
    if kind == "rcc":
        # the dataset once; per hypothesis its scan stays on the chip in principle
        scan = case["rays"] * case["n"]
        return {"bytes": 25 * case["rays"] + (64 + 128 + 352) * case["n"], "flops": (_RAY_FLOPS + 80 * (case["inner"] + 1)) * scan}
    if kind == "register":
        per = 26 + (12 if case["stat"] == "p2l" else 0) + (4 if case["ids"] else 0)
        return {"bytes": case["n"] * (case["seg"] * per + 192), "flops": 70 * case["n"] * case["seg"]}
    if kind == "noise":
        return {"bytes": 8 * case["n"], "flops": 100 * case["n"]}
    if kind == "closest":
        return {"bytes": 52 * case["n"], "flops": 200 * case["n"]}
    vertices, faces = case["grid"] ** 2, 2 * (case["grid"] - 1) ** 2
    scan = _scan_work(1024, 128, 1, ALL, "sphere")
    # vertices and faces in, triangles, normals and (at most) as many nodes as half the faces out
    return {"bytes": scan["bytes"] + 12 * vertices + (12 if kind == "rebuild" else 0) * faces + (64 + 32) * faces,
            "flops": scan["flops"] + 60 * faces}


# ---- the same results in 64 bits ------------------------------------------------------------------


def exact(case, seed):
    """What run() returns on a state's first pass, in 64-bit torch; None where only a walk of
    the whole map by brute force would tell.  Whole numbers are left out."""
    kind = case["kind"]
    if kind == "scan" and case["scene"] == "room" and case["model"] not in ("o1dn", "ondn"):
        return _exact_scan(case, seed)
    if kind == "particles" and case["scene"] == "room" and case["w"] * case["h"] * case["n"] <= 10_000_000:
        return _exact_particles(case, seed)
    if kind == "register":
        return _exact_register(case, seed)
    if kind == "noise":
        return _exact_noise(case, seed)
    if kind == "closest" and case["scene"] == "room":
        return _exact_closest(case, seed)
    return None


def _rot64(q):
    """(n, 3, 3) rotations of quaternions (x, y, z, w), of q p q* (no normalisation)."""
    x, y, z, w = q.double().unbind(-1)
    r = [w * w + x * x - y * y - z * z, 2 * (x * y - w * z), 2 * (x * z + w * y),
         2 * (x * y + w * z), w * w - x * x + y * y - z * z, 2 * (y * z - w * x),
         2 * (x * z - w * y), 2 * (y * z + w * x), w * w - x * x - y * y + z * z]
    return torch.stack(r, -1).reshape(*q.shape[:-1], 3, 3)


def _dirs64(model):
    """(rays, 3) sensor-frame directions of a spherical or pinhole model."""
    if isinstance(model, T.SphericalModel):
        a = [torch.tensor([np.float32(d.min) + np.float32(i) * np.float32(d.inc) for i in range(d.size)],
                          dtype=torch.float64, device=DEV) for d in (model.phi, model.theta)]
        phi, th = a[0][:, None], a[1][None, :]
        d = (torch.cos(phi) * torch.cos(th), torch.cos(phi) * torch.sin(th), torch.sin(phi).expand(-1, len(a[1])))
        return torch.stack(d, -1).reshape(-1, 3)
    u, v = torch.meshgrid(torch.arange(model.width, dtype=torch.float64, device=DEV),
                          torch.arange(model.height, dtype=torch.float64, device=DEV), indexing="xy")
    d = torch.stack([torch.ones_like(u), -(u - model.c[0]) / model.f[0], -(v - model.c[1]) / model.f[1]], -1)
    return (d / d.norm(dim=-1, keepdim=True)).reshape(-1, 3)


def _triangles64(case):
    V, F, _ = _mesh_of(case)
    return torch.as_tensor(V[F.astype(np.int64)], device=DEV).double()


def _cast64(tri, o, d, far):
    """Closest hit of rays o + t d (one origin) by brute force: t (inf where none within far)
    and the triangle's index."""
    a, b, c = (tri - o).unbind(1)
    edges = [torch.linalg.cross(c, b), torch.linalg.cross(a, c), torch.linalg.cross(b, a)]
    n = torch.linalg.cross(b - a, c - a)
    h = (a * n).sum(1)
    ts, ks = [], []
    for part in d.split(max(1, 40_000_000 // len(tri))):
        u, v, w = (part @ e.T for e in edges)
        inside = ((u >= 0) & (v >= 0) & (w >= 0)) | ((u <= 0) & (v <= 0) & (w <= 0))
        t = h / (part @ n.T)
        t = torch.where(inside & (t >= 0) & (t <= far), t, torch.full_like(t, math.inf))
        t, k = t.min(1)
        ts.append(t)
        ks.append(k)
    return torch.cat(ts), torch.cat(ks)


def _exact_scan(case, seed):
    model = _model(case["model"], case["w"], case["h"], seed)
    tri, d = _triangles64(case), _dirs64(model)
    unit = torch.linalg.cross(tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0])
    unit = unit / unit.norm(dim=1, keepdim=True)
    Tbm = torch.as_tensor(_poses(case, case["poses"], seed), device=DEV)
    out = {"ranges": [], "points": [], "normals": []}
    for R, o in zip(_rot64(Tbm[:, :4]), Tbm[:, 4:7].double()):
        t, k = _cast64(tri, o, d @ R.T, model.range.max)
        hit = torch.isfinite(t)
        n = unit[k] @ R
        n = torch.where((n * d).sum(1, keepdim=True) > 0, -n, n)
        nan = torch.full_like(d, math.nan)
        out["ranges"].append(torch.where(hit, t, torch.full_like(t, model.range.max + 1.0)))
        out["points"].append(torch.where(hit[:, None], d * t[:, None], nan))
        out["normals"].append(torch.where(hit[:, None], n, nan))
    return {k: torch.cat(out[k]) if k in out else None for k in case["attrs"].split(",")}


def _exact_particles(case, seed):
    model, true, T0, xi = _particle_inputs(case, seed)
    tri, d = _triangles64(case), _dirs64(model)
    unit = torch.linalg.cross(tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0])
    unit = unit / unit.norm(dim=1, keepdim=True)
    s = _prepare_particles(case, seed)  # the target scan is an input of the pass
    target, mask = s["target"].double(), s["mask"].bool()
    T0, xi = torch.as_tensor(T0, device=DEV).double(), torch.as_tensor(xi, device=DEV)
    loss, grad, delta = [], [], np.float32(0.05).item()
    for p in range(case["n"]):
        w = xi[p, 3:]
        a = w.norm()
        q1 = torch.cat([w * (torch.sin(0.5 * a) / a), torch.cos(0.5 * a)[None]])
        q0 = T0[p, :4]
        v = q1[3] * q0[:3] + q0[3] * q1[:3] + torch.linalg.cross(q1[:3], q0[:3])
        R = _rot64(torch.cat([v, (q1[3] * q0[3] - q1[:3] @ q0[:3])[None]]))
        o = T0[p, 4:7] + xi[p, :3]
        dm = d @ R.T
        t, k = _cast64(tri, o, dm, model.range.max)
        use = torch.isfinite(t) & (t >= model.range.min) & mask
        t, n, dm = t[use], unit[k[use]], dm[use]
        e = t - target[use]
        rho = torch.where(e.abs() <= delta, 0.5 * e * e, delta * (e.abs() - 0.5 * delta))
        g = -n / (n * dm).sum(1, keepdim=True) * e.clamp(-delta, delta)[:, None]
        local = torch.linalg.cross(t[:, None] * dm, g).sum(0)
        W = torch.tensor([[0.0, -w[2], w[1]], [w[2], 0.0, -w[0]], [-w[1], w[0], 0.0]], dtype=torch.float64, device=DEV)
        J = torch.eye(3, dtype=torch.float64, device=DEV) + (1 - torch.cos(a)) / a ** 2 * W + (a - torch.sin(a)) / a ** 3 * (W @ W)
        loss.append(rho.sum())
        grad.append(torch.cat([g.sum(0), J.T @ local]))
    return {"loss": torch.stack(loss), "grad": torch.stack(grad)}


def _exact_register(case, seed):
    i = _register_inputs(case, seed)
    n, seg = case["n"], case["seg"]
    R, t = _rot64(i["pre"][:, :4]), i["pre"][:, 4:7].double()
    rows, moves = [], []
    for s in range(n):
        at = slice(s * seg, (s + 1) * seg)
        d, m = i["d"][at].double() @ R[s].T + t[s], i["m"][at].double()
        keep = i["dmask"][at].bool() & i["mmask"][at].bool()
        if case["ids"]:
            keep &= i["ids"][at] == MODEL_ID
        if case["stat"] == "p2l":
            nrm = i["nrm"][at].double()
            off = ((m - d) * nrm).sum(1)
            keep &= off.abs() < GATE
            m = d + nrm * off[:, None]
        else:
            keep &= (m - d).norm(dim=1) < GATE
        d, m = d[keep], m[keep]
        if len(d) == 0:
            rows.append(torch.zeros(16, dtype=torch.float64, device=DEV))
            moves.append(torch.tensor([0, 0, 0, 1, 0, 0, 0, 0], dtype=torch.float64, device=DEV))
            continue
        dm, mm = d.mean(0), m.mean(0)
        C = (m - mm).T @ (d - dm) / len(d)
        # the count sits as a 32-bit integer in the last double
        count = torch.tensor([len(d), 0], dtype=torch.int32, device=DEV).view(torch.float64)
        rows.append(torch.cat([dm, mm, C.T.reshape(-1), count]))
        U, _, Vh = torch.linalg.svd(C)
        sign = torch.ones(3, dtype=torch.float64, device=DEV)
        sign[2] = torch.sign(torch.det(U) * torch.det(Vh))
        B = U @ torch.diag(sign) @ Vh
        w = 0.5 * torch.sqrt(1.0 + B.trace())  # small rotations: the trace is near 3
        q = torch.stack([B[2, 1] - B[1, 2], B[0, 2] - B[2, 0], B[1, 0] - B[0, 1]]) / (4.0 * w)
        moves.append(torch.cat([q, w[None], mm - B @ dm, torch.zeros(1, dtype=torch.float64, device=DEV)]))
    return {"stats": torch.stack(rows), "T": torch.stack(moves)}


def _philox(n, words, key):
    """Philox4x32-10 (Salmon et al., SC 2011) of counters (i, 0, words...), i < n, as int64."""
    low = 0xFFFFFFFF
    c = [torch.arange(n, dtype=torch.int64, device=DEV), 0, words[0], words[1]]
    k0, k1 = key

    def halves(m, x):  # 32 x 32 -> 64 bits without passing 2^63
        hi, lo = m >> 16, m & 0xFFFF
        a, b = lo * x, hi * x
        s = (a >> 16) + (b & 0xFFFF)
        return ((b >> 16) + (s >> 16)) & low, ((s << 16) | (a & 0xFFFF)) & low

    for _ in range(10):
        h0, l0 = halves(0xD2511F53, c[0])
        h1, l1 = halves(0xCD9E8D57, c[2])
        c = [h1 ^ c[1] ^ k0, l1, h0 ^ c[3] ^ k1, l0]
        k0, k1 = (k0 + 0x9E3779B9) & low, (k1 + 0xBB67AE85) & low
    return c


def _exact_noise(case, seed):
    kinds = list(NOISE)
    a, b, *c = (float(np.float32(p)) for p in NOISE[case["model"]][1])
    r = _noise_ranges(case, seed).double()
    x, y, z, _ = _philox(case["n"], (0, kinds.index(case["model"])), (seed & 0xFFFFFFFF, 0x5EED))
    if case["model"] == "uniform_dust":
        d = r.clamp(max=MAX_RANGE)
        # the particle's distance is a float before its return probability is taken
        near = ((y >> 8).double() * 2.0 ** -24 * d).float().double()
        seen = ((x >> 8).double() * 2.0 ** -24 < 1.0 - (1.0 - a) ** d) & ((z >> 8).double() * 2.0 ** -24 < b ** near)
        return torch.where(seen, near, r)
    n = torch.sqrt(-2.0 * torch.log(((x >> 8).double() + 1.0) * 2.0 ** -24)) * torch.cos(2.0 * math.pi * ((y >> 8).double() * 2.0 ** -24))
    sd = b * r ** c[0] if c else b
    return torch.where(r <= MAX_RANGE, r + n * sd + a, r)


def _exact_closest(case, seed):
    tri = _triangles64(case)
    q = torch.as_tensor(_queries(case, seed), device=DEV).double()
    far = case["max_distance"] or math.inf
    dist, points = [], []
    corners = tri.unbind(1)
    unit = torch.linalg.cross(corners[1] - corners[0], corners[2] - corners[0])
    unit = unit / unit.norm(dim=1, keepdim=True)
    for p in q.split(max(1, 4_000_000 // len(tri))):
        best, at = torch.full((len(p),), math.inf, dtype=torch.float64, device=DEV), torch.zeros_like(p)
        inside = torch.ones((len(p), len(tri)), dtype=torch.bool, device=DEV)

        def offer(d2, where):
            nonlocal best, at
            least, k = d2.min(1)
            at = torch.where((least < best)[:, None], where(k), at)
            best = torch.minimum(best, least)

        for e in range(3):  # the edges, and on which side of each the point's foot lies
            a, b = corners[e], corners[(e + 1) % 3]
            ab = b - a
            inside &= p @ torch.linalg.cross(unit, ab).T >= (torch.linalg.cross(unit, ab) * a).sum(1)
            s = ((p @ ab.T - (a * ab).sum(1)) / (ab * ab).sum(1)).clamp(0.0, 1.0)
            d2 = sum((p[:, j, None] - a[:, j] - s * ab[:, j]) ** 2 for j in range(3))
            offer(d2, lambda k: a[k] + s.gather(1, k[:, None]) * ab[k])
        off = p @ unit.T - (unit * corners[0]).sum(1)
        offer(torch.where(inside, off * off, torch.full_like(off, math.inf)), lambda k: p - off.gather(1, k[:, None]) * unit[k])
        hit = torch.sqrt(best) < far
        dist.append(torch.where(hit, torch.sqrt(best), torch.full_like(best, torch.finfo(torch.float32).max)))
        points.append(torch.where(hit[:, None], at, torch.full_like(at, math.nan)))
    return {"dist": torch.cat(dist), "points": torch.cat(points), "normals": None, "face_ids": None, "geom_ids": None,
            "object_ids": None}
