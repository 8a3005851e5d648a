"""Workloads of the sensor path as its callers run them, for timing and comparison.

A case names an entry point, a batch size and its options.  Inputs follow the
seeded generator of the tests and the benchmark (csrc/synth.c): standard
normal state values, LiDAR ranges uniform in [0.2, 300) m with 10% no-return,
missions uniform in [-1.5, 1.5) with a boolean arena flag, camera depth uniform
in [0.5, 200) m with 15% far plane.  A `cluttered` scene has a quarter of its
returns within 12 m, as near an obstacle course or the ground.

`exact` restates each entry in 64 bits with plain torch.
"""
import math

import numpy as np
import torch

from turbinator_c_amd import actor, features

OBS, MISSION, CAMERA, FEATURES = 4148, 10, 16384, 142
# Byte offsets of one observation in a replay transition (66,672 bytes).
RECORD, RECORD_OBS, RECORD_MISSION, RECORD_CAMERA = 66672, 0, 16592, 16632
DEVICE = "cuda"


def listed():
    return [
        # One acting step at the trainer's default batch: features, then the
        # compact actor on them, without leaving the device.
        {"name": "step_32", "entry": "step", "n": 32, "hidden": 128, "stochastic": True},
        # The headline: one call over 16,384 resident environments.
        {"name": "features_16384", "entry": "features", "layout": "batch", "n": 16384},
        # A whole replay shard read in place from its transition records.
        {"name": "records_65536", "entry": "features", "layout": "records", "n": 65536},
        # A replay sample: rows picked by index from the field arrays.
        {"name": "sampled_4099", "entry": "features", "layout": "sampled", "n": 4099,
         "capacity": 20000},
        # Cameras as fp32 depth, at the parity configuration's batch.
        {"name": "depth_1024", "entry": "features", "layout": "depth", "n": 1024},
        # The onboard features of a mid-sized rollout.
        {"name": "onboard_1000", "entry": "onboard", "n": 1000, "cluttered": False,
         "diag": False},
        # The onboard features of a large rollout in cluttered scenes.
        {"name": "onboard_39999", "entry": "onboard", "n": 39999, "cluttered": True,
         "diag": False},
        # The large actor's sensor preparation: a few environments acting,
        # and a full training batch.
        {"name": "actor_inputs_64", "entry": "actor_inputs", "n": 64, "cluttered": False},
        {"name": "actor_inputs_16384", "entry": "actor_inputs", "n": 16384, "cluttered": False},
        # The compact actor on a full batch of feature rows, sampling actions.
        {"name": "act_16384", "entry": "act", "n": 16384, "hidden": 128, "stochastic": True},
        # One step of a learner: its new weights packed, then acted with.
        {"name": "refresh_256", "entry": "refresh", "n": 256, "hidden": 256, "stochastic": True},
        # The trainer's host call: 32 environments in pageable host memory.
        {"name": "host_32", "entry": "host", "how": "object", "n": 32},
    ]


def _log_size(rng, least, most):
    return min(most, int(math.exp(rng.uniform(math.log(least), math.log(most + 1)))))


def draw(rng):
    entry = rng.choice(["features", "features", "step", "onboard", "actor_inputs", "act",
                        "refresh", "host"])
    if entry == "features":
        layout = rng.choice(["batch", "records", "sampled", "depth", "diagnostics", "blind"])
        n = _log_size(rng, 512, 16384)
        case = {"entry": entry, "layout": layout, "n": n}
        if layout == "sampled":
            case["capacity"] = rng.randint(n, 32768)
        return case
    if entry == "onboard":
        return {"entry": entry, "n": _log_size(rng, 1, 65536), "cluttered": rng.random() < 0.5,
                "diag": rng.random() < 0.25}
    if entry == "actor_inputs":
        return {"entry": entry, "n": _log_size(rng, 1, 16000), "cluttered": rng.random() < 0.5}
    if entry == "host":
        return {"entry": entry, "how": rng.choice(["object", "copied", "direct"]),
                "n": rng.randint(1, 256)}
    least, most = (1024, 65536) if entry == "act" else (1, 4096)
    return {"entry": entry, "n": _log_size(rng, least, most), "hidden": rng.randint(16, 256),
            "stochastic": rng.random() < 0.5}


# --------------------------------------------------------------------------
# Inputs


def _fill(g, n, obs, mission, cameras=None, depth=None, cluttered=False):
    """Writes n environments into the given views, a block at a time."""
    for i in range(0, n, 8192):
        k = min(8192, n - i)

        def uniform(lo, hi, *shape):
            return torch.empty(shape, device=DEVICE).uniform_(lo, hi, generator=g)

        row = torch.randn((k, OBS), device=DEVICE, generator=g)
        lidar = uniform(0.2, 300.0, k, 4096)
        pick = uniform(0.0, 1.0, k, 4096)
        if cluttered:
            lidar = torch.where(pick > 0.75, 0.2 + lidar * (11.8 / 300.0), lidar)
        row[:, 48:4144] = torch.where(pick < 0.1, -1.0, lidar)
        obs[i:i + k] = row
        m = uniform(-1.5, 1.5, k, MISSION)
        m[:, 6] = (uniform(0.0, 1.0, k) < 0.125).float()
        mission[i:i + k] = m
        if cameras is not None or depth is not None:
            far = uniform(0.0, 1.0, k, CAMERA) < 0.15
            d = torch.where(far, 200.0, uniform(0.5, 200.0, k, CAMERA))
            if depth is not None:
                depth[i:i + k] = d
            if cameras is not None:
                cameras[i:i + k] = torch.round(255.0 * (1.0 - d / 200.0)).to(torch.uint8)


def _generator(seed):
    return torch.Generator(DEVICE).manual_seed(seed)


def _float(*shape):
    return torch.empty(shape, dtype=torch.float32, device=DEVICE)


def _sensors(case, seed):
    n, layout = case["n"], case.get("layout", "batch")
    g = _generator(seed)
    rows = case.get("capacity", n)
    s = {"n": n, "stream": torch.cuda.current_stream()}
    if layout == "records":
        s["records"] = torch.zeros((n, RECORD), dtype=torch.uint8, device=DEVICE)
        words = s["records"].view(torch.float32)
        s["obs"] = words[:, RECORD_OBS // 4:RECORD_OBS // 4 + OBS]
        s["mission"] = words[:, RECORD_MISSION // 4:RECORD_MISSION // 4 + MISSION]
        s["cameras"] = s["records"][:, RECORD_CAMERA:RECORD_CAMERA + CAMERA]
    else:
        s["obs"], s["mission"] = _float(rows, OBS), _float(rows, MISSION)
        if case["entry"] != "onboard" and layout not in ("depth", "blind"):
            s["cameras"] = torch.empty((rows, CAMERA), dtype=torch.uint8, device=DEVICE)
        if layout == "depth":
            s["depth"] = _float(rows, CAMERA)
    _fill(g, rows, s["obs"], s["mission"], s.get("cameras"), s.get("depth"),
          case.get("cluttered", False))
    if layout == "sampled":
        s["indices"] = torch.randint(0, rows, (n,), device=DEVICE, generator=g).to(torch.int32)
        s["capacity"] = rows
    return s


def _policy(case, seed):
    """Feature-like rows, Glorot-uniform weights and normal draws."""
    n, hidden, g = case["n"], case["hidden"], _generator(seed + 1)
    s = {"n": n, "hidden": hidden, "stream": torch.cuda.current_stream()}
    if case["entry"] == "step":
        s.update(_sensors(case, seed))
    x = torch.randn((n, FEATURES), device=DEVICE, generator=g).mul_(0.5).clamp_(-1.0, 1.0)
    x[:, 62:] = _float(n, FEATURES - 62).uniform_(0.3, 0.7, generator=g)
    s["features"] = x
    s["normals"] = (torch.randn((n, actor.ACTIONS), device=DEVICE, generator=g)
                    if case["stochastic"] else None)
    s["weights"] = []
    for (rows, cols), bias in actor.layer_shapes(hidden):
        limit = math.sqrt(6.0 / (rows + cols))
        s["weights"].append(_float(rows, cols).uniform_(-limit, limit, generator=g))
        s["weights"].append(_float(bias).uniform_(-0.1, 0.1, generator=g))
    return s


class _Host:
    """The host object or pipeline a program keeps between its calls."""

    def __init__(self, how, n):
        self.batch = features.FeatureBatch.create(0, n) if how == "object" else None
        self.pipeline = None if how == "object" else features.FeaturePipeline.create(0, n, 1)

    def __del__(self):
        for h in (self.batch, self.pipeline):
            if h is not None:
                h.destroy()


def prepare(case, seed):
    entry, n = case["entry"], case["n"]
    if entry in ("act", "refresh", "step"):
        s = _policy(case, seed)
        s["packed"] = torch.empty(actor.packed_bytes(case["hidden"]), dtype=torch.uint8,
                                  device=DEVICE)
        if entry != "refresh" and _pack(s) != 1:
            raise RuntimeError("pack_device")
        s["actions"], s["log_prob"] = _float(n, actor.ACTIONS), _float(n)
        s["raw"] = _float(n, actor.RAW)
    else:
        s = _sensors(case, seed)
    s["case"] = case
    if entry == "features":
        s["features"] = _float(n, FEATURES)
        if case["layout"] == "diagnostics":
            s["diag"] = torch.empty((n, 432), dtype=torch.uint8, device=DEVICE)
    elif entry in ("onboard", "actor_inputs"):
        s["tactical"], s["prior"] = _float(n, 24), _float(n, 15)
        s["diag"] = _float(n, 5) if case.get("diag") else None
        if entry == "actor_inputs":
            s["proprio"], s["mission_vec"] = _float(n, 91), _float(n, 49)
            s["lidar"], s["luma"] = _float(n, 6, 16, 128), _float(n, 4, 64, 64)
    elif entry == "host":
        s["host"] = _Host(case["how"], n)
        arrays = [s.pop(k).cpu().numpy() for k in ("obs", "mission", "cameras")]
        s["out"] = np.empty((n, FEATURES), np.float32)
        if case["how"] == "object":
            s["arrays"] = arrays
        else:  # the producer writes its observations into the pinned slot
            for to, what in zip(s["host"].pipeline.inputs(0), arrays):
                to[...] = what
    return s


# --------------------------------------------------------------------------
# One pass


def _pack(s):
    return actor.pack_device(*s["weights"], s["hidden"], s["packed"], s["stream"])


def _act(s):
    return actor.act_device(s["packed"], s["hidden"], s["features"], s["normals"], s["actions"],
                            s["log_prob"], s["raw"], s["n"], s["stream"])


def _features(s):
    layout, n, stream = s["case"]["layout"], s["n"], s["stream"]
    obs, mission, out = s["obs"], s["mission"], s["features"]
    if layout in ("batch", "blind"):
        return features.extract_features_device(obs, mission, s.get("cameras"), out, n, stream)
    if layout == "records":
        return features.extract_features_strided_device(obs, RECORD, mission, RECORD,
                                                        s["cameras"], RECORD, out, n, stream)
    if layout == "sampled":
        return features.extract_features_indexed_device(
            obs, OBS * 4, mission, MISSION * 4, s["cameras"], CAMERA, s["capacity"],
            s["indices"], out, n, stream)
    if layout == "depth":
        return features.extract_features_depth_device(obs, mission, s["depth"], out, n, stream)
    return features.extract_features_diagnostics_device(obs, mission, s["cameras"], out,
                                                        s["diag"], n, stream)


def _host_pass(s):
    n, host, how = s["n"], s["host"], s["case"]["how"]
    if how == "object":
        return host.batch.extract_host(*s["arrays"], n, s["out"]), s["out"]
    submit = host.pipeline.submit if how == "copied" else host.pipeline.submit_direct
    ok = submit(0, n)
    np.copyto(s["out"], host.pipeline.wait(0, n))  # the slot's rows last until its next submit
    return ok, s["out"]


def run(s):
    entry = s["case"]["entry"]
    if entry == "features":
        ok = _features(s)
        out = {"features": s["features"]}
        if "diag" in s:
            out["diag"] = s["diag"]
    elif entry == "onboard":
        ok = features.onboard_tactical_prior_device(s["obs"], s["mission"], s["tactical"],
                                                    s["prior"], s["diag"], s["n"], s["stream"])
        out = {k: s[k] for k in ("tactical", "prior", "diag") if s[k] is not None}
    elif entry == "actor_inputs":
        ok = features.actor_inputs_device(
            s["obs"], s["mission"], s["cameras"], s["proprio"], s["mission_vec"], s["tactical"],
            s["prior"], s["lidar"], s["luma"], s["n"], s["stream"])
        out = {k: s[k] for k in ("proprio", "mission_vec", "tactical", "prior", "lidar", "luma")}
    elif entry == "host":
        ok, out = _host_pass(s)
    else:
        ok = 1
        if entry == "refresh":
            ok = _pack(s)
        elif entry == "step":
            ok = features.extract_features_device(s["obs"], s["mission"], s["cameras"],
                                                  s["features"], s["n"], s["stream"])
        ok = ok == 1 and _act(s)
        out = {k: s[k] for k in ("actions", "log_prob", "raw")}
        if entry == "step":
            out["features"] = s["features"]
    if ok != 1:
        raise RuntimeError(f"{entry}: not accepted")
    return out


# --------------------------------------------------------------------------
# What a pass cannot do without, and how far two correct results may lie apart


def work(case):
    n, entry = case["n"], case["entry"]
    if entry in ("features", "host"):
        layout = case.get("layout", "batch")
        camera = {"depth": 4 * CAMERA, "blind": 0}.get(layout, CAMERA)
        extra = {"diagnostics": 432, "sampled": 4}.get(layout, 0)
        return {"bytes": n * (4 * (OBS + MISSION + FEATURES) + camera + extra),
                "flops": n * (4096 * 17 + CAMERA)}
    if entry == "onboard":
        # 48 state values, the mission, the outputs, and the scan rays that
        # the missions use: all 1,536 for slalom (14.6% of the missions) or
        # with the diagnostics row, 1,024 for dodge (25%).
        rays = 1536.0 if case["diag"] else 0.146 * 1536 + 0.25 * 1024
        return {"bytes": n * (4 * (48 + MISSION + 24 + 15 + (5 if case["diag"] else 0)) +
                              4 * rays), "flops": n * 2000}
    if entry == "actor_inputs":
        return {"bytes": n * (4 * (OBS + MISSION + 91 + 49 + 24 + 15 + 12288 + CAMERA) + CAMERA),
                "flops": n * (12288 * 4 + 2 * CAMERA)}
    h = case["hidden"]
    weights = FEATURES * h + h * h + 30 * h + 2 * h + 30
    row = FEATURES + actor.ACTIONS + 1 + actor.RAW + (actor.ACTIONS if case["stochastic"] else 0)
    moved, flops = 4 * (n * row + weights), 2 * n * weights
    if entry == "step":
        moved += n * (4 * (OBS + MISSION) + CAMERA)
        flops += n * (4096 * 17 + CAMERA)
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    entry = case["entry"]
    if entry in ("features", "host"):
        # fp32 sums of 64 log1p values; the camera sums are whole numbers.
        return {"rel": 1e-6, "max": 1e-5}
    if entry in ("onboard", "actor_inputs"):
        # The controller's angles in fp32 behind clamps and gains of up to
        # 130; decisions are the same in every correct implementation.
        return {"rel": 5e-5, "max": 2e-2}
    # Three dense layers in fp32; log-probabilities of near-saturated
    # actions magnify the rounding of 1 - action^2.
    return {"rel": 2e-6, "max": 2e-3}


# --------------------------------------------------------------------------
# 64-bit restatements

_PI = math.pi


def _finite(x):
    return torch.where(torch.isfinite(x), x, 0.0)


def _exact_features(s, layout):
    obs, mission = s["obs"].double(), s["mission"].double()
    scale = torch.ones(48, dtype=torch.float64, device=DEVICE)
    scale[0:2], scale[2], scale[3:6], scale[10:13], scale[13:16] = 300, 100, 50, 5, 30
    scale[28:32], scale[32:40], scale[44:46] = _PI / 4, 5, _PI / 2
    state = (_finite(obs[:, :48]) / scale).clamp(-1, 1)
    quality = _finite(obs[:, 4144:]).clamp(0, 1)
    arena = mission[:, 6:7] > 0.5
    m = mission.clone()
    m[:, 7:] = torch.where(arena, 0.0, m[:, 7:])
    r = obs[:, 48:4144]
    bins = torch.log1p(r.clamp(0, 120)) / math.log1p(120.0)
    bins = torch.where(torch.isfinite(r) & (r >= 0), bins, -1.0)
    sectors = bins.view(-1, 2, 4, 4, 8, 16).mean(dim=(3, 5)).reshape(-1, 64)
    if layout == "blind":
        quads = torch.zeros((len(obs), 16), dtype=torch.float64, device=DEVICE)
    else:
        if layout == "depth":
            luma = torch.round(255.0 * (1.0 - s["depth"].double().clamp(0, 200) / 200.0))
        else:
            luma = s["cameras"].double()
        quads = luma.reshape(-1, 4, 2, 32, 2, 32).mean(dim=(3, 5)).reshape(-1, 16) / 255.0
    return torch.cat([state, quality, m.clamp(-1, 1), sectors, quads], dim=1)


def _atanh20(x, limit):
    return torch.atanh(x.clamp(-limit, limit)) * 20.0


def _norm(*v):
    return torch.sqrt(sum(x * x for x in v))


def _unrotate(qw, qx, qy, qz, v):
    """v in the body frame of the attitude quaternion."""
    ux, uy, uz = -qx, -qy, -qz
    cx, cy, cz = (uy * v[2] - uz * v[1] + qw * v[0], uz * v[0] - ux * v[2] + qw * v[1],
                  ux * v[1] - uy * v[0] + qw * v[2])
    return (v[0] + 2 * (uy * cz - uz * cy), v[1] + 2 * (uz * cx - ux * cz),
            v[2] + 2 * (ux * cy - uy * cx))


def _exact_tactical(o, m):
    o = [o[:, i] for i in range(48)]
    m = [m[:, i] for i in range(MISSION)]
    spool = [o[16 + i].clamp(0, 1) for i in range(4)]
    thrust = [0.036 + 0.964 * x for x in spool]
    fz = [thrust[i] * o[24 + i] * torch.cos(o[28 + i]) for i in range(4)]
    tz = [thrust[i] * o[20 + i] * torch.cos(o[28 + i]) for i in range(4)]
    mean = sum(spool) * 0.25
    qw, qx, qy, qz = o[6], o[7], o[8], o[9]
    bz_x, bz_y = 2 * (qx * qz + qw * qy), 2 * (qy * qz - qw * qx)
    ct = (1 - 2 * (qx * qx + qy * qy)).clamp(-1, 1)
    rx, ry, rz = (_atanh20(m[7 + i], 0.995) for i in range(3))
    yaw = torch.atan2(2 * (qx * qy + qw * qz), 1 - 2 * (qy * qy + qz * qz))
    cy, sy = torch.cos(yaw), torch.sin(yaw)
    dist = _norm(rx, ry, rz).clamp(min=1.0)
    flight = dist / 20.0
    w = (rx - o[3] * 0.5 * flight, ry - o[4] * 0.5 * flight,
         rz - o[5] * 0.5 * flight + 0.5 * 9.80665 * flight * flight)
    bx, by, bz = _unrotate(qw, qx, qy, qz, w)
    az = torch.atan2(by, bx).clamp(_PI / 12, _PI * 5 / 12)
    el = torch.atan2(bz, torch.hypot(bx, by).clamp(min=0.2)).clamp(-_PI / 6, _PI / 6)
    err = torch.hypot(az - o[44], el - o[45])
    ready = (o[46] <= 0.02) & (o[47] > 0.01) & (err < 0.26) & (dist < 34.0)
    return torch.stack([
        fz[1] - fz[3], fz[2] - fz[0], 0.5 * sum(tz), 0.25 * sum(fz) - 0.5,
        *[2 * (x - mean) for x in spool],
        cy * bz_y - sy * bz_x, -sy * bz_y - cy * bz_x, ct, (ct < 0.20).double(),
        torch.tanh((cy * rx + sy * ry) * 0.08), torch.tanh((-sy * rx + cy * ry) * 0.08),
        torch.tanh(rz * 0.12), torch.tanh(torch.hypot(rx, ry) * 0.05),
        torch.tanh((cy * o[3] + sy * o[4]) * 0.15), torch.tanh((-sy * o[3] + cy * o[4]) * 0.15),
        torch.exp(-(o[2] - 0.62).clamp(min=0)), (az - _PI * 0.25) / (_PI / 6), el / (_PI / 6),
        torch.tanh(err * 2.0), torch.where(ready, 1.0, -1.0).double(),
        torch.sin(torch.atan2(ry, rx) - _PI * 0.25 - yaw)], dim=1)


def _rays():
    head = torch.arange(2, dtype=torch.float64, device=DEVICE).view(2, 1, 1)
    el = torch.arange(6, dtype=torch.float64, device=DEVICE).view(1, 6, 1)
    azi = torch.arange(128, dtype=torch.float64, device=DEVICE).view(1, 1, 128)
    elev, azim = (1 - 2 * head) * (_PI * el / 30), _PI * (0.25 + azi / 64)
    d = torch.stack(torch.broadcast_tensors(torch.cos(elev) * torch.cos(azim),
                                            torch.cos(elev) * torch.sin(azim), torch.sin(elev)),
                    dim=-1)
    return d.reshape(1536, 3)


def _exact_scan(lidar, rot, py):
    """Closest return (range, world offset), corridor minimum, cluster."""
    n = len(lidar)
    ranges = lidar.view(n, 2, 16, 128)[:, :, :6].reshape(n, 1536)
    world = torch.einsum("nij,rj->nir", rot, _rays())
    window = (ranges > 0.35) & (ranges < 11.5)
    low = (torch.arange(1536, device=DEVICE) // 128) % 6 < 4
    near = torch.where(window & low, ranges, math.inf)
    min_r, ray = near.min(dim=1)
    found = torch.isfinite(min_r)
    at = world.gather(2, ray.view(n, 1, 1).expand(n, 3, 1))[:, :, 0]
    offset = torch.where(found[:, None], at * torch.where(found, min_r, 0.0)[:, None], 0.0)
    min_r = torch.where(found, min_r, 30.0)
    x = world[:, 0] * ranges + world[:, 0] * 1.10
    y = py[:, None] + world[:, 1] * ranges + world[:, 1] * 1.10
    z = world[:, 2] * ranges
    corridor = window & (z.abs() <= 2.1) & (x >= -0.35) & (x <= 10.5) & (y.abs() <= 3.5)
    centre = torch.where(corridor, x, math.inf)
    min_dx = centre.min(dim=1).values.clamp(max=30.0)
    member = centre <= min_dx[:, None] + 1.4
    return (min_r, offset[:, 0], offset[:, 1], min_dx, member.sum(dim=1),
            torch.where(member, y, 0.0).sum(dim=1), torch.where(found, ray, -1))


def _wrap(target, current):
    return torch.atan2(torch.sin(target - current), torch.cos(target - current))


def _exact_prior(obs, mission):
    """The 15 physics-prior features and the 5 scan diagnostics."""
    o = [obs[:, i] for i in range(48)]
    m = [mission[:, i] for i in range(MISSION)]
    where, hyp, at2 = torch.where, torch.hypot, torch.atan2

    def num(cond, a, b):  # where() of numbers, in 64 bits
        a, b = (v if isinstance(v, torch.Tensor) else
                torch.tensor(float(v), dtype=torch.float64, device=DEVICE) for v in (a, b))
        return where(cond, a, b)

    def clip(x, lo, hi):
        lo, hi = (v if isinstance(v, torch.Tensor) else torch.full_like(x, v) for v in (lo, hi))
        return torch.minimum(hi, torch.maximum(lo, x))

    full, g = 294.2 * 0.85, 9.80665
    px, py, pz, vx, vy, vz = o[:6]
    qn = _norm(*o[6:10]).clamp(min=1e-8)
    sign = num(o[6] < 0, -1, 1)
    qw, qx, qy, qz = (sign * q / qn for q in o[6:10])
    ux, uy, uz = -qx, -qy, -qz
    rot = torch.stack([
        1 - 2 * (qy * qy + qz * qz), 2 * (qx * qy - qw * qz), 2 * (qx * qz + qw * qy),
        2 * (qx * qy + qw * qz), 1 - 2 * (qx * qx + qz * qz), 2 * (qy * qz - qw * qx),
        2 * (qx * qz - qw * qy), 2 * (qy * qz + qw * qx), 1 - 2 * (qx * qx + qy * qy)],
        dim=1).view(-1, 3, 3)
    r = [[rot[:, i, j] for j in range(3)] for i in range(3)]
    ox, oy, oz = o[10:13]
    spool = [o[16 + i].clamp(0, 1) for i in range(4)]
    thrust = [full * (0.08 + 0.92 * x) for x in spool]
    outer = [at2(o[20 + i], o[24 + i]) for i in range(4)]
    inner = [torch.cos(o[28 + i]) for i in range(4)]
    fz = [thrust[i] * torch.cos(outer[i]) * inner[i] for i in range(4)]
    ft = [thrust[i] * torch.sin(outer[i]) * inner[i] for i in range(4)]

    landing, cargo = m[1] > 0.75, m[2] > 0.75
    inversion, turbine_out = (m[3] > 0.75) & (m[0] < -0.25), (m[3] > 0.75) & (m[2] < -0.25)
    lateral = (m[4] > 0.75) & (m[5] > 0.25)
    slalom, dodge, arena = (m[4] > 0.75) & ~lateral, m[5] > 0.75, m[6] > 0.75
    bwb_arena, bwb_cruise = arena & (m[4] < -0.25), (m[4] > 0.75) & (m[2] > 0.25)
    endurance = bwb_cruise & (m[0] > 0.25)
    bwb = bwb_arena | bwb_cruise | (arena & (m[5] > 0.60))
    payload = o[41] > 0.5
    mass = (num(arena, 40, 43) + o[40].clamp(0, 1) * 9 + o[47].clamp(0, 4) * 6 +
            num(payload, 30, 0))
    weight = mass * g
    bz_x, bz_y = 2 * (qx * qz + qw * qy), 2 * (qy * qz - qw * qx)
    ct = r[2][2].clamp(-1, 1)
    az_actual = (sum(fz) * ct - weight) / mass
    heavy = cargo & payload

    relx, rely, relz = (_atanh20(m[7 + i], 0.9995) for i in range(3))
    chase = arena | lateral
    tx = num(slalom, 36, num(cargo, 15, num(chase, px + relx, 0)))
    ty = num(chase, py + rely, 0)
    tz = num(cargo | arena, pz + relz, num(inversion, 14, num(landing, 0.6, 8)))
    dxy = hyp(tx - px, ty - py)
    valid = dxy > 1e-3
    safe = num(valid, dxy, 1)
    gap = num(arena & (m[0] > 0.75) & (m[5] < -0.25), 8.5, 12.5)
    ax, ay = (num(valid, t - (t - p) / safe * gap, t) for t, p in ((tx, px), (ty, py)))
    shrink = (16 / hyp(ax, ay).clamp(min=1e-3)).clamp(max=1.0)
    shrink = shrink * (1 - ((hyp(px, py) - 21) / 10).clamp(0, 1))
    az_t = num((pz < 8) | (vz < -1), 12.2, tz.clamp(8.5, 12.2))
    ex, ey, ez = num(arena, ax * shrink, tx), num(arena, ay * shrink, ty), num(arena, az_t, tz)
    horiz = hyp(ex - px, ey - py)

    to = (tx - px, ty - py, tz - pz)
    dist = _norm(*to).clamp(min=1.0)
    flight = dist / 20
    lead = 0.65 * flight
    aim = _unrotate(qw, qx, qy, qz, (to[0] - vx * lead, to[1] - vy * lead,
                                     to[2] - vz * lead + 0.53 * g * flight * flight))
    yaw, roll = at2(r[1][0], r[0][0]), at2(r[2][1], r[2][2])
    can_az = at2(aim[1], aim[0]).clamp(_PI / 12, _PI * 5 / 12)
    can_el = at2(aim[2], hyp(aim[0], aim[1]).clamp(min=0.2)).clamp(-_PI / 6, _PI / 6)

    scan = []
    for i in range(0, len(obs), 2048):
        part = slice(i, i + 2048)
        scan.append(_exact_scan(obs[part, 48:4144], rot[part], py[part]))
    min_r, off_x, off_y, min_dx, count, y_sum, ray = (torch.cat(v) for v in zip(*scan))
    min_az = at2(off_y, off_x)
    avoid = dodge & (min_r < 7.5)
    avoid_x, avoid_y = num(avoid, -2.2 * torch.sin(min_az), 0), num(avoid, 2.2 * torch.cos(min_az), 0)
    seen = slalom & (horiz > 2.5) & (min_dx < 10.2) & (count > 0)
    ey = num(seen, num(y_sum >= 0, -1.85, 1.85), ey)
    lane = (py - ey).abs()
    limit = num(lane > 1.05, 1.55, num(lane > 0.55, 2.75, 4.10))
    limit = num((min_dx >= 6.6) & (px > 4), 3.10, limit)
    slalom_speed = num(seen, limit, 3.8)
    hill = ((px - 6) / 30).clamp(0, 1)
    ez = num(slalom & (horiz > 3.5), 2.5 * torch.sin(_PI * hill) + 8, ez)
    upx, upy, upz = ex - px, ey - py, ez - pz
    up_h = hyp(upx, upy)
    active = slalom & (num(seen, min_dx, 30) < 10.2) & (horiz > 3)

    pad = ez.clamp(min=0.6)
    above, speed = pz - pad, hyp(vx, vy)
    cap = num(up_h > 1.8, num(heavy, 2.65, 3.4), num(above < 1.2, 0.55, num(heavy, 1.25, 1.6)))
    kp = num(heavy, 0.75, 1.05)
    low = num(cargo, (1.6 * (0.64 - pz)).clamp(-0.30, 0.18), num(pz > 0.635, -0.16, 0))
    mid = clip(-0.70 * above, num(cargo, -0.82, -1.4), -0.25)
    trans_z = num(heavy, (1.2 + 0.28 * up_h).clamp(min=2.0), 2.0)
    vz_land = num(above > 1.05, mid, low)
    vz_land = num(((up_h > 0.85) | (speed > 0.65)) & (above < 0.95),
                  (1.2 * (pad + 0.90 - pz)).clamp(-0.30, 0.60), vz_land)
    vz_land = num(up_h > 1.8, clip(1.3 * (trans_z - pz), num(heavy, -1.05, -1.6), 1.4), vz_land)
    most = num(heavy, 2.2, 2.6)
    ax_land = clip(2.4 * (clip(kp * upx, -cap, cap) - vx), -most, most)
    ay_land = clip(2.4 * (clip(kp * upy, -cap, cap) - vy), -most, most)
    az_land = clip(num(heavy, 5.0, 4.5) * (vz_land - vz) - num(heavy, 1.0, 0.8) * az_actual,
                   num(heavy, -1.8, -2.8), 5.5)

    fast = (up_h > 9) & (upz.abs() < 2.5) & (ct > 0.9)
    max_vx = num(inversion, num(fast, 6.2, 4.2), num(arena, 3.2, 3.0))
    max_vy = num(lateral, 3.4, max_vx)
    max_vx = num(lateral, num(upy.abs() > 1.35, 1.45, 3.8), max_vx)
    max_vx = num(active, slalom_speed, num(slalom, 3.5, max_vx))
    max_vy = num(active, 3.2, max_vy)
    kp_xy = num(inversion, 0.85, num(lateral, 0.95, 0.90))
    des_vx = clip(num(active, 1.25, kp_xy) * upx + avoid_x, -max_vx, max_vx)
    des_vy = clip(num(active, 1.45, num(lateral, 1.05, kp_xy)) * upy + avoid_y, -max_vy, max_vy)
    des_vz = clip(1.25 * upz, -2.6, num((vz < -2) | inversion, 6.5, 2.6))
    des_vz = num((inversion | arena) & (vz < -1), des_vz.clamp(min=0.8), des_vz)
    like = landing | heavy
    des_ax = num(like, ax_land, (num(active, 3.0, 2.4) * (des_vx - vx)).clamp(-3.8, 3.8))
    des_ay = num(like, ay_land, (num(active, 3.0, 2.6) * (des_vy - vy)).clamp(-3.8, 3.8))
    des_az = num(like, az_land, clip(3.8 * (des_vz - vz) - 0.8 * az_actual, -4.0,
                                     num((vz < -1.8) | inversion, 14.0, 6.5)))

    tilt = torch.acos(ct)
    headroom = inversion | arena | (ct < 0.88)
    urgent = arena & ((pz < 8.5) | (vz < -1.2)) & (ct > 0.58)
    room = (3.95 - 0.9 * _norm(ox, oy, oz) - 1.3 * tilt).clamp(2.55, 3.95)
    coll = num(headroom & ~urgent, room, 3.95)
    fz_des = clip((weight + mass * des_az) / ct.clamp(min=0.45), 0.10 * weight, coll * full)
    h_scale = num(headroom, (1 - 1.5 * (tilt - 0.15).clamp(min=0)).clamp(0, 1), 1)
    h_scale = num(urgent, 0, h_scale)
    comp, damp = num(turbine_out, 0.65, 0), num(active, 0.8, 0.4)
    fx_w = (mass * des_ax + damp * vx - comp * sum(fz) * bz_x) * h_scale
    fy_w = (mass * des_ay + damp * vy - comp * sum(fz) * bz_y) * h_scale
    max_fh = num(active, 105, num(lateral, 125, num(heavy, 52, 80)))
    cyaw, syaw = torch.cos(yaw), torch.sin(yaw)
    fx = clip(cyaw * fx_w + syaw * fy_w, -max_fh, max_fh)
    fy = clip(-syaw * fx_w + cyaw * fy_w, -max_fh, max_fh)

    cw_x, cw_y = bz_y, -bz_x
    t_x, t_y, t_z = 2 * (-uz * cw_y), 2 * (uz * cw_x), 2 * (ux * cw_y - uy * cw_x)
    te_x = cw_x + qw * t_x + (uy * t_z - uz * t_y)
    te_y = cw_y + qw * t_y + (uz * t_x - ux * t_z)
    te_z = qw * t_z + (ux * t_y - uy * t_x)
    te_n = _norm(te_x, te_y, te_z)
    t_scale = num(te_n > 1e-5, tilt / te_n.clamp(min=1e-5), 0)
    e_rx, e_ry = te_x * t_scale, te_y * t_scale
    hold = (inversion | arena) & ((pz < 6) | (vz < -0.5) | (ct < 0.88))
    bearing = num(arena & (m[1].abs() + m[2].abs() > 0.1), at2(m[1], m[2]), at2(ty - py, tx - px))
    des_yaw = num(arena & (horiz > 1) & ~hold, bearing - _PI / 4, num(hold, yaw, 0))

    # Fixed-wing (BWB) geometry and law.
    vb_x = r[0][0] * vx + r[1][0] * vy + r[2][0] * vz
    vb_y = r[0][1] * vx + r[1][1] * vy + r[2][1] * vz
    brx, bry, brz = (_atanh20(m[7 + i], 0.9999) for i in range(3))
    rxy = hyp(px, py)
    pull = num(arena & (rxy > 235), ((rxy - 235) / 45).clamp(0, 0.85), 0)
    btx, bty = (px + brx) * (1 - pull), (py + bry) * (1 - pull)
    btz = num(arena, (pz + brz).clamp(28, 135), pz + brz)
    gx, gy, gz = btx - px, bty - py, btz - pz
    gdist, gs = _norm(gx, gy, gz).clamp(min=1.0), hyp(vx, vy)
    course = num(gs > 2.5, at2(vy, vx), yaw)
    climb = (0.42 * gz).clamp(-5, 5)
    opp = (brx - vx * 0.10, bry - vy * 0.10, brz - vz * 0.10)
    bdist = _norm(*opp).clamp(min=1.0)
    head_on = bwb_arena & (btx * px + bty * py < -800) & (bdist > 45)
    bfl = bdist / num(head_on, 75 + 2 * vb_x.clamp(min=0), 75)
    baz = opp[2] + num(head_on, -vz * (0.85 * bfl), 0) + 0.5 * g * bfl * bfl
    bb = [r[0][k] * opp[0] + r[1][k] * opp[1] + r[2][k] * baz for k in range(3)]
    b_az = at2(bb[1], bb[0].clamp(min=0.2)).clamp(-_PI / 6, _PI / 6)
    b_el = at2(bb[2], hyp(bb[0], bb[1]).clamp(min=0.2)).clamp(
        -_PI / 6, _PI / 6)
    gamma = at2(climb, gs.clamp(min=14.0))

    yaw_err, can_err = _wrap(des_yaw, yaw), _wrap(can_az, o[44])
    course_err, b_can_err = _wrap(at2(gy, gx), course), _wrap(b_az, o[44])
    par = num(turbine_out, 0.35, 1)
    tx_par, ty_par = -0.1625 * fy * par, 0.1625 * fx * par
    max_t = num(heavy, 120, 260)
    tau_x = clip(95 * e_rx - 64 * ox - 0.9 * (fz[1] - fz[3] + tx_par) - tx_par, -max_t, max_t)
    tau_y = clip(95 * e_ry - 64 * oy - 0.9 * (fz[2] - fz[0] + ty_par) - ty_par, -max_t, max_t)
    tau_z = (22 * yaw_err - 18 * oz).clamp(-70, 70)
    fz_cmd = [0.25 * fz_des + 0.5 * t for t in (-tau_y, tau_x, tau_y, -tau_x)]
    yaw_ft = (tau_z - 0.4 * sum(ft)) * 0.25
    fx_rem, fy_rem = fx - (ft[3] - ft[1]), fy - (ft[0] - ft[2])
    max_sin = num(lateral, 0.44, num(active, 0.42, num(heavy, 0.22, 0.32)))
    gain = num(turbine_out, 10.5, num(heavy, 4.5, 2.4))
    idle = landing & (pz <= 0.638) & (up_h < 0.85) & (vz.abs() < 0.20)
    inv = ct < 0.20
    inv_rx = num(te_n > 1e-5, e_rx, tilt)
    tx_inv, ty_inv = 130 * inv_rx - 52 * ox, 130 * e_ry - 52 * oy
    raw_u, outer_cmd, inner_cmd = [], [], []
    for a, (dx, dy) in enumerate(((1, 0), (0, 1), (-1, 0), (0, -1))):
        alpha = torch.asin((yaw_ft / thrust[a].clamp(min=30.0)).clamp(-0.35, 0.35))
        outer_cmd.append((6.5 * _wrap(alpha, outer[a])).clamp(-2, 2))
        sin_in = clip(0.5 * (fx_rem * dx + fy_rem * dy) / thrust[a].clamp(min=40.0), -max_sin,
                      max_sin)
        inner_cmd.append(torch.asin(sin_in).clamp(-_PI / 4 * 0.9, _PI / 4 * 0.9))
        cos_in = (torch.cos(alpha) * torch.cos(inner_cmd[a])).clamp(min=0.7)
        want = num(idle, 0.15 * weight * 0.25, fz_cmd[a].clamp(min=0) / cos_in)
        u = ((want - full * 0.08) / (full - full * 0.08)).clamp(0, 1)
        raw_u.append(u + gain * (u - spool[a]))
    top = torch.stack(raw_u).max(dim=0).values
    excess = num(headroom, clip(top - 1, 0, num(urgent, 0.10, 0.45)), 0)
    throttle = [(u - excess).clamp(0, 1) for u in raw_u]
    moment = (-ty_inv, tx_inv, ty_inv, -tx_inv)
    throttle = [num(inv, num(moment[a] > 12, 0.58, 0), throttle[a]) for a in range(4)]
    outer_cmd = [num(inv, (-outer[a] * 6).clamp(-2, 2), outer_cmd[a]) for a in range(4)]
    inner_cmd = [num(inv, 0, inner_cmd[a]) for a in range(4)]
    ready = arena & (o[46] <= 0.02) & (o[47] > 0.01)
    fire = ready & ~inv & (hyp(can_err, can_el - o[45]) < 0.28) & (dist < 34)
    n_az = num(arena & ~inv, ((can_az - _PI / 4) / (_PI / 6)).clamp(-1, 1), 0)
    n_az = num(inv, -1, n_az)
    n_el = num(arena & ~inv, (can_el / (_PI / 6)).clamp(-1, 1), 0)
    n_fire = num(fire, 0.8, -0.8)

    want_v = num(endurance, 18.5, num(arena, num(gdist > 38, 26, 24), 22.4))
    u_coll = (num(endurance, 0.36, 0.44) + 0.065 * (want_v - vb_x) + 0.018 * gz).clamp(0.12, 0.9)
    diff = (0.9 * ((-1.35 * course_err).clamp(-0.55, 0.55) - roll) - 0.34 * ox).clamp(-0.45, 0.45)
    u0, u1 = (u_coll + diff).clamp(0.05, 1), (u_coll - diff).clamp(0.05, 1)
    cb, sb = torch.cos(roll), torch.sin(roll)
    pitch = (0.062831853 + 0.75 * gamma + 0.035 * (climb - vz) +
             0.09 * (1 - cb.clamp(min=0.5))).clamp(-0.15, 0.25)
    pitch = num(vb_x < 15.5, pitch.clamp(max=0.02), pitch)
    theta = 2.2 * (pitch - torch.asin(r[2][0].clamp(-1, 1)))
    psi = g / vb_x.clamp(min=12.0) * torch.tan((-roll).clamp(-0.75, 0.75)) + 0.35 * course_err
    q_up, r_left = cb * theta - sb * psi, sb * theta + cb * psi
    in0 = (0.85 * (q_up + oy) + 0.03).clamp(-_PI / 6, _PI / 6)
    in1 = (-0.65 * (r_left - oz) - 0.025 * vb_y).clamp(-_PI / 6, _PI / 6)
    b_fire = ready & (hyp(b_can_err, b_el - o[45]) < 0.045) & (bdist < 165) & (bb[0] > 0)
    throttle = [num(bwb, (u0, u1)[a & 1], throttle[a]) for a in range(4)]
    outer_cmd = [num(bwb, 0, x) for x in outer_cmd]
    inner_cmd = [num(bwb, (in0, in1, 0, 0)[a], inner_cmd[a]) for a in range(4)]
    n_az = num(bwb, num(arena, (b_az / (_PI / 6)).clamp(-1, 1), 0), n_az)
    n_el = num(bwb, num(arena, (b_el / (_PI / 6)).clamp(-1, 1), 0), n_el)
    n_fire = num(bwb, num(b_fire, 0.8, -0.8), n_fire)
    prior = torch.stack([*[(t * 2 - 1).clamp(-1, 1) for t in throttle],
                         *[(x / 2).clamp(-1, 1) for x in outer_cmd],
                         *[(x / (_PI / 4)).clamp(-1, 1) for x in inner_cmd],
                         n_az, n_el, n_fire], dim=1)
    diag = torch.stack([min_r, ray.double(), min_dx, count.double(), y_sum], dim=1)
    return prior, diag


def _exact_inputs(s, tactical, prior):
    raw = torch.cat([s["obs"][:, :48], s["obs"][:, 4144:]], dim=1).double()
    scale = torch.ones(52, dtype=torch.float64, device=DEVICE)
    scale[0:3], scale[3:6], scale[10:13], scale[13:16] = 0.05, 0.10, 0.20, 0.10
    scale[28:32], scale[32:36] = 0.5, 0.2
    x = raw.clamp(-1000, 1000) * scale
    symlog = (torch.sign(x) * torch.log1p(x.abs()) / math.sqrt(1.0001)).clamp(-8, 8)
    r = s["obs"][:, 48:4144].double().view(-1, 2, 16, 128)
    valid, near = r > 0, r.clamp(0.05, 30)
    lidar = torch.cat([torch.where(valid, 1 / near.clamp(min=0.2), 0.0),
                       torch.where(valid, near / 30, 1.0), valid.double()], dim=1)
    luma = (s["cameras"].double() / 255 - 0.5).view(-1, 4, 64, 64)
    return {"proprio": torch.cat([symlog, tactical, prior], dim=1),
            "mission_vec": torch.cat([s["mission"].double(), tactical, prior], dim=1),
            "lidar": lidar, "luma": luma}


def _exact_policy(s):
    w = [x.double() for x in s["weights"]]
    h = torch.tanh(s["features"].double() @ w[0].T + w[1])
    raw = torch.tanh(h @ w[2].T + w[3]) @ w[4].T + w[5]
    mean, log_std = raw[:, :actor.ACTIONS], raw[:, actor.ACTIONS:].clamp(-3.5, -1.6)
    eps = torch.zeros_like(mean) if s["normals"] is None else s["normals"].double()
    eps = eps * torch.tensor([1.0] * 14 + [0.15], dtype=torch.float64, device=DEVICE)
    act = torch.tanh((mean + log_std.exp() * eps).clamp(-8, 8))
    lp = (-0.5 * eps * eps - log_std - 0.5 * math.log(2 * _PI) -
          torch.log(1 - act * act + 1e-6)).sum(dim=1)
    return {"actions": act, "log_prob": None if s["normals"] is None else lp, "raw": raw}


def exact(case, seed):
    entry = case["entry"]
    if entry in ("act", "refresh", "step"):
        s = _policy(case, seed)
        if entry != "step":
            return _exact_policy(s)
        s["features"] = _exact_features(s, "batch")
        return {**_exact_policy(s), "features": s["features"]}
    s = _sensors(case, seed)
    if entry in ("features", "host"):
        layout = case.get("layout", "batch")
        if layout == "sampled":
            at = s["indices"].long()
            s.update({k: s[k][at] for k in ("obs", "mission", "cameras")})
        parts, n = [], case["n"]
        for i in range(0, n, 4096):
            part = {k: s[k][i:i + 4096] for k in ("obs", "mission", "cameras", "depth") if k in s}
            parts.append(_exact_features(part, layout))
        out = torch.cat(parts)
        if entry == "host":
            return out.cpu().numpy()
        return {"features": out, **({"diag": None} if layout == "diagnostics" else {})}
    obs, mission = s["obs"].double(), s["mission"].double()
    tactical = _exact_tactical(obs[:, :48], mission)
    prior, diag = _exact_prior(obs, mission)
    if entry == "onboard":
        return {"tactical": tactical, "prior": prior, **({"diag": diag} if case["diag"] else {})}
    return {"tactical": tactical, "prior": prior, **_exact_inputs(s, tactical, prior)}
