"""Performance cases of particular_amd: the calls a simulation makes, over the sizes it makes them at.

Every case goes through a public entry point (``BruteForce``, ``BruteForcePairs`` and ``BarnesHut``
``compute``, the leapfrog loop, the batched ensemble and the network's gradient). Inputs follow the
library's own workloads: Plummer spheres, pairs of them, massless test particles in a cube, and the
uniform cube of the reference's benchmark. ``exact`` gives the same quantities in 64 bits from plain
torch, without the library.
"""
import ctypes
import math

import numpy as np
import torch

import particular_amd as pa
from particular_amd import _lib, learned, workloads

DEV = "cuda:0"
MASS_CAP = 0.999  # Plummer spheres are cut at the radius holding this share of the mass


def listed():
    return [
        # The smallest call: a few dozen bodies, a planetary system stepped by the caller.
        {"name": "brute_force_64", "kind": "brute_force", "n": 64, "massive": 64, "eps": 0.0,
         "checked": True, "host": False},
        # The direct sum over 4,096 bodies held in host arrays, as the reference's own GPU path
        # takes and returns them.
        {"name": "brute_force_host_4096", "kind": "brute_force", "n": 4096, "massive": 4096,
         "eps": 0.0, "checked": True, "host": True},
        # Direct sum at scale: 1M softened bodies of which 64K are massive, interleaved; the
        # storage separates them on every call.
        {"name": "brute_force_1m_x_64k", "kind": "brute_force", "n": 1048576, "massive": 65536,
         "eps": 1e-3, "checked": True, "host": False},
        # The same interface for 64-bit particles.
        {"name": "brute_force_f64_10007", "kind": "brute_force_f64", "n": 10007, "eps": 0.0,
         "checked": True},
        # All bodies massive, every pair taken once.
        {"name": "pairs_30011", "kind": "pairs", "n": 30011, "eps": 1e-3, "checked": True},
        # Barnes-Hut on a small system, where the build's launches and the walk's latency count.
        {"name": "barnes_hut_4096", "kind": "barnes_hut", "n": 4096, "massive": 4096, "theta": 0.5,
         "eps": 0.0, "mlp": False, "alpha": 0.0},
        # An ordinary run: a ragged count, softened, a third of the bodies massless.
        {"name": "barnes_hut_100003", "kind": "barnes_hut", "n": 100003, "massive": 66667,
         "theta": 0.7, "eps": 1e-3, "mlp": False, "alpha": 0.0},
        # The largest tree: two Plummer spheres of 2M bodies each.
        {"name": "barnes_hut_4m", "kind": "barnes_hut", "n": 4194304, "massive": 4194304,
         "theta": 0.5, "eps": 0.0, "mlp": False, "alpha": 0.0},
        # The learned correction with the trained network, at the angle that gives 1e-4 rms.
        {"name": "corrected_1m", "kind": "barnes_hut", "n": 1048576, "massive": 1048576,
         "theta": 0.45, "eps": 0.0, "mlp": True, "alpha": 0.0},
        # The step loop (kick-drift-kick, FP64 state, graph replay), state read back at the end.
        {"name": "leapfrog_65536", "kind": "leapfrog", "n": 65536, "massive": 16384, "steps": 10,
         "eps": 1e-3},
        # Many independent systems of uneven sizes stepped together.
        {"name": "ensemble_128", "kind": "ensemble", "systems": 128, "n_min": 64, "n_max": 16384,
         "steps": 16, "eps": 1e-3},
        # Training the correction: the loss and its gradient over a set of rows.
        {"name": "network_gradient", "kind": "gradient", "waves": 128, "rows": 2000},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["brute_force", "brute_force", "brute_force_f64", "pairs", "barnes_hut",
                       "barnes_hut", "barnes_hut", "leapfrog", "ensemble", "gradient"])
    eps = rng.choice([0.0, 1e-3, 1e-2])
    if kind == "brute_force":
        n = _log_int(rng, 64, 500000)
        massive = n if rng.random() < 0.5 and n <= 130000 else max(1, min(65536, int(n * rng.uniform(0.05, 0.6))))
        return {"kind": kind, "n": n, "massive": massive, "eps": eps,
                "checked": eps == 0.0 or rng.random() < 0.5, "host": rng.random() < 0.25}
    if kind == "brute_force_f64":
        return {"kind": kind, "n": _log_int(rng, 100, 40000), "eps": eps,
                "checked": eps == 0.0 or rng.random() < 0.5}
    if kind == "pairs":
        return {"kind": kind, "n": _log_int(rng, 300, 130000), "eps": eps, "checked": True}
    if kind == "barnes_hut":
        n = _log_int(rng, 200, 2000000)
        mlp = rng.random() < 0.3
        return {"kind": kind, "n": n,
                "massive": n if mlp or rng.random() < 0.6 else max(1, int(n * rng.uniform(0.1, 0.9))),
                "theta": round(rng.uniform(0.4, 0.9), 3), "eps": eps, "mlp": mlp,
                "alpha": rng.choice([0.0, 0.0, 0.0, 3e-4])}
    if kind == "leapfrog":
        n = _log_int(rng, 256, 200000)
        return {"kind": kind, "n": n, "massive": max(1, int(n * rng.uniform(0.1, 0.5))),
                "steps": rng.randint(4, 20), "eps": rng.choice([1e-3, 1e-2])}
    if kind == "ensemble":
        return {"kind": kind, "systems": rng.randint(16, 256), "n_min": rng.choice([32, 64, 100]),
                "n_max": _log_int(rng, 500, 16384), "steps": rng.randint(4, 16),
                "eps": rng.choice([1e-3, 1e-2])}
    return {"kind": kind, "waves": rng.randint(16, 200), "rows": rng.randint(300, 2500)}


# ---- inputs -------------------------------------------------------------------------------------

_handle = None


def _resources():
    """The one device handle a program creates and keeps."""
    global _handle
    if _handle is None:
        _handle = pa.HipResources(0)
    return _handle


def _plummer(gen, n):
    """(n, 3) float64 positions of a Plummer sphere of scale radius 1."""
    u = torch.rand((n, 3), generator=gen, device=DEV, dtype=torch.float64)
    r = (torch.clamp(u[:, 0] * MASS_CAP, min=1e-12) ** (-2.0 / 3.0) - 1.0) ** -0.5
    cos = 2.0 * u[:, 1] - 1.0
    sin = torch.sqrt(torch.clamp(1.0 - cos * cos, min=0.0))
    phi = 2.0 * math.pi * u[:, 2]
    return torch.stack([sin * torch.cos(phi), sin * torch.sin(phi), cos], 1) * r[:, None]


def _particles(case, seed):
    """(n, 4) float64 {x, y, z, mu} on the GPU: two Plummer spheres for Barnes-Hut, one for the
    others, and massless bodies uniform in a cube around them, all in a random order."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(int(seed))
    n = case["n"]
    m = case.get("massive", n)
    pos = _plummer(gen, m)
    side = 4.0
    if case["kind"] == "barnes_hut":
        pos[: m // 2, 0] -= 5.0
        pos[m // 2:, 0] += 5.0
        side = 20.0
    cube = (torch.rand((n - m, 3), generator=gen, device=DEV, dtype=torch.float64) - 0.5) * side
    mu = torch.zeros(n, device=DEV, dtype=torch.float64)
    mu[:m] = 1.0 / m
    p = torch.cat([torch.cat([pos, cube]), mu[:, None]], 1)
    if case["kind"] == "brute_force_f64" or m == n and case.get("host"):
        # the reference benchmark's bodies: a uniform cube with masses spread over its range
        p[:, :3] = (torch.rand((n, 3), generator=gen, device=DEV, dtype=torch.float64) - 0.5) * 1e4
        p[:, 3] = 1e3 + torch.rand(n, generator=gen, device=DEV, dtype=torch.float64) * 1e9
    return p[torch.randperm(n, generator=gen, device=DEV)]


def _interaction(case):
    if case["eps"] > 0.0:
        make = pa.AccelerationSoftened.checked if case["checked"] else pa.AccelerationSoftened.unchecked
        return make(case["eps"])
    return pa.Acceleration.checked() if case["checked"] else pa.Acceleration.unchecked()


def _state(case, seed):
    """Host arrays (pos, vel, mu) of the step loop: positions as above, small random velocities."""
    p = _particles(case, seed).cpu().numpy()
    vel = np.random.default_rng(seed).normal(0.0, 0.3, (case["n"], 3))
    return np.ascontiguousarray(p[:, :3]), vel, p[:, 3].astype(np.float32)


def _offsets(case):
    """Sizes spread evenly over their logarithm, in a fixed random order; as system offsets."""
    u = (np.random.default_rng(case["systems"]).permutation(case["systems"]) + 0.5) / case["systems"]
    s = np.exp(np.log(case["n_min"]) + u * (np.log(case["n_max"]) - np.log(case["n_min"])))
    return np.concatenate([[0], np.cumsum(s.astype(np.int64))])


def _ensemble(case, seed):
    """Host arrays (pos, vel, mu, offsets) of Plummer systems of scale radius 0.5 to 2."""
    off = _offsets(case)
    pos, vel = workloads.plummer(int(off[-1]), seed)
    scale = np.random.default_rng(seed).uniform(0.5, 2.0, case["systems"])
    size = np.diff(off)
    scale = np.repeat(scale, size)[:, None]
    return pos * scale, vel / np.sqrt(scale), np.repeat(1.0 / size, size).astype(np.float32), off


def _rows(case, seed):
    """A training set as the walk lists it: per wavefront of 64 neighbouring bodies, the nodes its
    lanes accepted, nearer ones narrower, most of them taken by every lane."""
    rng = np.random.default_rng(seed)
    waves, per = case["waves"], case["rows"]
    rows = waves * per
    centre = rng.normal(0.0, 2.0, (waves, 3))
    lanes = np.zeros((waves, 64, 4))
    lanes[:, :, :3] = centre[:, None] + rng.normal(0.0, 0.02, (waves, 64, 3))
    wave = np.repeat(np.arange(waves), per)
    width = np.exp(rng.uniform(np.log(0.01), np.log(2.0), rows))
    way = rng.normal(0.0, 1.0, (rows, 3))
    way /= np.linalg.norm(way, axis=1)[:, None]
    geom = np.zeros((rows, learned.GEOM))
    geom[:, :3] = centre[wave] + way * (width * rng.uniform(2.0, 4.0, rows) + 0.1)[:, None]
    mass = width ** 3 * 1e-3
    geom[:, 3] = mass * width ** 2
    geom[:, 4] = mass * width ** 3
    feats = np.zeros((rows, learned.FEAT))
    feats[:, :6] = rng.normal(0.0, 0.15, (rows, 6))
    feats[:, 6] = rng.uniform(0.3, 1.0, rows)
    feats[:, 7] = rng.uniform(0.05, 0.6, rows)
    feats[:, 8] = rng.integers(2, 18, rows) / 64.0
    feats[:, 9:] = rng.normal(0.0, 0.3, (rows, 7))
    mask = np.full(rows, np.uint64(0xFFFFFFFFFFFFFFFF))
    some = rng.random(rows) < 0.3
    mask[some] = rng.integers(1, 1 << 63, int(some.sum()), dtype=np.uint64)
    target = np.zeros((waves, 64, 4))
    target[:, :, :3] = rng.normal(0.0, 1e-3, (waves, 64, 3))
    return {"feats": feats.astype(np.float32), "geom": geom.astype(np.float32), "mask": mask,
            "row_wave": wave.astype(np.uint32),
            "wave_rows": (np.arange(waves + 1) * per).astype(np.uint32),
            "lanes": lanes.astype(np.float32), "target": target.astype(np.float32),
            "wgt": rng.uniform(0.5, 2.0, (waves, 64)).astype(np.float32)}


def _network(seed):
    """The trained network, its weights moved a little, as a training run has them on the way."""
    p = learned.default_params().astype(np.float64)
    rng = np.random.default_rng(seed)
    return (p + rng.normal(0.0, 0.02, p.size)).astype(np.float32)


# ---- prepare and run ------------------------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    if kind == "leapfrog":
        res = pa.HipResources(0)  # the loop's state lives in its handle
        pos, vel, mu = _state(case, seed)
        res.check(_lib.lib().pnb_leapfrog_init(res.handle, pos.ctypes.data, vel.ctypes.data,
                                               mu.ctypes.data, case["n"], case["eps"], 1))
        return {"case": case, "res": res, "out": _step_outputs(case["n"])}
    if kind == "ensemble":
        res = pa.HipResources(0)
        pos, vel, mu, off = _ensemble(case, seed)
        res.check(_lib.lib().pnb_batch_init(res.handle, pos.ctypes.data, vel.ctypes.data,
                                            mu.ctypes.data, off.ctypes.data, case["systems"],
                                            case["eps"], 1))
        return {"case": case, "res": res, "out": _step_outputs(pos.shape[0])}
    if kind == "gradient":
        res = pa.HipResources(0)
        learned.init(res, 0)
        learned.set_params(res, _network(seed))
        learned.load(res, _rows(case, seed))
        return {"case": case, "res": res}
    p = _particles(case, seed)
    res = _resources()
    if kind == "brute_force_f64":
        return {"case": case, "algorithm": pa.BruteForce(res, _interaction(case)),
                "storage": p.cpu().numpy()}
    p = p.float()
    if kind == "pairs":
        return {"case": case, "algorithm": pa.BruteForcePairs(res, _interaction(case)), "storage": p}
    if kind == "brute_force":
        algorithm = pa.BruteForce(res, _interaction(case))
    else:
        if case["mlp"]:
            learned.init(res, 0)
            learned.set_params(res, learned.default_params())
        algorithm = pa.BarnesHut(res, case["theta"], _interaction(dict(case, checked=True)),
                                 mlp=case["mlp"], relative=case["alpha"] or None)
    if case.get("host"):
        p = p.cpu().numpy()
    return {"case": case, "algorithm": algorithm,
            "storage": p if case["massive"] == case["n"] else pa.Reordered.new(p)}


def _step_outputs(n):
    return np.empty((n, 3)), np.empty((n, 3)), np.empty((n, 4), np.float32)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("leapfrog", "ensemble"):
        res, (pos, vel, acc), lib = state["res"], state["out"], _lib.lib()
        step = lib.pnb_leapfrog_run if kind == "leapfrog" else lib.pnb_batch_run
        read = lib.pnb_leapfrog_read if kind == "leapfrog" else lib.pnb_batch_read
        res.check(step(res.handle, case["steps"], ctypes.c_double(2.0 ** -13), 1))
        res.check(read(res.handle, pos.ctypes.data, vel.ctypes.data, acc.ctypes.data))
        return {"pos": pos, "vel": vel, "acc": acc}
    if kind == "gradient":
        loss, grads = learned.grad(state["res"])
        return {"loss": loss, "grads": grads}
    return state["algorithm"].compute(state["storage"])


# ---- work -------------------------------------------------------------------------------------------

def _walk_terms(m, theta):
    """Pair terms a particle takes in a walk: about 13 log2(m) / theta^3, at most one per body."""
    return min(float(m), 13.0 * math.log2(max(m, 2)) / theta ** 3)


def work(case):
    """20 operations per pair term (38 with the correction's two fields); inputs and outputs once."""
    kind = case["kind"]
    if kind == "ensemble":
        sizes = np.diff(_offsets(case))
        total, pairs = float(sizes.sum()), float((sizes.astype(np.float64) ** 2).sum())
        return {"bytes": case["steps"] * total * 160.0 + total * 64.0,
                "flops": 20.0 * pairs * case["steps"]}
    if kind == "leapfrog":
        n, m = float(case["n"]), float(case["massive"])
        return {"bytes": case["steps"] * n * 160.0 + n * 64.0, "flops": 20.0 * n * m * case["steps"]}
    if kind == "gradient":
        rows = float(case["waves"] * case["rows"])
        return {"bytes": rows * (64 + 32 + 8 + 4), "flops": rows * (37e3 + 64 * 120)}
    n, m = float(case["n"]), float(case.get("massive", case["n"]))
    if kind == "brute_force_f64":
        return {"bytes": n * 64.0, "flops": 20.0 * n * m}
    if kind == "pairs":
        return {"bytes": n * 32.0, "flops": 15.0 * n * n}
    if kind == "barnes_hut":
        return {"bytes": n * 32.0, "flops": (38.0 if case["mlp"] else 20.0) * n * _walk_terms(m, case["theta"])}
    return {"bytes": n * 32.0, "flops": 20.0 * n * m}


# ---- the same quantities in 64 bits -----------------------------------------------------------------

def _direct(a, b, eps):
    """(n, 3) accelerations of a by b ((m, 4)) in 64 bits; pairs at zero distance add nothing."""
    out = torch.empty((a.shape[0], 3), dtype=torch.float64, device=a.device)
    step = max(1, int(1.5e8 // max(1, b.shape[0])))
    for i in range(0, a.shape[0], step):
        d = [b[None, :, k] - a[i:i + step, k, None] for k in range(3)]
        r2 = d[0] * d[0]
        r2.addcmul_(d[1], d[1]).addcmul_(d[2], d[2])
        zero = r2 == 0.0
        r2.add_(eps * eps)
        w = r2.rsqrt_() ** 3
        w.masked_fill_(zero, 0.0).mul_(b[None, :, 3])
        for k in range(3):
            out[i:i + step, k] = (d[k] * w).sum(1)
    return out


def _barnes_hut(a, b, theta, eps):
    """Barnes-Hut by the reference's rules, whole levels at a time: cells and opening decisions in
    the 32-bit arithmetic that defines them, node data and sums in 64 bits."""
    f32 = b[:, :3].float()
    lo, hi = f32.amin(0), f32.amax(0)
    centre, half = (lo + hi) * 0.5, (hi - lo).amax() * 0.5
    n = b.shape[0]
    mn, mx = (centre - half).expand(n, 3).clone(), (centre + half).expand(n, 3).clone()
    cell = torch.zeros(n, dtype=torch.int64, device=b.device)
    body = torch.arange(n, device=b.device)
    levels, parent_of_cell = [], None
    key = cell
    while True:
        # the nodes of this level: bodies with one key, and whether they all share one position
        ids, key = torch.unique(key, return_inverse=True)
        count = ids.numel()
        q = b[body]
        mass = torch.zeros(count, dtype=torch.float64, device=b.device).index_add_(0, key, q[:, 3])
        com = torch.zeros((count, 3), dtype=torch.float64, device=b.device)
        com.index_add_(0, key, q[:, :3] * q[:, 3:])
        first = torch.full((count,), n, dtype=torch.int64, device=b.device)
        first = first.scatter_reduce(0, key, torch.arange(body.numel(), device=b.device), "amin")
        differs = (q[:, :3] != q[first[key], :3]).any(1)
        internal = torch.zeros(count, dtype=torch.bool, device=b.device)
        internal[key[differs]] = True
        width = (mx - mn)[first, 0]
        com = torch.where(internal[:, None], com / mass[:, None], q[first, :3])
        parent = parent_of_cell[first] if parent_of_cell is not None else None
        levels.append({"com": com, "com32": com.float(), "mass": mass, "parent": parent,
                       "w2": torch.where(internal, width * width, -1.0)})
        keep = internal[key]
        if not bool(keep.any()):
            break
        body, parent_of_cell = body[keep], key[keep]
        mn, mx = mn[keep], mx[keep]
        x = f32[body]
        mid = (mn + mx) * 0.5
        low = x < mid
        mx, mn = torch.where(low, mid, mx), torch.where(low, mn, mid)
        child = low[:, 0] * 1 + low[:, 1] * 2 + low[:, 2] * 4
        key = parent_of_cell * 8 + child
    for l in range(len(levels) - 1):  # the children of each node of level l
        p = levels[l + 1]["parent"]
        order = torch.argsort(p, stable=True)
        num = torch.bincount(p, minlength=levels[l]["mass"].numel())
        levels[l]["kids"], levels[l]["num"] = order, num
        levels[l]["start"] = torch.cumsum(num, 0) - num
    out = torch.zeros((a.shape[0], 3), dtype=torch.float64, device=a.device)
    step = 8192
    for i in range(0, a.shape[0], step):
        pts = a[i:i + step, :3]
        pts32, theta32 = pts.float(), torch.tensor(theta, dtype=torch.float32, device=a.device)
        lane = torch.arange(pts.shape[0], device=a.device)
        node = torch.zeros_like(lane)
        for l, L in enumerate(levels):
            dx, dy, dz = (L["com32"][node] - pts32[lane]).unbind(1)
            near = (dx * dx + dy * dy) + dz * dz
            nz = near != 0.0
            opened = nz & (theta32 * theta32 * near < L["w2"][node])
            take = nz & ~opened
            d = L["com"][node] - pts[lane]
            d2 = (d * d).sum(1)
            w = torch.where(take, L["mass"][node] * torch.where(take, d2 + eps * eps, 1.0) ** -1.5, 0.0)
            out[i:i + step].index_add_(0, lane, d * w[:, None])
            lane, node = lane[opened], node[opened]
            if lane.numel() == 0:
                break
            num = L["num"][node]
            lane = torch.repeat_interleave(lane, num)
            base = torch.repeat_interleave(L["start"][node] - (torch.cumsum(num, 0) - num), num)
            node = L["kids"][base + torch.arange(lane.numel(), device=a.device)]
    return out


def _leapfrog(pos, vel, mu, eps, steps, dt):
    """Kick-drift-kick in 64 bits; the accelerations see the positions rounded to 32 bits, as the
    loop's particles are."""
    def force():
        p = torch.cat([pos.float().double(), mu[:, None]], 1)
        return _direct(p, p[mu != 0.0], eps)
    acc = force()
    for _ in range(steps):
        vel = vel + acc * (0.5 * dt)
        pos = pos + vel * dt
        acc = force()
        vel = vel + acc * (0.5 * dt)
    return pos, vel, acc


def _with_zero(acc):
    return torch.cat([acc, torch.zeros((acc.shape[0], 1), dtype=acc.dtype, device=acc.device)], 1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "gradient":
        return _gradient(case, seed)
    if kind == "ensemble":
        *host, off = _ensemble(case, seed)
        pos, vel, mu = (torch.from_numpy(v).to(DEV).double() for v in host)
        parts = []
        for b, t in zip(off[:-1], off[1:]):
            parts.append(_leapfrog(pos[b:t], vel[b:t], mu[b:t], case["eps"], case["steps"],
                                   2.0 ** -13))
        pos, vel, acc = (torch.cat(v) for v in zip(*parts))
        return {"pos": pos, "vel": vel, "acc": _with_zero(acc)}
    if kind == "leapfrog":
        pos, vel, mu = (torch.from_numpy(v).to(DEV) for v in _state(case, seed))
        pos, vel, acc = _leapfrog(pos, vel, mu.double(), case["eps"], case["steps"], 2.0 ** -13)
        return {"pos": pos, "vel": vel, "acc": _with_zero(acc)}
    p = _particles(case, seed)
    if kind == "brute_force_f64":
        return _direct(p, p, case["eps"])
    p = p.float().double()
    if kind == "barnes_hut":
        # the correction and the relative rule are the library's own methods; very large sets take long
        if case["mlp"] or case["alpha"] or case["n"] > 300000:
            return None
        return _with_zero(_barnes_hut(p, p[p[:, 3] != 0.0], case["theta"], case["eps"]))
    acc = _direct(p, p if kind == "pairs" else p[p[:, 3] != 0.0], case["eps"])
    return acc if case.get("host") else _with_zero(acc)


def _gradient(case, seed):
    """Loss and gradients of the correction's network (16-64-64-13, ReLU, a residual on the first
    six outputs) in 64 bits, by automatic differentiation."""
    d = _rows(case, seed)
    shapes = [(16, 64), (64,), (64, 64), (64,), (64, 13), (13,)]
    flat = torch.from_numpy(_network(seed).astype(np.float64)).to(DEV).requires_grad_(True)
    parts, at = [], 0
    for s in shapes:
        parts.append(flat[at:at + math.prod(s)].reshape(s))
        at += math.prod(s)
    w1, b1, w2, b2, w3, b3 = parts
    x = torch.from_numpy(d["feats"]).to(DEV).double()
    geom = torch.from_numpy(d["geom"]).to(DEV).double()
    lanes = torch.from_numpy(d["lanes"]).to(DEV).double()
    bits = (d["mask"][:, None] >> np.arange(64, dtype=np.uint64)[None, :]) & np.uint64(1)
    bits = torch.from_numpy(bits.astype(np.uint8)).to(DEV).double()
    h = torch.relu(torch.relu(x @ w1 + b1) @ w2 + b2)
    y = h @ w3 + b3
    y = torch.cat([y[:, :6] + x[:, :6], y[:, 6:]], 1)
    out = y.detach().requires_grad_(True)
    per = case["rows"]
    target = torch.from_numpy(d["target"]).to(DEV).double()[:, :, :3]
    wgt = torch.from_numpy(d["wgt"]).to(DEV).double()
    count = max(int((d["wgt"] > 0).sum()), 1)
    loss = 0.0
    for w in range(case["waves"]):  # one wavefront at a time: its rows against its 64 lanes
        s = slice(w * per, (w + 1) * per)
        v = geom[s, None, :3] - lanes[w, None, :, :3]
        r2 = (v * v).sum(2) + lanes[w, None, :, 3]
        inv = r2.rsqrt() * bits[s]
        dx, dy, dz = v.unbind(2)
        q = (out[s, :6] * geom[s, 3:4])[:, None].unbind(2)
        qx = q[0] * dx + q[3] * dy + q[4] * dz
        qy = q[3] * dx + q[1] * dy + q[5] * dz
        qz = q[4] * dx + q[5] * dy + q[2] * dz
        o = (out[s, 6:] * geom[s, 4:5])[:, None].unbind(2)  # xxx yyy zzz xxy xxz xyy xyz
        xzz, yzz, yyz = -o[0] - o[5], -o[3] - o[1], -o[4] - o[2]
        fx = o[0] * dx * dx + o[5] * dy * dy + xzz * dz * dz + 2 * (o[3] * dx * dy + o[4] * dx * dz + o[6] * dy * dz)
        fy = o[3] * dx * dx + o[1] * dy * dy + yzz * dz * dz + 2 * (o[5] * dx * dy + o[6] * dx * dz + yyz * dy * dz)
        fz = o[4] * dx * dx + yyz * dy * dy + o[2] * dz * dz + 2 * (o[6] * dx * dy + xzz * dx * dz + yzz * dy * dz)
        i5 = inv ** 5
        i7 = i5 * inv * inv
        along = 2.5 * (dx * qx + dy * qy + dz * qz) * i7 - 7.0 * (dx * fx + dy * fy + dz * fz) * i7 * inv * inv
        pred = torch.stack([(along * dx - qx * i5 + 3.0 * fx * i7).sum(0),
                            (along * dy - qy * i5 + 3.0 * fy * i7).sum(0),
                            (along * dz - qz * i5 + 3.0 * fz * i7).sum(0)], 1)
        part = (wgt[w, :, None] * (pred - target[w]) ** 2).sum() / count
        part.backward()
        loss += float(part.detach())
    y.backward(out.grad)
    return {"loss": loss, "grads": flat.grad}
