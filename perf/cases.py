"""The work that programs built on this framework have it do, as timed cases.

Six kinds of program, each through the package's public entry points:

  frame    the interactive / headless loop with the default parameters (the
           reference step as written): Headless.step, then the positions that
           the renderer and the octree read
  step     the same loop for a science run: every field it carries is read
           after each step; Newton-Raphson stopped near its fixed point,
           optionally with the learned guess, individual timesteps, and the
           precision form
  nbody    fixed-step self-gravity alone: octree, gravity, kick and drift
  density  smoothing lengths and densities of a particle set handed in from
           the host (initial conditions, another code's snapshot)
  sort     the allocation-free hash, radix sort and cell table on the caller's
           own buffers
  train    Adam steps of the smoothing-length network on dumped samples

The default Newton-Raphson rule stops on a threshold of 0.5% on h
(DENSITY_ETA): a last-bit difference in a sum moves one particle in 1e5 to
1e6 by that much, and with it its pressure and its neighbours' forces.
Cases that return h, rho or what depends on them therefore stop within
2.5e-6 of the fixed point (density_stop = 1, as bench.py's dumps and its
learned-h comparison do); the default rule's cases return the positions,
which such a difference does not reach.
"""
import importlib
import math

import numpy as np
import torch

sph = importlib.import_module("real-time-planetary-impacts-mps_amd")

# Newton-Raphson stopped within 2.5e-6 of the fixed point
FIXED_POINT = {"density_stop": 1, "density_eta": 2.5e-6, "max_nr_iterations": 400}
# second-order and third-order corrected gravity
NEAR = {"fixes": sph.SPH_FIX_ALL}
PRECISION = {"fixes": sph.SPH_FIX_ALL, "precision": 1, "expansion_order": 3, "mac_order": 2, "gravity_eta": 1e-3,
             "max_unchecked_pointers": 4096}
FORMS = {"written": {}, "near": NEAR, "precision": PRECISION}

STATE = ("pos", "vel", "u", "h", "rho", "pressure", "gradterm", "soundspeed", "du", "balsara", "dhdt", "gravnorm")
ALWAYS_ACTIVE = 1 << 30  # next_active of a run without individual timesteps


def listed():
    return [
        # the smallest demonstration impact (2e4 particles), a frame at a time: launches and latency count
        {"name": "frame_2e4", "kind": "frame", "n": 20000},
        # the headline impact at 1e6 particles, the reference step as written
        {"name": "frame_1e6", "kind": "frame", "n": 1000000},
        # a science run at the particle count that the reference quotes its rate for
        {"name": "step_1e5", "kind": "step", "n": 100003, "form": "written", "rungs": 0, "learned": False,
         "headon": False},
        # the headline impact with the learned starting guess
        {"name": "step_1e6_learned", "kind": "step", "n": 1000000, "form": "written", "rungs": 0, "learned": True,
         "headon": False},
        # the largest particle count the repository runs, a frame at a time
        {"name": "frame_4e6", "kind": "frame", "n": 4000000},
        # learned guess and precision form together on a head-on impact, individual timesteps: most steps have few
        # active particles (a size at which a timed block holds many of the rungs' cycles of 8 steps)
        {"name": "step_2e5_precision_rungs", "kind": "step", "n": 200000, "form": "precision", "rungs": 4,
         "learned": True, "headon": True},
        # self-gravity alone: small, as written; and third-order precision with every particle active
        {"name": "nbody_2e4", "kind": "nbody", "n": 20011, "form": "written"},
        {"name": "nbody_2e5_precision", "kind": "nbody", "n": 200000, "form": "precision"},
        # densities of a particle set of another code
        {"name": "density_3e5", "kind": "density", "n": 300007},
        # the sort in a caller's loop, small and near the largest it takes
        {"name": "sort_2e4", "kind": "sort", "n": 20000, "cell_power": 8},
        {"name": "sort_4e6", "kind": "sort", "n": 4000037, "cell_power": 8},
        # the network's training as bench.py runs it, 50 of its steps
        {"name": "train_65536", "kind": "train", "batch": 65536, "steps": 50},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("frame", "step", "step", "nbody", "density", "sort", "train"))
    if kind == "frame":
        return {"kind": kind, "n": _log_int(rng, 5000, 1000000)}
    if kind == "step":
        # the precision form with every particle active would cost more than the largest case
        form = rng.choice(("written", "near", "precision"))
        rungs = 4 if form == "precision" else rng.choice((0, 0, 4))
        top = 1000000 if rungs else (700000 if form == "written" else 300000)
        return {"kind": kind, "n": _log_int(rng, 10000, top), "form": form, "rungs": rungs,
                "learned": rng.random() < 0.5, "headon": rng.random() < 0.5}
    if kind == "nbody":
        form = rng.choice(("written", "near", "precision"))
        return {"kind": kind, "n": _log_int(rng, 5000, 800000 if form == "written" else 200000), "form": form}
    if kind == "density":
        return {"kind": kind, "n": _log_int(rng, 10000, 700000)}
    if kind == "sort":
        return {"kind": kind, "n": _log_int(rng, 2000, 4194304), "cell_power": rng.choice((6, 7, 8))}
    return {"kind": kind, "batch": 32 * rng.randrange(64, 2049), "steps": rng.randrange(10, 51)}


# ------------------------------------------------------------------- inputs
def two_bodies(n, seed):
    """A uniform target and impactor (89% / 11% of the particles, the radii
    and masses of the default impact) of equal-mass particles each, shortly
    before contact: positions, velocities, masses, materials and the smoothing
    lengths of the mean densities, FP32 (host)."""
    g = np.random.default_rng(seed)
    counts = (n - max(1, int(round(0.11 * n))), max(1, int(round(0.11 * n))))
    centres = ((18.0, 18.0, 20.0), (25.5, 24.5, 20.0))
    pos, vel, mass, mat, h = [], [], [], [], []
    for k, (radius, total, centre, v) in enumerate(((6.4, 5.3, centres[0], (0.0009, 0.0, 0.0)),
                                                    (3.6, 0.8, centres[1], (-0.0081, 0.0, 0.0)))):
        m = counts[k]
        d = g.standard_normal((m, 3))
        r = radius * np.cbrt(g.random(m))
        x = np.zeros((m, 4), np.float32)
        x[:, :3] = d * (r / np.linalg.norm(d, axis=1))[:, None] + np.array(centre)
        pos.append(x)
        vel.append(np.tile(np.array(v + (0.0,), np.float32), (m, 1)))
        mass.append(np.full(m, total / m, np.float32))
        mat.append(np.where(r < 0.55 * radius, 402, 400).astype(np.int32))
        h.append(np.full(m, 1.2348 * (4.0 / 3.0 * math.pi * radius ** 3 / m) ** (1.0 / 3.0), np.float32))
    out = {"pos": np.concatenate(pos), "vel": np.concatenate(vel), "mass": np.concatenate(mass),
           "mat": np.concatenate(mat), "h": np.concatenate(h)}
    out["rho"] = (1.2348 ** 3 * out["mass"] / out["h"] ** 3).astype(np.float32)
    out["u"] = np.full(n, 2e-6, np.float32)
    out["pressure"] = np.zeros(n, np.float32)
    return out


class _DeviceArray:
    """A per-particle buffer of a context, for torch (zero copy); torch keeps
    this object, and with it the buffer's owner, as long as the tensor lives."""

    def __init__(self, owner, ctx, field):
        self.owner = owner
        ptr, nbytes = ctx.device_field(field)
        shape = (ctx.n, 4) if nbytes == 16 * ctx.n else (ctx.n,)
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "data": (ptr, False), "version": 2}


def views(owner, fields):
    ctx = getattr(owner, "ctx", owner)  # a Headless or a Context
    return {f: torch.as_tensor(_DeviceArray(owner, ctx, f), device="cuda") for f in fields}


def trained_guess(samples_n, seed, steps):
    """A network trained on the dumps of a seeded impact, and the samples."""
    prm = sph.default_params(**FIXED_POINT)
    smp = sph.Samples(6 * samples_n)
    hl = sph.Headless(prm, sph.impact_config(samples_n, seed), tree_mode=sph.TREE_GPU)
    hl.step()
    hl.ctx.set_sample_dump(smp)
    for _ in range(6):
        hl.step()
    hl.ctx.set_sample_dump(None)
    hl.close()
    net = sph.Mlp(seed=13)
    net.fit_norm(smp)
    if steps:
        net.train(smp, steps=steps, batch=65536, lr=2e-3, seed=14)
    return net, smp


def prepare(case, seed):
    torch.cuda.current_device()
    n, kind = case.get("n"), case["kind"]
    if kind == "frame":
        hl = sph.Headless(sph.default_params(), sph.impact_config(n, seed), tree_mode=sph.TREE_GPU)
        for _ in range(3):
            hl.step()
        return {"kind": kind, "hl": hl, "out": views(hl, ("pos",))}
    if kind == "step":
        kw = dict(FORMS[case["form"]], **FIXED_POINT)
        if case["rungs"]:
            # the step as written runs away with inactive particles: the drift correction is needed
            kw.update(activity_rule=sph.SPH_ACTIVE_README, max_rungs=case["rungs"])
            kw["fixes"] = kw.get("fixes", 0) | sph.SPH_FIX_INACTIVE_DRIFT
        hl = sph.Headless(sph.default_params(**kw), sph.impact_config(n, seed, headon=case["headon"]),
                          tree_mode=sph.TREE_GPU)
        net = None
        if case["learned"]:
            net, smp = trained_guess(50000, seed + 1000, 200)
            smp.close()
            hl.ctx.set_learned_guess(net)
        for _ in range(4):
            hl.step()
        fields = STATE + (("potential",) if case["form"] == "precision" else ())
        return {"kind": kind, "hl": hl, "net": net, "out": views(hl, fields)}
    if kind == "nbody":
        ctx = sph.Context(sph.default_params(**FORMS[case["form"]]), two_bodies(n, seed), _eos())
        ctx.upload("next_active", np.full(n, ALWAYS_ACTIVE, np.int32))
        ctx.upload("dt", np.array([DT_TICKS], np.int32))
        ctx.build_tree()
        ctx.gravity()  # the field that the acceptance test of the next pass weighs against
        ctx.sync()
        fields = ("pos", "vel", "gravnorm") + (("potential",) if case["form"] == "precision" else ())
        return {"kind": kind, "ctx": ctx, "out": views(ctx, fields)}
    if kind == "density":
        ic = two_bodies(n, seed)
        # with the rescanned density started from zero: as written, a particle of 128 or more neighbours counts them twice
        ctx = sph.Context(sph.default_params(fixes=sph.SPH_FIX_DENSITY_CACHE, **FIXED_POINT), ic, _eos())
        return {"kind": kind, "ctx": ctx, "pos": ic["pos"], "h": ic["h"],
                "out": views(ctx, ("h", "rho", "gradterm", "pressure", "soundspeed", "balsara"))}
    if kind == "sort":
        pos = torch.from_numpy(two_bodies(n, seed)["pos"]).cuda()
        pairs = torch.empty((n, 2), dtype=torch.int32, device="cuda")
        cells = torch.empty((1 << (3 * case["cell_power"]), 2), dtype=torch.int32, device="cuda")
        width = sph.default_params().cell_width * (1 << (8 - case["cell_power"]))
        return {"kind": kind, "pos": pos, "n": n, "width": width, "power": case["cell_power"], "pairs": pairs,
                "cells": cells}
    net, smp = trained_guess(100000, seed, 0)
    return {"kind": kind, "net": net, "smp": smp, "steps": case["steps"], "batch": case["batch"], "seed": seed}


_tables = {}


def _eos():
    if not _tables:
        _tables.update(sph.make_eos_tables(sph.default_params(), 256))
    return _tables


DT_TICKS = 256  # the nbody run's step, 0.125 s


def run(state):
    kind = state["kind"]
    if kind in ("frame", "step"):
        state["hl"].step()
        return state["out"]
    if kind == "nbody":
        ctx = state["ctx"]
        ctx.build_tree()
        ctx.gravity()
        ctx.step()
        ctx.sync()
        return state["out"]
    if kind == "density":
        ctx = state["ctx"]
        ctx.upload("pos", state["pos"])
        ctx.upload("h", state["h"])
        ctx.sort()
        ctx.density()
        ctx.sync()
        return state["out"]
    if kind == "sort":
        sph.sort_noalloc(state["pos"].data_ptr(), state["n"], state["width"], state["power"],
                         state["pairs"].data_ptr(), state["cells"].data_ptr(),
                         torch.cuda.current_stream().cuda_stream)
        return {"pairs": state["pairs"], "cells": state["cells"]}
    losses = state["net"].train(state["smp"], state["steps"], batch=state["batch"], lr=2e-3, seed=state["seed"])
    return {"params": state["net"].get()[0], "losses": losses}


def work(case):
    """Bytes and FP32 operations a pass cannot do without, per particle.

    63 neighbours lie within 2h; a Newton-Raphson scan takes 18 operations
    for each, the density pass's last sum 54, a force pair 110.  3 scans with
    the default rule, 18 near the fixed point (12 with the learned guess).
    Gravity: about 500 (as written) to 2500 (third order, tight acceptance)
    interactions of 92 and 200 operations per leaf of 2.5 particles."""
    kind = case["kind"]
    if kind == "sort":
        n, cells = case["n"], 1 << (3 * case["cell_power"])
        return {"bytes": 16 * n + 8 * n + 8 * cells, "flops": 9 * n}
    if kind == "train":
        s = case["steps"] * case["batch"]
        return {"bytes": 64 * s, "flops": 6 * 4928 * s}
    n = case["n"]
    if kind == "density":
        return {"bytes": (2 * 16 + 69) * n, "flops": 63 * (18 * 18 + 54) * n}
    form = case.get("form", "written")
    gravity = n / 2.5 * {"written": 500 * 92, "near": 700 * 92, "precision": 2500 * 200}[form]
    if kind == "nbody":
        return {"bytes": (16 + 48 + 36) * n, "flops": gravity}
    # individual timesteps of up to 4 rungs: about 15% of the particles in a step
    active = 0.15 if case.get("rungs", 0) else 1.0
    scans = 3 if kind == "frame" else (12 if case["learned"] else 18)
    hydro = 63 * (18 * scans + 54 + 110) * n
    return {"bytes": (20 + 92 + active * (69 + 93)) * n, "flops": active * (hydro + gravity)}


# -------------------------------------------------------- the same in 64 bits
def exact(case, seed):
    if case["kind"] == "nbody" and case["form"] != "written":
        # as written, the field is not that of the particles: leaves accept any source however near
        return _exact_nbody(case, seed)
    if case["kind"] == "density":
        return _exact_density(case, seed)
    return None


def _exact_nbody(case, seed):
    """One kick and drift in the field of the direct sum over all particles,
    each pair softened within GRAVITY_SMOOTHING_LENGTH by the polynomial
    whose derivatives the expansions use."""
    G, eps, dt = 6.67e-5, 0.04, DT_TICKS * 32.0 / 65536
    ic = two_bodies(case["n"], seed)
    x = torch.from_numpy(ic["pos"][:, :3].astype(np.float64)).cuda()
    m = torch.from_numpy(ic["mass"].astype(np.float64)).cuda()
    acc, phi = torch.empty_like(x), torch.empty_like(m)
    rows = max(1, (1 << 28) // x.shape[0])
    for i in range(0, x.shape[0], rows):
        d = [x[i:i + rows, None, k] - x[None, :, k] for k in range(3)]
        r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
        r2[r2 == 0] = math.inf  # the particle itself
        inv = r2.rsqrt_()
        w = inv ** 3
        p = inv.clone()
        near = (inv > 1.0 / eps).nonzero(as_tuple=True)
        u = 1.0 / (inv[near] * eps)
        p[near] = (((((((-3 * u + 15) * u - 28) * u + 21) * u) * u - 7) * u) * u + 3) / eps
        w[near] = -(((((-21 * u + 90) * u - 140) * u + 84) * u) * u - 14) * u / eps ** 2 * inv[near]
        w *= m
        for k in range(3):
            acc[i:i + rows, k] = -(w * d[k]).sum(1)
        phi[i:i + rows] = -G * (p @ m)
    a = G * acc
    v = torch.from_numpy(ic["vel"][:, :3].astype(np.float64)).cuda()
    pos = torch.cat([x + dt * v + 0.5 * dt * dt * a, m[:, None]], 1)
    out = {"pos": pos, "vel": torch.cat([v + dt * a, torch.zeros_like(m)[:, None]], 1), "gravnorm": acc.norm(dim=1)}
    if case["form"] == "precision":
        out["potential"] = phi
    return out


def _pairs(x, reach):
    """(i, j, r) of every ordered pair closer than i's reach, itself included."""
    size = float(reach.max())
    cell = ((x - x.min(0).values) / size).floor().long() + 1
    dims = cell.max(0).values + 2
    key = (cell[:, 0] * dims[1] + cell[:, 1]) * dims[2] + cell[:, 2]
    key, order = key.sort()
    found = []
    for dx in (-1, 0, 1):
        for dy in (-1, 0, 1):
            for dz in (-1, 0, 1):
                other = key + (dx * dims[1] + dy) * dims[2] + dz
                first = torch.searchsorted(key, other)
                count = torch.searchsorted(key, other, right=True) - first
                a = torch.repeat_interleave(torch.arange(len(key), device=x.device), count)
                b = torch.arange(len(a), device=x.device) - (count.cumsum(0) - count)[a] + first[a]
                i, j = order[a], order[b]
                r = (x[i] - x[j]).norm(dim=1)
                keep = r < reach[i]
                found.append((i[keep], j[keep], r[keep]))
    return tuple(torch.cat(t) for t in zip(*found))


def _exact_density(case, seed):
    """h at the fixed point of h = 1.2348 (m / rho(h))^(1/3) by Newton's
    method, and rho and the grad-h factor there."""
    ic = two_bodies(case["n"], seed)
    x = torch.from_numpy(ic["pos"][:, :3].astype(np.float64)).cuda()
    m = torch.from_numpy(ic["mass"].astype(np.float64)).cuda()
    h = torch.from_numpy(ic["h"].astype(np.float64)).cuda()
    reach = 2 * 2.2 * h
    i, j, r = _pairs(x, reach)
    mj = m[j]

    def sums(h):
        hi = h[i]
        q = r / hi
        a, b = (2 - q).clamp(min=0), (1 - q).clamp(min=0)
        w = (0.25 * a ** 3 - b ** 3) / (math.pi * hi ** 3)
        dw = -3 / (math.pi * hi ** 4) * (0.25 * a * a * (a - q) - b * b * (b - q))
        rho = torch.zeros_like(h).index_add_(0, i, mj * w)
        return rho, torch.zeros_like(h).index_add_(0, i, mj * dw)

    for it in range(40):
        rho, drho = sums(h)
        want = (1.2348 * (m / rho) ** (1.0 / 3.0)).clamp(max=1.0)
        if it < 25:
            h = 0.5 * (h + want)
        else:
            h = (h - (h - want) / (1 + want * drho / (3 * rho))).clamp(min=0.2 * h, max=2.0 * h)
    if bool((2 * h > reach).any()):
        return None  # the pair list does not hold every neighbour
    rho, drho = sums(h)
    return {"h": h, "rho": rho, "gradterm": 1 / (1 + h / (3 * rho) * drho), "pressure": None, "soundspeed": None,
            "balsara": None}
