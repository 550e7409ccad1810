"""The workloads this library is timed on, each one pass through its public
entry points on inputs made from a seed.

A case is a dict of plain values:

    kind    "force":    nbody_hip_force on the current stream (asynchronous)
            "table":    the algorithm-table entry HIP (synchronous)
            "share":    nbody_hip_force on one GPU's i range of a larger run
            "system":   device-resident stepping of one system, state read back
            "ensemble": batched stepping of many systems, state read back
    n       bodies (ensemble: the largest system)
    ic      "ball" (uniform ball, unit masses), "plummer" (Plummer sphere, m = 1/N)
            or "random" (a cube with masses in [0.5, 1), as the reference driver's)
    acc     the compensated option (-1 the library's choice, 2 FP64 accumulation)
    shares, share    share: how many GPUs, and which one of them this is
    steps            system, ensemble: steps per pass
    count, n_lo      ensemble: systems, and the smallest one's bodies

The force is f_i = sum_j m_j (x_j - x_i) / (|x_j - x_i|^2 + eps2)^(3/2).
"""
import ctypes
import math

import numpy as np
import torch

from nbody_amd import _native, algorithms
from nbody_amd.engine import BATCHED_GRAPH, Ensemble, System

DEVICE = "cuda"
EPS2 = {"ball": 0.01, "plummer": 0.0001, "random": 0.01}
STEP_EPS2, DT, DAMPING = 0.01, 0.002, 1.0  # stepping: a virialised Plummer sphere, softly softened


def listed():
    return [
        # the smallest systems a driver steps: all launch and latency
        {"name": "force_256_random", "kind": "force", "n": 256, "ic": "random", "acc": -1},
        # a small odd size through the reference driver's table call
        {"name": "table_1000_random", "kind": "table", "n": 1000, "ic": "random", "acc": -1},
        # the reference driver's smoke run (--bodies 4)
        {"name": "table_4096_random", "kind": "table", "n": 4096, "ic": "random", "acc": -1},
        # the single-system crosscheck workload
        {"name": "force_16384_ball", "kind": "force", "n": 16384, "ic": "ball", "acc": -1},
        # a mid size that no block divides, masses 1/N
        {"name": "force_49999_plummer", "kind": "force", "n": 49999, "ic": "plummer", "acc": -1},
        # the headline workload, and the same size with the reference driver's unequal masses
        {"name": "force_98304_ball", "kind": "force", "n": 98304, "ic": "ball", "acc": -1},
        {"name": "table_98304_random", "kind": "table", "n": 98304, "ic": "random", "acc": -1},
        # the largest single system
        {"name": "force_1048576_plummer", "kind": "force", "n": 1048576, "ic": "plummer", "acc": -1},
        # FP64 accumulation, for callers that need the error bound on every evolved state
        {"name": "force64_65536_random", "kind": "force", "n": 65536, "ic": "random", "acc": 2},
        # one GPU's eighth of the headline system, split by i range as the reference's multi-GPU path
        {"name": "share_98304_of_8", "kind": "share", "n": 98304, "ic": "ball", "acc": -1, "shares": 8, "share": 3},
        # a small system stepped in HBM, as a simulation loop does between two outputs
        {"name": "system_8192_plummer", "kind": "system", "n": 8192, "ic": "plummer", "acc": -1, "steps": 32},
        # the batched ensemble: 512 systems of 256 .. 16384 bodies
        {"name": "ensemble_512", "kind": "ensemble", "n": 16384, "ic": "plummer", "acc": -1, "count": 512,
         "n_lo": 256, "steps": 8},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["force", "force", "force", "table", "table", "force64", "share", "system", "system",
                       "ensemble"])
    ic = rng.choice(["ball", "plummer", "random"])
    if kind == "force64":
        return {"kind": "force", "n": _log_int(rng, 256, 131072), "ic": ic, "acc": 2}
    if kind == "share":
        shares = rng.randint(2, 8)
        return {"kind": "share", "n": _log_int(rng, 16384, 262144), "ic": ic, "acc": -1, "shares": shares,
                "share": rng.randrange(shares)}
    if kind == "system":
        n = _log_int(rng, 256, 131072)
        return {"kind": "system", "n": n, "ic": "plummer", "acc": -1, "steps": rng.randint(8, 32)}
    if kind == "ensemble":
        return {"kind": "ensemble", "n": _log_int(rng, 1024, 16384), "ic": "plummer", "acc": rng.choice([-1, -1, 2]),
                "count": _log_int(rng, 8, 512), "n_lo": _log_int(rng, 64, 1024), "steps": rng.randint(4, 8)}
    return {"kind": kind, "n": _log_int(rng, 64, 524288 if kind == "force" else 131072), "ic": ic, "acc": -1}


# ---- inputs ------------------------------------------------------------------


def _in_ball(n, g):
    """n points uniform in the unit ball."""
    d = torch.randn(n, 3, generator=g, device=DEVICE)
    r = torch.rand(n, 1, generator=g, device=DEVICE) ** (1.0 / 3.0)
    return d / d.norm(dim=1, keepdim=True) * r


def _bodies(n, ic, seed):
    """(posMass, velInvMass), float4 records on the GPU."""
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(seed) * 1000003 + n)
    pm = torch.empty(n, 4, device=DEVICE)
    vm = torch.empty(n, 4, device=DEVICE)
    if ic == "ball":
        pm[:, :3] = _in_ball(n, g) * (1.54 * (n / 16384.0) ** (1.0 / 3.0))
        pm[:, 3] = 1.0
        vm[:, :3] = _in_ball(n, g)
        vm[:, 3] = 1.0
    elif ic == "plummer":
        # scale radius 1 and total mass 1, cut at the radius that holds 99.9 % of the mass
        x = torch.rand(n, 1, generator=g, device=DEVICE) * 0.999
        r = (x.clamp_min(1e-9) ** (-2.0 / 3.0) - 1.0).rsqrt()
        d = torch.randn(n, 3, generator=g, device=DEVICE)
        pm[:, :3] = d / d.norm(dim=1, keepdim=True) * r
        pm[:, 3] = 1.0 / n
        # isotropic velocities of the sphere's local dispersion, 1 / (6 sqrt(1 + r^2)) per component
        vm[:, :3] = torch.randn(n, 3, generator=g, device=DEVICE) * (1.0 / (6.0 * (1.0 + r * r).sqrt())).sqrt()
        vm[:, 3] = 1.0
    else:
        pm[:, :3] = (torch.rand(n, 3, generator=g, device=DEVICE) * 2.0 - 1.0) * 0.9
        pm[:, 3] = torch.rand(n, generator=g, device=DEVICE) * 0.5 + 0.5
        vm[:, :3] = (torch.rand(n, 3, generator=g, device=DEVICE) * 2.0 - 1.0) * 8.0
        vm[:, 3] = 1.0 / pm[:, 3]
    return pm, vm


def _sizes(case, seed):
    """The ensemble's sizes, log-uniform in [n_lo, n]. They belong to the case,
    not to the seed, so every seed is the same amount of work."""
    rng = np.random.default_rng(case["count"] * 7919 + case["n"] + case["n_lo"])
    lo, hi = math.log(case["n_lo"]), math.log(case["n"] + 1)
    return np.exp(rng.uniform(lo, hi, size=case["count"])).astype(np.int64).clip(case["n_lo"], case["n"]).tolist()


def _ensemble_bodies(case, seed):
    return [_bodies(n, "plummer", seed * 4099 + k) for k, n in enumerate(_sizes(case, seed))]


def _share_range(case):
    n, g, k = case["n"], case["shares"], case["share"]
    lo, hi = n * k // g, n * (k + 1) // g
    return lo, hi - lo


# ---- one pass ----------------------------------------------------------------


def prepare(case, seed):
    kind = case["kind"]
    opt = _native.Options.make(compensated=case["acc"]) if case["acc"] >= 0 else None
    if kind in ("force", "table", "share"):
        pm, _ = _bodies(case["n"], case["ic"], seed)
        base, count = _share_range(case) if kind == "share" else (0, case["n"])
        force = torch.zeros(count, 4, device=DEVICE)
        state = {"kind": kind, "pm": pm, "force": force, "n": case["n"], "base": base, "count": count,
                 "eps2": EPS2[case["ic"]], "opt": opt}
        if kind == "table":
            state["entry"] = algorithms.find("HIP")
        return state
    extra = {"compensated": case["acc"]} if case["acc"] >= 0 else {}
    if kind == "system":
        pm, vm = _bodies(case["n"], case["ic"], seed)
        handle = System(pm.cpu().numpy(), vm.cpu().numpy(), STEP_EPS2, dt=DT, damping=DAMPING, **extra)
        total = case["n"]
    else:
        bodies = _ensemble_bodies(case, seed)
        handle = Ensemble([(p.cpu().numpy(), v.cpu().numpy()) for p, v in bodies], STEP_EPS2, dt=DT, damping=DAMPING,
                          **extra)
        total = handle.total
    # the program's own page-locked buffers for the state it reads back
    out = [torch.zeros(total, 4, pin_memory=True) for _ in range(3)]
    return _Stepping(kind, handle, case["steps"], out)


class _Stepping:
    """A stepping handle and the buffers its state is read into; closes the
    handle with itself."""

    def __init__(self, kind, handle, steps, out):
        self.kind, self.handle, self.steps, self.out = kind, handle, steps, out

    def __del__(self):
        self.handle.close()


def run(state):
    L = _native.lib()
    if isinstance(state, _Stepping):
        h, (pm, vm, force) = state.handle, state.out
        if state.kind == "system":
            h.run(state.steps)
            read = L.nbody_hip_system_read
        else:
            h.run(state.steps, BATCHED_GRAPH)
            read = L.nbody_hip_ensemble_read
        _native.check(read(h.h, pm.data_ptr(), vm.data_ptr(), force.data_ptr()), "read")
        return {"pos_mass": pm, "vel_inv_mass": vm, "force": force}
    if state["kind"] == "table":
        ms = state["entry"](state["force"].data_ptr(), state["pm"].data_ptr(), state["eps2"], state["n"])
        _native.check_ms(ms, "HIP")
        return state["force"]
    opt = ctypes.byref(state["opt"]) if state["opt"] is not None else None
    _native.check(L.nbody_hip_force(state["force"].data_ptr(), state["pm"].data_ptr(), state["eps2"], state["n"],
                                    state["base"], state["count"], opt, torch.cuda.current_stream().cuda_stream),
                  "nbody_hip_force")
    return state["force"]


def work(case):
    """One interaction of two bodies, in one direction, counts 20 flops (the
    reference's convention). Bytes: each record read once and written once."""
    n = case["n"]
    if case["kind"] == "share":
        count = _share_range(case)[1]
        return {"bytes": 16 * n + 16 * count, "flops": 20.0 * n * count}
    if case["kind"] == "system":
        # a step reads and writes positions and velocities and writes forces; the state is read back once
        return {"bytes": (80 * case["steps"] + 48) * n, "flops": 20.0 * n * n * case["steps"]}
    if case["kind"] == "ensemble":
        sizes = _sizes(case, 0)
        return {"bytes": (80 * case["steps"] + 48) * sum(sizes),
                "flops": 20.0 * sum(s * s for s in sizes) * case["steps"]}
    return {"bytes": 32 * n, "flops": 20.0 * n * n}


# ---- the same in 64 bits -----------------------------------------------------


def _f32(v):
    """The value a float argument holds once it is passed as a C float."""
    return float(np.float32(v))


def _force64(x, m, eps2, lo=0, count=None):
    """Forces on bodies [lo, lo + count) in FP64, (count, 4) with w = 0."""
    n = x.shape[0]
    count = n if count is None else count
    out = torch.zeros(count, 4, dtype=torch.float64, device=x.device)
    rows = max(1, min(count, (1 << 27) // n))
    d2 = torch.empty(rows, n, dtype=torch.float64, device=x.device)
    for a in range(0, count, rows):
        b = min(count, a + rows)
        xi = x[lo + a:lo + b]
        w = d2[:b - a]
        w.fill_(eps2)
        for c in range(3):
            d = x[None, :, c] - xi[:, None, c]
            w.addcmul_(d, d)
        w.rsqrt_()
        w.mul_(w * w).mul_(m[None, :])
        out[a:b, :3] = w @ x - xi * w.sum(dim=1, keepdim=True)
    return out


def _steps64(pm, vm, eps2, dt, damping, steps):
    x, m = pm[:, :3].double().contiguous(), pm[:, 3].double().contiguous()
    v, inv = vm[:, :3].double().contiguous(), vm[:, 3:].double()
    f = None
    for _ in range(steps):
        f = _force64(x, m, eps2)
        v = (v + inv * (f[:, :3] * dt)) * damping
        x = x + v * dt
    return torch.cat([x, m[:, None]], 1), torch.cat([v, inv], 1), f


def exact(case, seed):
    kind, n = case["kind"], case["n"]
    if work(case)["flops"] > 20.0 * 2.0e11:  # over about ten seconds of FP64 sums
        return None
    if kind in ("force", "table", "share"):
        pm, _ = _bodies(n, case["ic"], seed)
        lo, count = _share_range(case) if kind == "share" else (0, n)
        return _force64(pm[:, :3].double().contiguous(), pm[:, 3].double().contiguous(), _f32(EPS2[case["ic"]]), lo,
                        count)
    bodies = [_bodies(n, case["ic"], seed)] if kind == "system" else _ensemble_bodies(case, seed)
    got = [_steps64(p, v, _f32(STEP_EPS2), _f32(DT), _f32(DAMPING), case["steps"]) for p, v in bodies]
    pos, vel, force = (torch.cat([s[k] for s in got]) for k in range(3))
    return {"pos_mass": pos, "vel_inv_mass": vel, "force": force}
