"""Stepping in HBM with the integrator in the force's last launch, and graphs
of several steps: runs of every length against the same steps launched one by
one, and one step against the force entry and the integrator called apart,
all bit for bit (the same operations in the same order), for each plan family:
the one-launch kernel (which steps into a second position buffer), split and
whole symmetric block pairs, column bands, FP64 accumulation, LDS slices.
"""
import ctypes

import numpy as np
import pytest

from gpu_util import dev, force_buffer, host, ptr

from nbody_amd import _native, ics
from nbody_amd.engine import BATCHED, BATCHED_GRAPH, Ensemble, System

pytestmark = pytest.mark.gpu

PLANS = [(1, {}), (700, {}), (5001, {}), (10240, {}), (10241, {}), (12000, {}), (5001, dict(compensated=2)),
         (5001, dict(variant=_native.LDS, i_per_lane=2, jslice=1024)), (5001, dict(compensated=1)),
         (9 * 512 + 37, dict(variant=_native.SYMMETRIC, i_per_lane=8, jslice=512, slot_bytes=12 * 512 * 20))]
IDS = [f"{n}-{'-'.join(f'{k}{v}' for k, v in o.items())}" for n, o in PLANS]


def bits(a):
    return np.ascontiguousarray(a).view(np.uint32)


@pytest.mark.parametrize("n,opt", PLANS, ids=IDS)
def test_graphs_match_single_steps(n, opt):
    pm, vm = ics.plummer(n, seed=3)
    kw = dict(dt=0.002, damping=0.97, **opt)
    with System(pm, vm, 0.01, **kw) as a, System(pm, vm, 0.01, **kw) as b:
        for steps in (1, 16, 3, 35, 0, 17, 2):
            a.run(steps, graph=True)
            b.run(steps, graph=False)
            for x, y in zip(a.read(), b.read()):
                assert np.array_equal(bits(x), bits(y)), (n, opt, steps)


@pytest.mark.parametrize("n,opt", PLANS, ids=IDS)
def test_step_is_force_then_integrate(n, opt):
    pm, vm = ics.random_unit_bodies(n, seed=5)
    L = _native.lib()
    o = _native.Options.make(**opt)
    d_pm, d_vm, f = dev(pm), dev(vm), force_buffer(n)
    with System(pm, vm, 0.01, dt=0.002, damping=0.97, **opt) as s:
        for _ in range(3):
            s.run(1)
            _native.check(L.nbody_hip_force(ptr(f), ptr(d_pm), 0.01, n, 0, n, ctypes.byref(o), None), "force")
            _native.check(L.nbody_hip_integrate(ptr(d_pm), ptr(d_vm), ptr(f), 0.002, 0.97, n, None), "integrate")
            p, v, g = s.read()
            assert np.array_equal(bits(p), bits(host(d_pm))) and np.array_equal(bits(v), bits(host(d_vm)))
            assert np.array_equal(bits(g[:, :3]), bits(host(f)[:, :3])) and np.all(g[:, 3] == 0.0)


def test_ensemble_graphs_match_single_steps():
    systems = [ics.plummer(int(n), seed=50 + k) for k, n in enumerate((1, 300, 512, 1500, 4000))]
    kw = dict(dt=0.002, damping=0.97)
    with Ensemble(systems, 0.01, **kw) as a, Ensemble(systems, 0.01, **kw) as b:
        for steps in (1, 16, 5, 34):
            a.run(steps, BATCHED_GRAPH)
            b.run(steps, BATCHED)
            for x, y in zip(a.read(), b.read()):
                assert np.array_equal(bits(x), bits(y)), steps
