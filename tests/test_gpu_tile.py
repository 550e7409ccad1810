"""The one-launch plan of small evaluations (whole systems up to 10240 bodies,
small i ranges): sizes at the edges of its workgroups, of a
step of its lane groups and of its 2048-body chunks, one for each of its
shapes, against the FP64 oracle; i ranges; masses that change in the middle
of a chunk and after a whole chunk of one mass.

Tolerance: the path's own (max 1e-5, RMS 1e-6 per body): a lane adds at most
N / 128 terms (80 at N = 10240), 8 or 16 lanes are added pairwise and the 16
waves in FP64.
"""
import ctypes

import numpy as np
import pytest
import torch

from conftest import EPS2
from gpu_util import dev, force_buffer, host, ptr, run_force
from oracle_lib import force_errors

from nbody_amd import _native, algorithms, ics
from nbody_amd.engine import System

pytestmark = pytest.mark.gpu

TOL_MAX, TOL_RMS = 1e-5, 1e-6


def plan(n, count, **opt):
    o, out = _native.Options.make(**opt), _native.Options()
    _native.check(_native.lib().nbody_hip_plan(n, count, ctypes.byref(o), ctypes.byref(out)), "plan")
    return out


@pytest.mark.parametrize("n", [1, 2, 3, 5, 255, 257, 1000, 2047, 2049, 2500, 4097, 6001, 7000, 9001, 10239, 10240])
@pytest.mark.parametrize("masses", ["unequal", "one", "heavier late", "zero late"])
def test_sizes_and_masses(oracle, n, masses):
    pm, _ = ics.random_unit_bodies(n, seed=41)
    if masses != "unequal":
        pm[:, 3] = 0.37
    if masses == "heavier late":
        pm[n - 1, 3] = 0.6
    if masses == "zero late":
        pm[n // 2:, 3] = 0.0
    p = plan(n, n)
    assert p.variant == _native.LDS and p.i_per_lane == 0 and p.jslice == 0
    d = dev(pm)
    f = run_force(d, EPS2)
    assert np.all(f[:, 3] == -7.0)
    again = run_force(d, EPS2)
    assert np.array_equal(f.view(np.uint32), again.view(np.uint32))
    f64 = oracle.fp64_forces(pm, EPS2)
    felt = np.any(f64 != 0.0, axis=1)  # bodies that any other body pulls
    assert np.all(f[~felt, :3] == 0.0)
    if felt.any():
        mx, rms = force_errors(f[felt], f64[felt])
        assert mx <= TOL_MAX and rms <= TOL_RMS, (n, masses, mx, rms)


@pytest.mark.parametrize("n,base,count", [(5000, 0, 1), (5000, 4999, 1), (5000, 123, 1777), (16384, 4096, 6400),
                                          (30000, 7, 3000), (65536, 60000, 100), (65536, 1, 20000)])
def test_i_ranges(oracle, n, base, count):
    """Ranges, in one launch or (the last two) in slices, against the oracle,
    and with a mass scaled by a power of two exactly (one mass and unequal
    masses)."""
    assert (plan(n, count).jslice == 0) == (n < 60000)
    for one in (False, True):
        pm, _ = ics.random_unit_bodies(n, seed=42)
        if one:
            pm[:, 3] = 1.0
        f = run_force(dev(pm), EPS2, base=base, count=count)
        mx, rms = force_errors(f, oracle.fp64_forces(pm, EPS2, np.arange(base, base + count)))
        assert mx <= TOL_MAX and rms <= TOL_RMS, (n, base, count, one, mx, rms)
        pm[:, 3] *= 0.25
        g = run_force(dev(pm), EPS2, base=base, count=count)
        assert np.array_equal(0.25 * f[:, :3], g[:, :3])


def test_other_options_keep_their_plans():
    """What fixes a shape, compensates or takes a Newton step runs as before,
    and so does a system past the limit."""
    assert plan(4096, 4096, compensated=1).variant == _native.SYMMETRIC
    assert plan(4096, 4096, compensated=2).variant == _native.SYMMETRIC
    assert plan(4096, 4096, newton=1).variant == _native.SYMMETRIC
    assert plan(4096, 4096, slot_bytes=1 << 20).variant == _native.SYMMETRIC
    assert plan(10241, 10241).variant == _native.SYMMETRIC
    assert plan(4096, 4096, variant=_native.LDS, i_per_lane=1).jslice > 0
    assert plan(4096, 4096, variant=_native.LDS, compensated=1).jslice > 0
    assert plan(98304, 12288).jslice > 0 and plan(60000, 15000).jslice > 0


def test_empty_range_writes_nothing():
    pm, _ = ics.random_unit_bodies(100, seed=43)
    d, f = dev(pm), force_buffer(1)
    rc = _native.lib().nbody_hip_force(ptr(f), ptr(d), EPS2, 100, 50, 0, None, None)
    assert rc == 0 and np.all(np.isnan(host(f)[:, :3]))


@pytest.mark.parametrize("slices", [1, 2, 3, 4, 5, 7, 16, 17, 33])
@pytest.mark.parametrize("comp", [0, 1])
def test_slice_sum(oracle, slices, comp):
    """The sum over j slices, a quarter of them per wave, at slice counts below,
    at and past the waves and the loads in flight, on a body count that is no
    multiple of 64."""
    n = 256 * slices
    pm, _ = ics.random_unit_bodies(n, seed=44)
    f = run_force(dev(pm), EPS2, base=1, count=min(n - 1, 777), variant=_native.LDS, i_per_lane=1, jslice=256,
                  compensated=comp)
    f64 = oracle.fp64_forces(pm, EPS2, np.arange(1, 1 + f.shape[0]))
    mx, rms = force_errors(f, f64)
    assert mx <= TOL_MAX and rms <= TOL_RMS, (slices, comp, mx, rms)
    assert np.all(f[:, 3] == -7.0)


@pytest.mark.parametrize("n", [1, 300, 10240, 10241])
def test_table_entry_returns_when_the_forces_are_there(n):
    """The table's synchronous entry, whose end event is the one launch itself
    (N <= 10240) or a marker behind two: bit for bit the queued entry's forces,
    read straight from host memory, with no further wait."""
    pm, _ = ics.random_unit_bodies(n, seed=42)
    d = dev(pm)
    want = run_force(d, EPS2)
    f = torch.empty(n, 4, pin_memory=True)
    for _ in range(3):
        f.fill_(-7.0)
        ms = algorithms.find("HIP")(f.data_ptr(), d.data_ptr(), EPS2, n)
        assert np.array_equal(f.numpy().view(np.uint32), want.view(np.uint32))
        assert 0.0 < ms < 1e3


@pytest.mark.parametrize("n,base,count", [(1, 0, 1), (2, 0, 2), (255, 0, 255), (300, 0, 300), (1023, 0, 1023),
                                          (2049, 0, 2049), (4097, 0, 4097), (5000, 4999, 1), (5000, 123, 1777),
                                          (16384, 4096, 2048)])
@pytest.mark.parametrize("masses", ["unequal", "one", "heavier late"])
def test_fp64_accumulation(oracle, n, base, count, masses):
    """The one-launch kernel with every term added in FP64: below 1024 bodies,
    the LDS variant's whole systems, i ranges."""
    pm, _ = ics.random_unit_bodies(n, seed=43)
    if masses != "unequal":
        pm[:, 3] = 0.37
    if masses == "heavier late":
        pm[n - 1, 3] = 0.6
    opt = dict(compensated=2, variant=_native.LDS if count == n >= 1024 else _native.AUTO)
    p = plan(n, count, **opt)
    assert p.variant == _native.LDS and p.i_per_lane == 0 and p.jslice == 0 and p.compensated == 2
    d = dev(pm)
    f = run_force(d, EPS2, base, count, **opt)
    again = run_force(d, EPS2, base, count, **dict(opt, variant=p.variant, i_per_lane=p.i_per_lane, jslice=p.jslice))
    assert np.array_equal(f.view(np.uint32), again.view(np.uint32))
    assert np.all(f[:, 3] == -7.0)
    if n == 1:
        assert np.all(f[:, :3] == 0.0)
        return
    mx, rms = force_errors(f, oracle.fp64_forces(pm, EPS2)[base:base + count])
    assert mx <= TOL_MAX and rms <= TOL_RMS, (n, masses, mx, rms)


@pytest.mark.parametrize("n", [1, 700])
def test_fp64_accumulation_steps(n):
    """A step in that launch against the force entry and the integrator apart."""
    pm, vm = ics.random_unit_bodies(n, seed=44)
    o = _native.Options.make(compensated=2)
    L = _native.lib()
    d_pm, d_vm, f = dev(pm), dev(vm), force_buffer(n)
    with System(pm, vm, EPS2, dt=0.002, damping=0.97, compensated=2) as s:
        for steps in (1, 1, 17):
            s.run(steps)
            for _ in range(steps):
                _native.check(L.nbody_hip_force(ptr(f), ptr(d_pm), EPS2, n, 0, n, ctypes.byref(o), None), "force")
                _native.check(L.nbody_hip_integrate(ptr(d_pm), ptr(d_vm), ptr(f), 0.002, 0.97, n, None), "integrate")
            p, v, g = s.read()
            assert np.array_equal(p.view(np.uint32), host(d_pm).view(np.uint32))
            assert np.array_equal(v.view(np.uint32), host(d_vm).view(np.uint32))
            assert np.array_equal(g[:, :3].copy().view(np.uint32), host(f)[:, :3].copy().view(np.uint32))
