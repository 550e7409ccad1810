"""The symmetric plan with 8 bodies per lane and blocks of 512, whose block
pairs are 1, 2 or 4 tasks each: every split at the sizes where a block, a
half or a tile is ragged, empty or alone, on unequal masses, one mass, and
one mass with one heavier body, against the FP64 oracle.

Tolerance: the path's own (max 1e-5, RMS 1e-6 per body): FP32 terms, sums of
at most 512 terms per lane, TwoSum over the slots.
"""
import numpy as np
import pytest

from conftest import EPS2
from gpu_util import dev, run_force
from oracle_lib import force_errors

from nbody_amd import _native, ics
from nbody_amd.engine import Ensemble

pytestmark = pytest.mark.gpu

TOL_MAX, TOL_RMS = 1e-5, 1e-6
SHAPE = dict(variant=_native.SYMMETRIC, i_per_lane=8, jslice=512)


@pytest.mark.parametrize("n", [2, 64, 511, 512, 513, 577, 1024, 1500, 3 * 512 + 320, 5003])
@pytest.mark.parametrize("split", [1, 2, 4])
@pytest.mark.parametrize("newton", [0, 1])
def test_every_split(oracle, n, split, newton):
    """A slot budget of `split` times one task's slots (12 bytes per body and
    block) allows at most that many tasks per pair."""
    nb = -(-n // 512)
    budget = split * 12 * 512 * nb * nb
    pm, _ = ics.random_unit_bodies(n, seed=31)
    one = pm.copy()
    one[:, 3] = 0.37
    heavier = one.copy()
    heavier[n // 2, 3] = 0.6
    for what, x in (("unequal", pm), ("one mass", one), ("one heavier", heavier)):
        d = dev(x)
        f = run_force(d, EPS2, slot_bytes=budget, newton=newton, **SHAPE)
        mx, rms = force_errors(f, oracle.fp64_forces(x, EPS2))
        assert mx <= TOL_MAX and rms <= TOL_RMS, (what, n, split, newton, mx, rms)
        assert np.all(f[:, 3] == -7.0)
        again = run_force(d, EPS2, slot_bytes=budget, newton=newton, **SHAPE)
        assert np.array_equal(f.view(np.uint32), again.view(np.uint32)), (what, n, split, newton)


def test_batched_blocks(oracle):
    """The batched form (one task per pair, taken from a queue): a last block
    of 1..8 tiles, ragged or full, beside none, one or two full blocks, with
    every kind of masses in one batch, and some of the systems alone."""
    sizes = sorted({b * 512 + 64 * t - r for b in (0, 1, 2) for t in range(1, 9) for r in (0, 1, 63)})
    systems = []
    for k, n in enumerate(sizes):
        pm, vm = ics.random_unit_bodies(n, seed=400 + k)
        if k % 3:
            pm[:, 3] = 0.37
        if k % 3 == 2:
            pm[n // 2, 3] = 0.6
        systems.append((pm, vm))

    def forces(which):
        with Ensemble(which, EPS2, dt=0.002) as e:
            e.run(1)
            return e.split(e.read()[2])

    got = forces(systems)
    for (pm, _), f in zip(systems, got):
        if len(pm) == 1:
            assert np.all(f[:, :3] == 0.0)
            continue
        mx, rms = force_errors(f, oracle.fp64_forces(pm, EPS2))
        assert mx <= TOL_MAX and rms <= TOL_RMS, (len(pm), mx, rms)
    for k in (0, 7, len(systems) - 1):
        assert np.array_equal(forces([systems[k]])[0].view(np.uint32), got[k].view(np.uint32)), sizes[k]


def test_fp64_blocks(oracle):
    """With FP64 accumulation (four waves share block Q's tiles, one or two to a
    wave): a last block of every tile count, ragged or full, and every kind of
    masses, in both shapes against the oracle; the batched form gives the bits
    of the 4-body one."""
    sizes = [1, 63, 64, 65] + [256 * b + 64 * t - r for b in (1, 2, 5) for t in (1, 2, 3, 4) for r in (0, 1, 63)]
    systems = []
    for k, n in enumerate(sizes):
        pm, vm = ics.random_unit_bodies(n, seed=600 + k)
        if k % 3:
            pm[:, 3] = 0.37
        if k % 3 == 2:
            pm[n // 2, 3] = 0.6
        systems.append((pm, vm))
    with Ensemble(systems, EPS2, dt=0.002, compensated=2) as e:
        e.run(1)
        batched = e.split(e.read()[2])
    for (pm, _), got in zip(systems, batched):
        for a in (4, 8):
            f = run_force(dev(pm), EPS2, variant=_native.SYMMETRIC, i_per_lane=a, jslice=64 * a, compensated=2)
            if len(pm) == 1:
                assert np.all(f[:, :3] == 0.0)
                continue
            mx, rms = force_errors(f, oracle.fp64_forces(pm, EPS2))
            assert mx <= TOL_MAX and rms <= TOL_RMS, (len(pm), a, mx, rms)
            if a == 4:
                assert np.array_equal(f[:, :3].view(np.uint32), np.ascontiguousarray(got[:, :3]).view(np.uint32)), len(pm)
