"""Shares of the block pairs where the default blocks depend on how much work
one share has: below 1e8 N^2 / shares the finer blocks, bit for bit the plan
that names them, and past it blocks of 512. The shares add up to the force
within the path's tolerance either way."""
import ctypes

import numpy as np
import pytest

from conftest import EPS2
from gpu_util import dev, host, ptr
from oracle_lib import force_errors

from nbody_amd import _native, ics

pytestmark = pytest.mark.gpu

TOL_MAX, TOL_RMS = 1e-5, 1e-6


def shares_of(d_pm, n, shares, **opt):
    o = _native.Options.make(**opt) if opt else None
    out = []
    for k in range(shares):
        f = dev(np.full((n, 4), -9.0, np.float64))
        _native.check(_native.lib().nbody_hip_force_pair_share(ptr(f), ptr(d_pm), EPS2, n, k, shares,
                                                               ctypes.byref(o) if o else None, None), "share")
        out.append(host(f))
    return out


def test_blocks_of_a_share_within_a_slot_budget():
    """Too small a budget for the fine blocks' slots: blocks of 512, in bands."""
    n, shares = 8192, 4
    pm, _ = ics.random_unit_bodies(n, seed=62)
    d = dev(pm)
    for budget, shape in ((12 * 64 * 64 * 128, (2, 128)), (12 * 64 * 64 * 128 - 1, (8, 512)), (1 << 18, (8, 512))):
        got = shares_of(d, n, shares, slot_bytes=budget)
        named = shares_of(d, n, shares, slot_bytes=budget, i_per_lane=shape[0], jslice=shape[1])
        for a, b in zip(got, named):
            assert np.array_equal(a.view(np.uint64), b.view(np.uint64)), (budget, shape)


@pytest.mark.parametrize("n,shares,shape", [(5119, 2, (2, 128)), (6000, 2, (2, 128)), (8192, 8, (2, 128)),
                                            (12000, 2, (2, 128)), (16383, 4, (2, 128)), (16384, 4, (4, 256)),
                                            (24576, 8, (4, 256)), (16384, 2, (8, 512)), (24576, 4, (8, 512))])
def test_default_blocks_of_a_share(oracle, n, shares, shape):
    pm, _ = ics.random_unit_bodies(n, seed=61)
    d = dev(pm)
    got = shares_of(d, n, shares)
    named = shares_of(d, n, shares, i_per_lane=shape[0], jslice=shape[1])
    for a, b in zip(got, named):
        assert np.array_equal(a.view(np.uint64), b.view(np.uint64)) and np.all(a[:, 3] == -9.0)
    some = np.arange(0, n, max(1, n // 2000))
    mx, rms = force_errors(sum(a[some, :3] for a in got), oracle.fp64_forces(pm, EPS2, some))
    assert mx <= TOL_MAX and rms <= TOL_RMS, (n, shares, mx, rms)
