"""The rounding of the library's own plan for mid-size systems, whose force is
summed from few block slots, against the finer blocks of 128 and 256 bodies.

Bound: the RMS error may not exceed that of the finer blocks. Each estimate
comes from 3 x 8192 components (standard deviation 0.45 %), so 3 % covers
their spread more than four times.
"""
import numpy as np
import pytest

from conftest import EPS2
from gpu_util import dev, run_force
from oracle_lib import force_errors

from nbody_amd import _native, ics

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [10241, 13312, 16383, 16384, 24576, 32767])
@pytest.mark.parametrize("opt", [{}, dict(newton=1), dict(slot_bytes=1 << 22)], ids=["plain", "newton", "bands"])
@pytest.mark.parametrize("masses", ["unequal", "one"])
def test_no_coarser_than_finer_blocks(oracle, n, opt, masses):
    if masses == "one":
        pm, _ = ics.uniform_ball(n, seed=51, radius=ics.ball_radius(n))
    else:
        pm, _ = ics.random_unit_bodies(n, seed=51)
    some = np.sort(np.random.default_rng(n).choice(n, 8192, replace=False))
    f64 = oracle.fp64_forces(pm, EPS2, some)
    ipl, block = (2, 128) if n < 16384 else (4, 256)
    d = dev(pm)
    _, rms = force_errors(run_force(d, EPS2, **opt)[some], f64)
    _, finer = force_errors(run_force(d, EPS2, variant=_native.SYMMETRIC, i_per_lane=ipl, jslice=block, **opt)[some], f64)
    assert rms <= 1.03 * finer, (n, opt, masses, rms, finer)
