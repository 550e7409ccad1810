"""Launches of at most one wave per SIMD run the same chains without wave
priorities: the same bits as larger launches that run them with priorities,
for every kernel that has both."""
import numpy as np
import pytest

from conftest import EPS2
from gpu_util import dev, run_force

from nbody_amd import _native, ics

pytestmark = pytest.mark.gpu


def masses(pm, kind):
    if kind == "one":
        pm[:, 3] = 0.37
    return pm


@pytest.mark.parametrize("kind", ["unequal", "one"])
@pytest.mark.parametrize("comp", [0, 1])
@pytest.mark.parametrize("variant,ipl", [(v, i) for v in (_native.LDS, _native.SGPR, _native.DPP) for i in (1, 2, 4)] +
                         [(_native.DPP, 8)])
def test_ranges_of_one_sided_kernels(variant, ipl, comp, kind):
    """100 bodies in 20 slices (at most 80 waves) and the whole system (over 6000)."""
    n, base, count = 20011, 5001, 100
    pm, _ = ics.random_unit_bodies(n, seed=81)
    d = dev(masses(pm, kind))
    opt = dict(variant=variant, i_per_lane=ipl, jslice=1024, compensated=comp)
    whole = run_force(d, EPS2, **opt)[base:base + count]
    part = run_force(d, EPS2, base, count, **opt)
    assert np.array_equal(np.ascontiguousarray(whole[:, :3]).view(np.uint32),
                          np.ascontiguousarray(part[:, :3]).view(np.uint32))


@pytest.mark.parametrize("kind", ["unequal", "one"])
@pytest.mark.parametrize("shape", [(2, 128), (2, 512), (4, 256), (4, 512), (4, 1024), (8, 1024), (8, 2048)])
def test_symmetric_shapes(shape, kind):
    """A cap of one wave per SIMD against none."""
    n = 40013
    pm, _ = ics.random_unit_bodies(n, seed=82)
    d = dev(masses(pm, kind))
    opt = dict(variant=_native.SYMMETRIC, i_per_lane=shape[0], jslice=shape[1])
    alone = run_force(d, EPS2, waves_per_simd=1, **opt)
    many = run_force(d, EPS2, **opt)
    assert np.array_equal(alone.view(np.uint32), many.view(np.uint32))
