"""The synchronous table call leaves the stream finished: a synchronisation
right after a small system's call (one launch) waits for nothing, like one after
a larger system's (two launches). Medians of 300; a call that left its end
marker to the launch took three times as long."""
import statistics
import time

import pytest
import torch

from conftest import EPS2
from gpu_util import dev, force_buffer

from nbody_amd import algorithms, ics

pytestmark = pytest.mark.gpu


def sync_after_call(n):
    pm, _ = ics.random_unit_bodies(n, seed=71)
    d, f = dev(pm), force_buffer(n)
    entry = algorithms.find("HIP")
    took = []
    for k in range(350):
        assert entry(f.data_ptr(), d.data_ptr(), EPS2, n) > 0.0
        t0 = time.perf_counter()
        torch.cuda.synchronize()
        took.append(time.perf_counter() - t0)
    return statistics.median(took[50:])


@pytest.mark.parametrize("n", [256, 1000, 9000])
def test_nothing_is_left_to_wait_for(n):
    assert sync_after_call(n) <= 2.0 * sync_after_call(20000)
