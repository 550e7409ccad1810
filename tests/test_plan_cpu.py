"""The library's choice of plans, asked through its internal host functions
(tests/native/plan_probe.cpp, linked against the built library): no GPU call
is made."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT, TESTS

from nbody_amd import _native

ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="session")
def probe(tmp_path_factory):
    """probe(line, ...) -> one list of ints per line."""
    exe = str(tmp_path_factory.mktemp("plan") / "plan_probe")
    libdir = os.path.dirname(_native.LIB_PATH)
    subprocess.run([shutil.which("g++") or "g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__",
                    "-I", os.path.join(ROCM, "include"), "-I", os.path.join(ROOT, "nbody_amd", "csrc"),
                    "-I", os.path.join(ROOT, "include"), os.path.join(TESTS, "native", "plan_probe.cpp"), "-o", exe,
                    "-L", libdir, "-lnbody_hip", "-L", os.path.join(ROCM, "lib"), "-lamdhip64",
                    f"-Wl,-rpath,{libdir}", f"-Wl,-rpath,{os.path.join(ROCM, 'lib')}"], check=True)

    def ask(*lines):
        out = subprocess.run([exe], input="\n".join(lines) + "\n", stdout=subprocess.PIPE, check=True, text=True)
        return [[int(v) for v in row.split()] for row in out.stdout.splitlines()]

    return ask


@pytest.mark.parametrize("n_all", [160_000_000, 215_000_000, 1 << 28])
def test_lds_slices_of_the_largest_systems(probe, n_all):
    """The slice length stays within the system and the slices within a launch's
    second dimension, for whole systems, halves and single bodies."""
    counts = [n_all, n_all // 2, n_all // 3, 1000, 1]
    for n, (_, ipl, jslice, nslices, li) in zip(counts, probe(*[f"default {_native.LDS} {n_all} {n} 256"
                                                               for n in counts])):
        assert 1 <= jslice <= n_all and ipl in (1, 2) and (li == 0 or nslices == 1), (n, jslice)
        assert nslices == -(-n_all // jslice) and nslices <= 65535, (n, jslice, nslices)


@pytest.mark.parametrize("acc64", [0, 1])
def test_one_launch_shape_follows_the_cu_count(probe, acc64):
    """A quarter of the compute units with a quarter of the i bodies has the same
    number of workgroups per unit, so the same shape (480 bodies are whole
    workgroups of every shape)."""
    cases = [(n, 480 * k) for n in (1000, 4096, 8192, 30000) for k in range(1, 9)]
    whole = probe(*[f"tile {n} {4 * ni} {acc64} 256" for n, ni in cases])
    quarter = probe(*[f"tile {n} {ni} {acc64} 64" for n, ni in cases])
    assert whole == quarter
    assert len({tuple(s) for s in whole}) > 1


def test_tasks_per_block_pair_follow_the_cu_count(probe):
    """Block pairs are split to fill the chip: not where a small one is full anyway."""
    small, large, small_chip = [r[0] for r in probe("tasks 12288 256", "tasks 98304 256", "tasks 12288 16")]
    assert small > 1 and large == 1 and small_chip == 1


def test_lead_needs_every_task_resident(probe):
    """Four workgroups to a compute unit, or as many as the plan's cap leaves."""
    lines = {"1024 256 0": 1, "1025 256 0": 0, "512 256 2": 1, "513 256 2": 0, "768 256 3": 1, "769 256 3": 0,
             "1024 256 6": 1, "1025 256 6": 0, "128 32 0": 1, "129 32 0": 0}
    assert [r[0] for r in probe(*[f"lead {k}" for k in lines])] == list(lines.values())


def test_small_symmetric_blocks(probe):
    """Blocks of 128 up to 44 of them, with a Newton step up to 72; 512 past that."""
    sym = _native.SYMMETRIC
    shapes = {f"default {sym} {n} {n} 256": (2, 128) for n in (1024, 5121, 5632)}
    shapes |= {f"default {sym} {n} {n} 256": (8, 512) for n in (5633, 9216)}
    shapes |= {f"newton {sym} {n} {n} 256": (2, 128) for n in (1024, 5633, 9216)}
    shapes |= {f"newton {sym} {n} {n} 256": (8, 512) for n in (9217, 30000)}
    assert [(r[1], r[2]) for r in probe(*shapes)] == list(shapes.values())


def test_bodies_per_lane_of_large_lds_evaluations(probe):
    """Two past 5e8 pairs, but one with a Newton step and plain sums (the default up to N = 65536)."""
    lds = _native.LDS
    want = {f"default {lds} 30000 30000 256": 2, f"newton {lds} 30000 30000 256": 1,
            f"newton {lds} 65536 65536 256": 1, f"newton {lds} 98304 12288 256": 2, f"default {lds} 98304 12288 256": 2}
    assert [r[1] for r in probe(*want)] == list(want.values())


def test_autotune_times_the_default(probe):
    """The plan a call uses untuned is one of those the tuner compares, once."""
    cases = [(v, n) for v in (_native.AOS, _native.LDS, _native.DPP, _native.SGPR)
             for n in (1, 300, 1000, 8192, 16384, 30000, 65537, 98304, 1 << 20)]
    for (v, n), (count, same) in zip(cases, probe(*[f"tuned {v} {n} 256" for v, n in cases])):
        assert same >= 1 and count >= 1, (v, n)
        if n >= 8192 and v != _native.AOS:
            assert same == 1 and count >= 8, (v, n)
