"""The device memory that the library's launches and captured graphs name, on
the CPU: tests/cpp/host_memory_check.cpp stands in for the HIP runtime and fails
on a launch or a replay that names freed memory."""
from __future__ import annotations

import subprocess
from pathlib import Path

import pytest

from fullc0ntact_amd import build

ROOT = Path(__file__).resolve().parents[1]


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = tmp_path_factory.mktemp("host_memory") / "host_memory_check"
    cmd = [build.hipcc(), "-x", "hip", "--offload-host-only", "-std=c++17", "-O1",
           f"-I{ROOT / 'include'}", f"-I{build.CSRC}",
           str(ROOT / "tests" / "cpp" / "host_memory_check.cpp"), f"-L{build.PKG}", "-lfc_dem",
           f"-Wl,-rpath,{build.PKG}", "-rdynamic", "-o", str(exe)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return exe


def holds(program, scenario):
    r = subprocess.run([str(program), scenario], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, f"{scenario}: {r.stdout}{r.stderr}"


# Runs before and after calls that grow the context's sort scratch (labels, a
# map, a larger system, a larger sort): up to 4,096 spheres, over that by radix
# sort, batches that sort by radix in updates and in runs, and by rows.
@pytest.mark.parametrize("scenario", ["system-small", "system-radix", "batch-cells",
                                      "batch-radix", "batch-rows"])
def test_captured_steps_and_grown_scratch(program, scenario):
    holds(program, scenario)


def test_an_error_is_returned_once(program):
    holds(program, "errors-once")


# A growth without memory: the callers' systems and batches keep their scratch.
@pytest.mark.parametrize("scenario", ["growth-fails-small", "growth-fails-radix",
                                      "no-room-for-both"])
def test_growth_that_fails(program, scenario):
    holds(program, scenario)


@pytest.mark.parametrize("scenario", ["row-tables-small", "row-tables"])
def test_captured_steps_and_new_row_tables(program, scenario):
    holds(program, scenario)


def test_runs_without_row_tables(program):
    holds(program, "no-row-tables")


def test_memory_is_cleared_on_the_stream_that_reads_it(program):
    holds(program, "clears")


def test_large_meshes_are_not_kept(program):
    holds(program, "large-meshes")


@pytest.mark.parametrize("scenario", ["no-cell-tables-small", "no-cell-tables"])
def test_grids_without_memory(program, scenario):
    holds(program, scenario)
