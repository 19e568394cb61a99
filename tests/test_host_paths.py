"""Host paths of csrc/plife.hip on a HIP runtime made of host memory
(host_paths.cpp): what a run on a device cannot show."""
from __future__ import annotations

import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("host_paths")
    obj, exe = str(d / "host_paths.o"), str(d / "host_paths")
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "--offload-arch=gfx950", "-fuse-cuid=none", "-O1",
                    "-std=c++17", "-fPIC", "-c", "-o", obj, os.path.join(HERE, "host_paths.cpp")], check=True)
    subprocess.run(["g++", "-o", exe, obj, "-lpthread"], check=True)
    return exe


CASES = ["failed_growth", "measured_cells_are_no_step", "stopped_update_keeps_the_last_step",
         "new_state_forgets_measured_work", "extreme_forces_take_the_literal_law",
         "empty_noalloc_step_reads_no_matrix", "lds_limit_is_raised_ahead",
         "kept_homes_follow_the_plan", "timed_steps_do_not_wait"]


@pytest.mark.parametrize("case", CASES)
def test_host_path(program, case):
    r = subprocess.run([program, case], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
