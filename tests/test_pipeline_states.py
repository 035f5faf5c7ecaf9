"""What Pipeline promises its caller, against a played library (tests/native/pipeline_states.cpp): no device needed."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("pipeline") / "pipeline_states")
    subprocess.run(["g++", "-std=c++14", "-O1", "-Wall", "-Wextra", "-Werror", "-I" + os.path.join(ROOT, "visualmesh_amd", "cpp"), "-I" + os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "native", "pipeline_states.cpp"), "-o", out, "-pthread"], check=True)
    return out


def _run(program, what):
    done = subprocess.run([program, what], capture_output=True, text=True, timeout=60)
    assert done.returncode == 0 and done.stdout.strip() == "ok", done.stdout + done.stderr


def test_results_stay_until_two_more_calls(program):
    _run(program, "held")


def test_batches_without_frames(program):
    _run(program, "empty")


def test_a_step_that_fails(program):
    _run(program, "failures")
