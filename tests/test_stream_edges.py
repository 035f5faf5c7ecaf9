"""Streams of batches behind other work of the same engine."""
import os
import subprocess

import pytest

from visualmesh_amd import native

pytestmark = pytest.mark.gpu


def test_behind_frames_never_run_and_runs_never_fetched(tmp_path):
    """tests/native/stream_edges.cpp"""
    root, lib_dir, exe = os.path.dirname(os.path.dirname(os.path.abspath(__file__))), os.path.dirname(native.HIP_LIB), str(tmp_path / "stream_edges")
    subprocess.run(["g++", "-std=c++14", "-O1", "-Wall", "-Wextra", "-Werror", "-I" + os.path.join(root, "visualmesh_amd", "cpp"), "-I" + os.path.join(root, "include"),
                    os.path.join(root, "tests", "native", "stream_edges.cpp"), "-L" + lib_dir, "-lvisualmesh_hip", "-Wl,-rpath," + lib_dir, "-pthread", "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout + out.stderr
