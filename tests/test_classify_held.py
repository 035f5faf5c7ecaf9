"""A call's results left in the engine's block: C++ (Engine::classify_held) and C (vmh_engine_classify_held)."""
import ctypes as C
import math
import os
import subprocess

import numpy as np
import pytest

from visualmesh_amd import engine as eng
from visualmesh_amd import native
from visualmesh_amd import workloads as wl

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    lib_dir, exe = os.path.dirname(native.HIP_LIB), str(tmp_path_factory.mktemp("held") / "classify_held")
    subprocess.run(["g++", "-std=c++14", "-O1", "-Wall", "-Wextra", "-Werror", "-I" + os.path.join(ROOT, "visualmesh_amd", "cpp"), "-I" + os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "native", "classify_held.cpp"), "-L" + lib_dir, "-lvisualmesh_hip", "-Wl,-rpath," + lib_dir, "-pthread", "-o", exe], check=True)
    return exe


def test_the_interface_is_there(program):
    assert native.host().vmh_engine_classify_held


@pytest.mark.gpu
def test_cpp_calls(program):
    out = subprocess.run([program], capture_output=True, text=True, timeout=100)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout + out.stderr


@pytest.mark.gpu
def test_c_calls():
    engine = eng.Engine(wl.glorot_network(np.random.default_rng(3), [3, 16, 3], 6, wl.SELU), wl.RING6)
    lens, image = native.make_lens(320, 240, wl.EQUISOLID, 105.0, math.pi), wl.random_image(np.random.default_rng(5), 320, 240, 4)
    for k in (2.0, 0.4, 6.0):
        mesh, Hoc, r = eng.Mesh(wl.RING6, wl.SPHERE, 0.0949, 1.0, k, 6.0), np.ascontiguousarray(wl.make_hoc(1.0, math.radians(40.0), 0.0, 0.0), np.float32), native.Result()
        want = engine(mesh, Hoc, lens, image, wl.fourcc("RGBA"))
        native.host_check(native.host().vmh_engine_classify_held(engine.ptr, mesh.ptr, Hoc.ctypes.data_as(C.POINTER(C.c_float)), C.byref(lens), image.ctypes.data, wl.fourcc("RGBA"), C.byref(r)))
        V = r.n_visible
        for key, p, shape in (("px", r.pixel_coordinates, (V, 2)), ("gidx", r.global_indices, (V,)), ("nb", r.neighbourhood, (V + 1, 6)), ("cls", r.classifications, (V + 1, 3))):
            assert V > 0 and np.array_equal(np.ctypeslib.as_array(p, shape), want[key]), key
