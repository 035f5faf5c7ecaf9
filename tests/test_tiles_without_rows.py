"""Frames with many more candidates than visible nodes: most row tiles hold no rows, and nothing that lies there from earlier is worked on."""
import ctypes as C
import math

import numpy as np
import pytest

from visualmesh_amd import engine as eng
from visualmesh_amd import native
from visualmesh_amd import workloads as wl

pytestmark = pytest.mark.gpu

# a network for every family of layer kernels (widths, activation, precision); conv_mfma takes 40- and 48-wide rows, and 64-wide ones with tanh
CASES = {"mfma 64": ([3, 64, 64, 4], wl.TANH, native.FP32), "mfma 40, 48": ([3, 40, 48, 10, 3], wl.SELU, native.FP32),
         "rows": ([3, 72, 72, 5], wl.SELU, native.FP32), "lds, flow": ([3, 24, 32, 32, 16, 3], wl.RELU, native.FP32),
         "three parts, half tiles": ([3, 64, 64, 64, 4], wl.SELU, native.FP32), "three parts, tiles": ([3, 16, 32, 32, 3], wl.SELU, native.FP32),
         "pairs": ([3, 64, 64, 64, 4], wl.SELU, native.SPLIT), "bf16": ([3, 64, 64, 64, 64, 4], wl.SELU, native.BF16),
         # eight neighbours
         "mfma, nine slots": ([3, 40, 48, 24, 8, 40, 48, 4], wl.SELU, native.FP32), "lds, nine slots": ([3, 24, 24, 32, 4], wl.RELU, native.FP32)}


def _pointer(a):
    return a.ctypes.data_as(C.POINTER(C.c_int32))


def _results(batch, mesh, lens, poses, image, ranges, nn, n_out):
    lib, frames = native.hip(), (native.Frame * len(poses))()
    for f, Hoc, r in zip(frames, poses, ranges):
        f.mesh, f.lens, f.ranges, f.n_ranges = mesh, lens, _pointer(r), len(r)
        f.Rco = (C.c_float * 9)(*np.ascontiguousarray(Hoc[:3, :3].T, np.float32).ravel())
        f.image, f.fourcc = image.ctypes.data, wl.fourcc("RGBA")
    native.hip_check(lib.vmhip_batch_stage(batch, frames, len(poses), 1))
    raw = (native.Result * len(poses))()
    for _ in range(3):  # kernel by kernel, captured, replayed
        native.hip_check(lib.vmhip_batch_run(batch))
    native.hip_check(lib.vmhip_batch_fetch_held(batch, raw))
    return [dict(gidx=np.ctypeslib.as_array(r.global_indices, (r.n_visible,)).copy(), nb=np.ctypeslib.as_array(r.neighbourhood, (r.n_visible + 1, nn)).copy(),
                 cls=np.ctypeslib.as_array(r.classifications, (r.n_visible + 1, n_out)).copy()) for r in raw]


@pytest.mark.parametrize("case", sorted(CASES))
def test_ranges_of_the_whole_mesh(case):
    """One batch object stages wide views, whose rows reach far, then narrow ones with the whole mesh for ranges: the results of the ranges
    that hold the visible nodes alone, bit for bit."""
    widths, activation, precision = CASES[case]
    grid = "nine slots" in case
    nn, model = (8, wl.NMGRID8) if grid else (6, wl.RING6)
    lib, mesh = native.hip(), eng.Mesh(model, wl.CIRCLE, 0.05, 1.2, 3.65, 5.0) if grid else eng.Mesh(model, wl.SPHERE, 0.0949, 1.0, 3.0, 8.0)
    rays, neighbours = mesh.arrays()
    engine, device_mesh, batch = C.c_void_p(), C.c_void_p(), C.c_void_p()
    network = native.Network(wl.glorot_network(np.random.default_rng(3), widths, nn, activation))
    native.hip_check(lib.vmhip_engine_create(C.byref(network.c), nn, precision, C.byref(engine)))
    native.hip_check(lib.vmhip_mesh_upload(rays.ctypes.data_as(C.POINTER(C.c_float)), _pointer(neighbours), len(rays), nn, C.byref(device_mesh)))
    native.hip_check(lib.vmhip_batch_create(engine, C.byref(batch)))
    try:
        image, whole = wl.random_image(np.random.default_rng(2), 333, 266, 4), np.array([[0, len(rays)]], np.int32)
        poses = [wl.make_hoc(1.0, math.radians(p), 0.03, 0.4 * p) for p in (35.0, 50.0, 70.0)]
        wide, narrow = native.make_lens(333, 266, wl.EQUIDISTANT, 109.0, math.pi), native.make_lens(333, 266, wl.RECTILINEAR, 700.0, 0.6)
        _results(batch, device_mesh, wide, poses, image, [whole] * 3, nn, widths[-1])
        got = _results(batch, device_mesh, narrow, poses, image, [whole] * 3, nn, widths[-1])
        ranges = []
        for r in got:
            assert 0 < len(r["gidx"]) < len(rays) - 4 * 256  # tiles without rows
            cut = np.flatnonzero(np.diff(r["gidx"]) != 1)
            ranges.append(np.stack([r["gidx"][np.r_[0, cut + 1]], r["gidx"][np.r_[cut, -1]] + 1], 1).astype(np.int32))
        want = _results(batch, device_mesh, narrow, poses, image, ranges, nn, widths[-1])
        for g, w in zip(got, want):
            for key in w:
                assert np.array_equal(g[key], w[key]), key
    finally:
        lib.vmhip_batch_destroy(batch)
        lib.vmhip_mesh_release(device_mesh)
        lib.vmhip_engine_destroy(engine)
