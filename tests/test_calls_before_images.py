"""Calls of one frame, whose geometry is worked out and brought home before the image is there: the same bits as a staged batch's."""
import ctypes as C
import math

import numpy as np
import pytest

from visualmesh_amd import engine as eng
from visualmesh_amd import native
from visualmesh_amd import workloads as wl

pytestmark = pytest.mark.gpu

BPP = {"RGBA": 4, "BGR3": 3, "GREY": 1, "GRBG": 1}


def _frame(rng, fourcc="RGBA", model=wl.RING6, k=2.3, size=(321, 243), pitch=40.0):
    size = size if fourcc != "GRBG" else (320, 240)
    shape, radius = (wl.SPHERE, 0.0949) if model == wl.RING6 else (wl.CIRCLE, 0.05)
    return dict(mesh=eng.Mesh(model, shape, radius, 1.0, k, 6.0), Hoc=wl.make_hoc(1.0, math.radians(pitch), 0.05, 0.3),
                lens=native.make_lens(size[0], size[1], wl.EQUISOLID, 0.33 * size[0], math.pi), image=wl.random_image(rng, size[0], size[1], BPP[fourcc]), fourcc=wl.fourcc(fourcc))


def _staged(engine, frame):
    engine.stage([frame])
    engine.run()
    return {key: a.copy() for key, a in engine.fetch_pinned()[0].items()}


def _call(engine, f):
    return engine(f["mesh"], f["Hoc"], f["lens"], f["image"], f["fourcc"])


def _same(got, want):
    for key in want:
        assert got[key].shape == want[key].shape and np.array_equal(got[key], want[key]), key


# first layers inside the sampling kernel (one and two blocks of columns, partly filled ones) and outside it, each format and activation, tiles with neighbours that are not
# staged, nodes of one tile and of some fifty
@pytest.mark.parametrize("hidden,fourcc,model,activation,k,halo_cap", [
    ([16], "RGBA", wl.RING6, wl.SELU, 2.3, None), ([12], "BGR3", wl.RING6, wl.RELU, 0.4, None), ([24, 24], "GRBG", wl.NMGRID8, wl.TANH, 2.0, None), ([32, 32, 32], "GREY", wl.RING6, wl.SELU, 6.0, None),
    ([16, 16], "GRBG", wl.RING6, wl.SELU, 2.3, 8), ([20], "RGBA", wl.NMGRID8, wl.RELU, 2.3, 0), ([64, 64], "RGBA", wl.RING6, wl.SELU, 2.3, None), ([10], "RGBA", wl.RING6, wl.TANH, 2.3, None)])
@pytest.mark.parametrize("precision", ["fp32", "split"])
def test_the_same_bits_as_a_staged_frame(hidden, fourcc, model, activation, k, halo_cap, precision, monkeypatch):
    if precision == "split" and hidden != [64, 64]:
        pytest.skip("layers of 64 channels only")
    if halo_cap is not None:
        monkeypatch.setenv("VMHIP_HALO_CAP", str(halo_cap))
    rng = np.random.default_rng(5)
    net = wl.glorot_network(np.random.default_rng(3), [3] + hidden + [4], wl.N_NEIGHBOURS[model], activation)
    engine, other = (eng.Engine(net, model, native.SPLIT if precision == "split" else native.FP32) for _ in range(2))
    frame = _frame(rng, fourcc, model, k)
    want = _staged(other, frame)
    assert len(want["gidx"]) > 0
    for _ in range(2):
        _same(_call(engine, frame), want)
    frame = dict(frame, image=frame["image"] ^ 0x55)  # another image in the same place
    _same(_call(engine, frame), _staged(other, frame))


def test_a_device_that_decides_wrongly():
    """The verdict comes before the layers run: overruled decisions are worked out again, with the image already there."""
    rng, lib = np.random.default_rng(5), native.hip()
    net = wl.glorot_network(np.random.default_rng(3), [3, 16, 3], 6, wl.SELU)
    engine, frame = eng.Engine(net, wl.RING6), _frame(rng, k=4.0)
    right = _call(engine, frame)
    native.hip_check(lib.vmhip_debug_set(native.DEBUG_PROJECTION_ERROR, 0.5))
    native.hip_check(lib.vmhip_debug_set(native.DEBUG_EDGE_BAND, 0.6))
    try:
        got = _call(engine, frame)
        assert native.guard_stats(engine.native_batch())["reruns"] >= 1
        assert np.array_equal(got["gidx"], right["gidx"]) and np.array_equal(got["nb"], right["nb"]) and got["cls"].shape == right["cls"].shape
    finally:
        native.hip_check(lib.vmhip_debug_set(native.DEBUG_PROJECTION_ERROR, 0.0))
        native.hip_check(lib.vmhip_debug_set(native.DEBUG_EDGE_BAND, 0.0))
    _same(_call(engine, frame), right)


def test_calls_cut_short_or_left_open():
    """A call that could not be launched to its end, one that nobody finished, entry points that refuse to work on an open one: the next call is right."""
    rng, lib = np.random.default_rng(5), native.hip()
    net = wl.glorot_network(np.random.default_rng(3), [3, 16, 32, 32, 4], 6, wl.SELU)
    engine, frame, small = eng.Engine(net, wl.RING6), _frame(rng, k=4.0), _frame(rng, k=1.0, pitch=20.0)
    want, want_small = _call(engine, frame), _call(engine, small)
    native.hip_check(lib.vmhip_debug_set(native.DEBUG_CUT_SHORT, 1.0))
    try:
        with pytest.raises(native.VisualMeshError, match="cut short"):
            _call(engine, frame)
    finally:
        native.hip_check(lib.vmhip_debug_set(native.DEBUG_CUT_SHORT, 0.0))
    _same(_call(engine, small), want_small)
    host, r = native.host(), native.Result()
    H = np.ascontiguousarray(frame["Hoc"], np.float32)
    native.host_check(host.vmh_engine_classify_begin(engine.ptr, frame["mesh"].ptr, H.ctypes.data_as(C.POINTER(C.c_float)), C.byref(frame["lens"]), frame["image"].ctypes.data, frame["fourcc"], C.byref(r)))
    assert r.n_visible == len(want["gidx"])
    with pytest.raises(native.VisualMeshError, match="still open"):
        engine.run()
    _same(_call(engine, small), want_small)
    _same(_call(engine, frame), want)
    engine._staged = [frame["mesh"]]
    engine.run()  # the call's frame is staged, its image there
    _same(engine.fetch_pinned()[0], want)


def test_the_geometry_is_there_when_the_first_half_returns():
    """Megabytes of geometry and nothing that would hold the host up behind the verdict (a small page-locked image, one layer): what the first half returns
    is whole as it returns, in a block that still has another pose's geometry."""
    rng, host = np.random.default_rng(5), native.host()
    net = wl.glorot_network(np.random.default_rng(3), [3, 4], 6, wl.SELU)
    engine, other = (eng.Engine(net, wl.RING6) for _ in range(2))
    image = native.pinned_empty((256, 320), np.uint8)
    image[:] = rng.integers(0, 256, image.shape, np.uint8)
    mesh, lens = eng.Mesh(wl.RING6, wl.SPHERE, 0.0949, 1.0, 10.0, 20.0), native.make_lens(320, 256, wl.EQUISOLID, 105.0, math.pi)
    wants = []
    for pitch in (30.0, 50.0):
        frame = dict(mesh=mesh, Hoc=wl.make_hoc(1.0, math.radians(pitch), 0.05, 0.3), lens=lens, image=image, fourcc=wl.fourcc("GREY"))
        wants.append((frame, _staged(other, frame)))
    for turn in range(6):
        frame, want = wants[turn % 2]
        V, r, H = len(want["gidx"]), native.Result(), np.ascontiguousarray(frame["Hoc"], np.float32)
        assert V > 100000
        native.host_check(host.vmh_engine_classify_begin(engine.ptr, mesh.ptr, H.ctypes.data_as(C.POINTER(C.c_float)), C.byref(lens), image.ctypes.data, frame["fourcc"], C.byref(r)))
        nb, px, gidx = (np.ctypeslib.as_array(p, shape).copy() for p, shape in ((r.neighbourhood, (V + 1, 6)), (r.pixel_coordinates, (V, 2)), (r.global_indices, (V,))))
        native.host_check(host.vmh_engine_classify_end(engine.ptr))
        assert r.n_visible == V
        _same(dict(px=px, nb=nb, gidx=gidx, cls=np.ctypeslib.as_array(r.classifications, (V + 1, 4))), want)
