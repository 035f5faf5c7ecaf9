"""Pipeline: geometry beside the upload, one copy at a time each way. What the ordinary test of it does not reach: overruled decisions, batches that fail.
(Empty batches, and results held across a call: test_pipeline_states.py.)"""
import math
import time

import numpy as np
import pytest

from visualmesh_amd import engine as eng
from visualmesh_amd import native
from visualmesh_amd import workloads as wl

pytestmark = pytest.mark.gpu


def _batches(rng, ks, fourcc="RGBA", model=wl.RING6):
    shape, radius = (wl.SPHERE, 0.0949) if model == wl.RING6 else (wl.CIRCLE, 0.05)
    lens, out = native.make_lens(320, 240, wl.EQUISOLID, 105.0, math.pi), []
    for batch in ks:
        images = native.pinned_empty((len(batch), 240, 320 * (4 if fourcc == "RGBA" else 1)), np.uint8)
        images[:] = rng.integers(0, 256, images.shape, np.uint8)
        out.append([dict(mesh=eng.Mesh(model, shape, radius, 1.0, k, 6.0), Hoc=wl.make_hoc(1.0, math.radians(rng.uniform(20, 60)), 0.0, rng.uniform(-3, 3)), lens=lens,
                         image=image, fourcc=wl.fourcc(fourcc)) for k, image in zip(batch, images)])
    return out


def _through(pipe, batches):
    out = []
    for b in batches + [None, None]:  # the arrays are valid until two more calls
        done = pipe.submit(b) if b else pipe.flush()
        if done is not None:
            out.append([{k: v.copy() for k, v in r.items()} for r in done])
    return out


def _wanted(engine, batches):
    out = []
    for b in batches:
        engine.stage(b)
        engine.run()
        out.append([{k: v.copy() for k, v in r.items()} for r in engine.fetch_pinned()])
    return out


def _same(got, want, keys=("px", "nb", "gidx", "cls")):
    assert len(got) == len(want)
    for g, w in zip(got, want):
        assert len(g) == len(w)
        for a, b in zip(g, w):
            for key in keys:
                assert a[key].shape == b[key].shape and np.array_equal(a[key], b[key]), key


@pytest.mark.parametrize("widths,model,fourcc,precision", [([3, 16, 32, 32, 3], wl.RING6, "RGBA", native.FP32), ([3, 24, 4], wl.NMGRID8, "GRBG", native.FP32), ([3, 64, 64, 4], wl.RING6, "RGBA", native.SPLIT),
                                                           ([3, 40, 100], wl.RING6, "RGBA", native.FP32)])
def test_the_same_bits_as_staged_batches(widths, model, fourcc, precision):
    net = wl.glorot_network(np.random.default_rng(3), widths, wl.N_NEIGHBOURS[model], wl.SELU)
    batches = _batches(np.random.default_rng(5), [(2.0, 1.3), (0.4,), (3.1, 2.0, 0.7), (2.0, 1.3), (2.0,), (5.0, 1.0)], fourcc, model)
    pipe, engine = eng.Pipeline(net, model, precision), eng.Engine(net, model, precision)
    want = _wanted(engine, batches)
    for _ in range(2):
        _same(_through(pipe, batches), want)


def test_overruled_decisions_and_a_batch_cut_short():
    net, lib = wl.glorot_network(np.random.default_rng(3), [3, 16, 32, 3], 6, wl.SELU), native.hip()
    batches = _batches(np.random.default_rng(5), [(4.0, 3.0), (2.5,), (4.0, 1.0), (3.0,)])
    pipe, engine = eng.Pipeline(net, wl.RING6), eng.Engine(net, wl.RING6)
    want = _wanted(engine, batches)
    native.hip_check(lib.vmhip_debug_set(native.DEBUG_PROJECTION_ERROR, 0.5))
    native.hip_check(lib.vmhip_debug_set(native.DEBUG_EDGE_BAND, 0.6))
    try:
        _same(_through(pipe, batches), want, ("nb", "gidx"))
    finally:
        native.hip_check(lib.vmhip_debug_set(native.DEBUG_PROJECTION_ERROR, 0.0))
        native.hip_check(lib.vmhip_debug_set(native.DEBUG_EDGE_BAND, 0.0))
    _same(_through(pipe, batches), want)
    other = eng.Pipeline(net, wl.RING6)
    other.submit(batches[0])
    native.hip_check(lib.vmhip_debug_set(native.DEBUG_CUT_SHORT, 1.0))
    try:
        with pytest.raises(native.VisualMeshError, match="cut short"):
            other.submit(batches[1])
    finally:
        native.hip_check(lib.vmhip_debug_set(native.DEBUG_CUT_SHORT, 0.0))
    del other  # with a batch under way
    fresh = eng.Pipeline(net, wl.RING6)
    _same(_through(fresh, batches), want)


def test_batches_that_fail():
    """One that cannot be queued is as if it had not been submitted, one whose network fails is lost and told in its turn; all others come as they would have."""
    cfg, lib = wl.config(2, n_frames=1), native.hip()
    batches = _batches(np.random.default_rng(5), [(4.0, 3.0), (6.0,), (4.0, 1.0), (3.0,), (2.0, 2.0)])
    pipe, engine = eng.Pipeline(cfg.network, wl.RING6), eng.Engine(cfg.network, wl.RING6)
    want = _wanted(engine, batches)

    def submit(i):
        done = pipe.submit(batches[i])
        return None if done is None else [{k: v.copy() for k, v in r.items()} for r in done]

    for _ in range(2):
        assert submit(0) is None
        native.hip_check(lib.vmhip_debug_set(native.DEBUG_CUT_SHORT, 1.0))
        try:
            with pytest.raises(native.VisualMeshError, match="cut short"):
                submit(1)
        finally:
            native.hip_check(lib.vmhip_debug_set(native.DEBUG_CUT_SHORT, 0.0))
        native.hip_check(lib.vmhip_debug_set(native.DEBUG_FLOW_POLL_LIMIT, 1))
        try:
            assert submit(1) is None
            time.sleep(0.1)  # its network fails now
        finally:
            native.hip_check(lib.vmhip_debug_set(native.DEBUG_FLOW_POLL_LIMIT, 0))
        _same([submit(2)], [want[0]])
        with pytest.raises(native.VisualMeshError, match="gave up waiting"):
            submit(3)
        _same([submit(4)], [want[2]])
        _same([pipe.flush(), pipe.flush()], want[3:])
        assert pipe.flush() is None
