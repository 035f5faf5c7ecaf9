"""A run that fails while its results are on their way into an announced block."""
import ctypes as C

import numpy as np
import pytest

from visualmesh_amd import engine as eng
from visualmesh_amd import native
from visualmesh_amd import workloads as wl

pytestmark = pytest.mark.gpu


def test_nothing_is_stored_behind_a_failed_run():
    """The wait that ran out is known before the pass's last kernel has stored the classifications: the caller, who may free the block now, has the run back when it has."""
    cfg = wl.config(2, n_frames=1)
    f, lib, v = cfg.frames[0], native.hip(), cfg.visualmesh
    mesh = eng.VisualMesh(cfg.model, cfg.shape, cfg.radius, v["min_h"], v["max_h"], cfg.k, v["max_error"], cfg.max_distance)
    engine = eng.Engine(cfg.network, cfg.model)
    engine.stage([dict(mesh=mesh, Hoc=f["Hoc"], lens=native.make_lens(*cfg.lens_tuple()), image=f["image"], fourcc=cfg.fourcc)])
    engine.run()
    want, batch = [{k: a.copy() for k, a in r.items()} for r in engine.fetch_pinned()], engine.native_batch()
    block = native.pinned_empty((int(lib.vmhip_batch_fetch_packed_size(batch)),), np.uint8)
    native.hip_check(lib.vmhip_debug_set(native.DEBUG_FLOW_POLL_LIMIT, 1))
    try:
        for _ in range(4):
            block[:] = 0xee
            native.hip_check(lib.vmhip_batch_announce_packed(batch, block.ctypes.data, block.nbytes))
            with pytest.raises(RuntimeError, match="gave up waiting"):
                engine.run()
            there = block[::-64].copy()  # the classifications, which come last, first
            native.hip_check(lib.vmhip_batch_announce_packed(batch, None, 0))  # waits for everything
            assert np.array_equal(there, block[::-64])
    finally:
        native.hip_check(lib.vmhip_debug_set(native.DEBUG_FLOW_POLL_LIMIT, 0))
    native.hip_check(lib.vmhip_batch_announce_packed(batch, block.ctypes.data, block.nbytes))
    engine.run()
    raw = native.Result()
    native.hip_check(lib.vmhip_batch_fetch_packed_async(batch, block.ctypes.data, block.nbytes, C.byref(raw)))
    native.hip_check(lib.vmhip_batch_fetch_wait(batch))
    V, classes = raw.n_visible, want[0]["cls"].shape[1]
    assert V == len(want[0]["gidx"]) and np.array_equal(np.ctypeslib.as_array(raw.classifications, (V + 1, classes)), want[0]["cls"])
