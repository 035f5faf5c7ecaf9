"""Packed fetches whose pixels, indices and neighbourhoods were delivered while the layers ran: the same bytes as array by array."""
import math

import numpy as np
import pytest

from visualmesh_amd import engine as eng
from visualmesh_amd import native
from visualmesh_amd import workloads as wl

pytestmark = pytest.mark.gpu


def _frames(rng, n, k=2.0, model=wl.RING6, blind=()):
    shape, radius = (wl.SPHERE, 0.0949) if model == wl.RING6 else (wl.CIRCLE, 0.05)
    mesh, lens, fcc = eng.Mesh(model, shape, radius, 1.0, k, 5.0), native.make_lens(160, 120, wl.EQUISOLID, 52.0, math.pi), wl.fourcc("RGBA")
    sky = native.make_lens(160, 120, wl.RECTILINEAR, 88.0, math.pi / 2)
    image = wl.random_image(rng, 160, 120, 4)
    return [dict(mesh=mesh, Hoc=wl.make_hoc(1.0, math.radians(-80.0 if i in blind else rng.uniform(20, 60)), 0.0, rng.uniform(-3, 3)),
                 lens=sky if i in blind else lens, image=image, fourcc=fcc) for i in range(n)]


def _engine(widths=(3, 16, 32, 4), precision=native.FP32, model=wl.RING6):
    return eng.Engine(wl.glorot_network(np.random.default_rng(3), list(widths), wl.N_NEIGHBOURS[model], wl.SELU), model, precision)


def _copied(results):
    return [{k: np.array(v) for k, v in r.items()} for r in results]


def _same(got, want):
    assert len(got) == len(want)
    for g, w in zip(got, want):
        for key in w:
            assert g[key].shape == w[key].shape and np.array_equal(g[key], w[key]), key


@pytest.mark.parametrize("case", ["one", "several", "grid", "split", "nothing", "wide offsets"])
def test_batches_of_changing_size(case):
    """Seven batches through one engine, larger and smaller ones, frames that see nothing among them: the first two passes go as ever,
    the others deliver early, kernel by kernel at first, then as graphs; a batch that outgrew the block falls back for one pass."""
    rng = np.random.default_rng(21)
    model = wl.NMGRID8 if case == "grid" else wl.RING6
    engine = _engine((3, 64, 64, 4) if case == "split" else (3, 16, 32, 4), native.SPLIT if case == "split" else native.FP32, model)
    lib, early = native.hip(), 0
    native.hip_check(lib.vmhip_debug_set(native.DEBUG_WIDE_OFFSETS, 1.0 if case == "wide offsets" else 0.0))
    try:
        for turn, (n, k) in enumerate([(2, 2.0), (2, 2.0), (3, 2.0), (1, 1.5), (3, 2.0), (3, 3.0), (3, 3.0)]):
            if case == "one":
                n = 1
            engine.stage(_frames(rng, n, k, model, range(n) if case == "nothing" else [1] if case == "several" else ()))
            for _ in range(2):
                engine.run()
                delivered = lib.vmhip_batch_delivered(engine.native_batch())
                early += bool(delivered)
                got = engine.fetch_packed()
                _same(got, engine.fetch_pinned())
    finally:
        native.hip_check(lib.vmhip_debug_set(native.DEBUG_WIDE_OFFSETS, 0.0))
    assert early == 0 if case == "nothing" else early >= 8, early


def test_arrays_stay_until_the_next_packed_fetch():
    """The run that delivers early writes beside the arrays that the last fetch returned."""
    rng = np.random.default_rng(4)
    engine, last = _engine(), None
    for turn in range(6):
        engine.stage(_frames(rng, 2))
        engine.run()
        if last is not None:
            _same(last[0], last[1])
        got = engine.fetch_packed()
        last = (got, _copied(got))
        engine.run_async()  # nothing was fetched of this one
        engine.wait()
        _same(last[0], last[1])


def test_overruled_decisions():
    """A device that decides wrongly at the screen's edge: the pass is repeated, and what was delivered of the first one is not used."""
    rng = np.random.default_rng(5)
    engine, lib = _engine(), native.hip()
    frames = _frames(rng, 3)
    for _ in range(3):
        engine.stage(frames)
        engine.run()
        right = _copied(engine.fetch_packed())
    native.hip_check(lib.vmhip_debug_set(native.DEBUG_PROJECTION_ERROR, 0.5))
    native.hip_check(lib.vmhip_debug_set(native.DEBUG_EDGE_BAND, 0.6))
    try:
        engine.stage(frames)
        engine.run()
        assert native.guard_stats(engine.native_batch())["reruns"] >= 1
        assert not lib.vmhip_batch_delivered(engine.native_batch())
        got = engine.fetch_packed()
        for g, w in zip(got, right):
            assert np.array_equal(g["gidx"], w["gidx"]) and np.array_equal(g["nb"], w["nb"])
        engine.run()
        assert lib.vmhip_batch_delivered(engine.native_batch())
        again = engine.fetch_packed()
        for g, w in zip(again, right):
            assert np.array_equal(g["gidx"], w["gidx"]) and np.array_equal(g["nb"], w["nb"])
    finally:
        native.hip_check(lib.vmhip_debug_set(native.DEBUG_PROJECTION_ERROR, 0.0))
        native.hip_check(lib.vmhip_debug_set(native.DEBUG_EDGE_BAND, 0.0))


def test_announcements_that_are_not_used():
    """A block that is too small, memory that is not page-locked, more frames than the gathering kernel takes, an announcement that is
    withdrawn, a fetch into another block: everything is fetched as without one."""
    lib, rng = native.hip(), np.random.default_rng(6)
    engine = _engine()
    engine.stage(_frames(rng, 2))
    engine.run()
    want, batch = engine.fetch_pinned(), engine.native_batch()
    need = int(lib.vmhip_batch_fetch_packed_size(batch))
    block, other, plain = native.pinned_empty((need,), np.uint8), native.pinned_empty((need,), np.uint8), np.zeros(need, np.uint8)

    def fetched(into):
        raw = (native.Result * 2)()
        native.hip_check(lib.vmhip_batch_fetch_packed_async(batch, into.ctypes.data, into.nbytes, raw))
        native.hip_check(lib.vmhip_batch_fetch_wait(batch))
        for r, w in zip(raw, want):
            V = r.n_visible
            assert V == len(w["gidx"])
            for pointer, key in ((r.pixel_coordinates, "px"), (r.global_indices, "gidx"), (r.neighbourhood, "nb"), (r.classifications, "cls")):
                assert np.array_equal(np.ctypeslib.as_array(pointer, w[key].shape), w[key]), key

    for announced, nbytes, used in ((block, need - 1, False), (plain, need, False), (block, need, True), (block, need, False)):
        native.hip_check(lib.vmhip_batch_announce_packed(batch, announced.ctypes.data, nbytes))
        if announced is block and nbytes == need and not used:
            native.hip_check(lib.vmhip_batch_announce_packed(batch, None, 0))
        block[:] = 0xee
        engine.run()
        assert bool(lib.vmhip_batch_delivered(batch)) == used
        fetched(other)  # another block than the one announced
        fetched(block)
    engine.stage(_frames(rng, 257, 1.0))
    for _ in range(4):
        engine.run()
        assert not lib.vmhip_batch_delivered(batch)
        got = engine.fetch_packed()
    _same(got, engine.fetch_pinned())


def test_a_delivery_serves_one_fetch():
    """What a packed fetch has brought is the caller's: changed in place, or its block freed and another one at the address, a further fetch
    of the same run brings the run's results."""
    lib, rng = native.hip(), np.random.default_rng(8)
    engine = _engine()
    engine.stage(_frames(rng, 2))
    for _ in range(4):
        engine.run()
        want = _copied(engine.fetch_pinned())
        for _ in range(3):
            got = engine.fetch_packed()
            _same(got, want)
            for g in got:
                g["px"] += 0.5
                g["gidx"][:], g["nb"][:], g["cls"][:] = 7, -1, 0.0
        engine.run()  # not fetched
    batch = engine.native_batch()
    need = int(lib.vmhip_batch_fetch_packed_size(batch))
    for freed in (False, True):
        block = native.pinned_empty((need,), np.uint8)
        native.hip_check(lib.vmhip_batch_announce_packed(batch, block.ctypes.data, need))
        engine.run()
        assert lib.vmhip_batch_delivered(batch) == block.ctypes.data
        for _ in range(2):
            raw = (native.Result * 2)()
            native.hip_check(lib.vmhip_batch_fetch_packed_async(batch, block.ctypes.data, need, raw))
            native.hip_check(lib.vmhip_batch_fetch_wait(batch))
            assert not lib.vmhip_batch_delivered(batch)
            for r, w in zip(raw, want):
                for pointer, key in ((r.pixel_coordinates, "px"), (r.global_indices, "gidx"), (r.neighbourhood, "nb"), (r.classifications, "cls")):
                    assert np.array_equal(np.ctypeslib.as_array(pointer, w[key].shape), w[key]), (freed, key)
            if freed:
                del block
                block = native.pinned_empty((need,), np.uint8)  # at the same address, as a rule
            block[:] = 0xee


def test_cpp_calls(tmp_path):
    """tests/native/packed_fetch.cpp: announce_packed and fetch_packed_async of the C++ engine."""
    import os
    import subprocess
    root, lib_dir, exe = os.path.dirname(os.path.dirname(os.path.abspath(__file__))), os.path.dirname(native.HIP_LIB), str(tmp_path / "packed_fetch")
    subprocess.run(["g++", "-std=c++14", "-O1", "-Wall", "-Wextra", "-Werror", "-I" + os.path.join(root, "visualmesh_amd", "cpp"), "-I" + os.path.join(root, "include"),
                    os.path.join(root, "tests", "native", "packed_fetch.cpp"), "-L" + lib_dir, "-lvisualmesh_hip", "-Wl,-rpath," + lib_dir, "-pthread", "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout + out.stderr
