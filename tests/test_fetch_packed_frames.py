"""A packed fetch of many frames: what a frame costs does not depend on how many there are."""
import math
import time

import numpy as np
import pytest

from visualmesh_amd import engine as eng
from visualmesh_amd import native
from visualmesh_amd import workloads as wl

pytestmark = pytest.mark.gpu


def _staged(engine, n, rng, k, max_distance):
    """n small frames, every ninth of which sees nothing"""
    mesh, lens, fcc = eng.Mesh(wl.RING6, wl.SPHERE, 0.0949, 1.0, k, max_distance), native.make_lens(64, 48, wl.EQUISOLID, 21.0, math.pi), wl.fourcc("RGBA")
    image = wl.random_image(rng, 64, 48, 4)
    sky = native.make_lens(64, 48, wl.RECTILINEAR, 35.0, math.pi / 2)
    engine.stage([dict(mesh=mesh, Hoc=wl.make_hoc(1.0, math.radians(-80.0 if i % 9 == 4 else rng.uniform(20, 60)), 0.0, rng.uniform(-3, 3)),
                       lens=sky if i % 9 == 4 else lens, image=image, fourcc=fcc) for i in range(n)])
    engine.run()


def test_hundreds_of_arrays_in_one_fetch():
    """1000 arrays of all lengths, empty ones among them: the same bytes as array by array."""
    engine = eng.Engine(wl.glorot_network(np.random.default_rng(5), [3, 8, 3], 6, wl.SELU), wl.RING6)
    _staged(engine, 250, np.random.default_rng(6), 1.5, 4.0)
    want, got = engine.fetch_pinned(), engine.fetch_packed()
    assert sum(len(w["gidx"]) == 0 for w in want) == 28 and sum(len(w["gidx"]) for w in want) > 10000
    for w, g in zip(want, got):
        for key in w:
            assert w[key].shape == g[key].shape and np.array_equal(w[key], g[key]), key


def test_the_time_of_a_fetch_goes_with_its_frames():
    """Eight times the frames, of some KB each: eight times the time at most, since fixed costs only make it less. The line lies
    at half as much again (7.7 times measured); with a kernel whose every block reads the table of all arrays it was 18.7 times."""
    lib, seconds = native.hip(), []
    for n in (1000, 8000):
        engine = eng.Engine(wl.glorot_network(np.random.default_rng(5), [3, 8, 3], 6, wl.SELU), wl.RING6)
        _staged(engine, n, np.random.default_rng(6), 1.0, 2.0)
        batch, raw = engine.native_batch(), (native.Result * n)()
        block = native.pinned_empty((int(lib.vmhip_batch_fetch_packed_size(batch)),), np.uint8)
        best = math.inf
        for _ in range(10):
            start = time.perf_counter()
            native.hip_check(lib.vmhip_batch_fetch_packed_async(batch, block.ctypes.data, block.nbytes, raw))
            native.hip_check(lib.vmhip_batch_fetch_wait(batch))
            best = min(best, time.perf_counter() - start)
        seconds.append(best)
        print("%d frames, %.1f MB: %.0f us" % (n, block.nbytes / 1e6, best * 1e6), flush=True)
    assert seconds[1] <= 12 * seconds[0], seconds
