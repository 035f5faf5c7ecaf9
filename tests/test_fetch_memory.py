"""What fetch() and the calls of one frame keep of the results they bring home: a page-locked block of 64 MB at most, nothing else."""
import ctypes as C
import gc
import math

import numpy as np
import pytest

from visualmesh_amd import engine as eng
from visualmesh_amd import native
from visualmesh_amd import workloads as wl

pytestmark = pytest.mark.gpu

MB = 1 << 20


def _device_used():
    free, total = C.c_size_t(), C.c_size_t()
    assert C.CDLL("libamdhip64.so").hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return total.value - free.value


def _resident():
    gc.collect()
    C.CDLL("libc.so.6").malloc_trim(0)
    return int(open("/proc/self/statm").read().split()[1]) * 4096


@pytest.mark.parametrize("frames", [8, 60])  # some 26 and 200 MB: below and above what is kept page-locked
def test_fetch_keeps_no_second_copy_of_the_results(frames):
    """On the device nothing (a quarter of the results' size for the runtime's own blocks), on the host the results themselves, which the
    library's C interface keeps until its next fetch, and the page-locked block (64 MB and half the results for whatever else)."""
    mesh, lens = eng.Mesh(wl.RING6, wl.SPHERE, 0.0949, 1.2, 6.0, 20.0), native.make_lens(1280, 1024, wl.EQUISOLID, 420.0, math.pi)
    rng = np.random.default_rng(6)
    image = wl.random_image(rng, 1280, 1024, 4)
    engine = eng.Engine(wl.glorot_network(np.random.default_rng(5), [3, 16, 3], 6, wl.SELU), wl.RING6)
    one = dict(mesh=mesh, Hoc=wl.make_hoc(1.2, math.radians(30.0), 0.0, 0.3), lens=lens, image=image, fourcc=wl.fourcc("RGBA"))
    engine.classify_batch([one])
    engine.stage([one] * frames)
    engine.run()
    size = int(native.hip().vmhip_batch_fetch_packed_size(engine.native_batch()))
    device, host = _device_used(), _resident()
    results = engine.fetch()
    assert len(results) == frames and sum(a.nbytes for r in results for a in r.values()) > 0.99 * size
    del results
    grown = _device_used() - device, _resident() - host
    print("%.1f MB of results: device memory grown by %.1f MB, host by %.1f" % (size / MB, grown[0] / MB, grown[1] / MB), flush=True)
    assert grown[0] < 0.25 * size
    assert grown[1] < 1.5 * size + 64 * MB
    if size > 64 * MB:
        assert grown[1] < 1.5 * size


def test_a_single_frame_past_the_block():
    """77 MB of projection, 106 MB of classification, by the calls of one frame, by value and through the C entry points: the same
    results, and a small frame after them."""
    lib, host = native.hip(), native.host()
    mesh, small = eng.Mesh(wl.NMGRID8, wl.CIRCLE, 0.05, 1.0, 15.0, 5.0), eng.Mesh(wl.NMGRID8, wl.CIRCLE, 0.05, 1.0, 2.0, 5.0)
    lens, Hoc = native.make_lens(1280, 1024, wl.EQUIDISTANT, 310.0, math.pi), wl.make_hoc(1.0, math.radians(90.0), 0.0, 0.3)
    image, fcc = wl.random_image(np.random.default_rng(6), 1280, 1024, 4), wl.fourcc("RGBA")
    engine = eng.Engine(wl.glorot_network(np.random.default_rng(5), [3, 8, 4], 8, wl.SELU), wl.NMGRID8)
    p, c = engine.project(mesh, Hoc, lens), engine(mesh, Hoc, lens, image, fcc)
    V = len(p["gidx"])
    assert V * 44 > 64 * MB
    engine.stage([dict(mesh=mesh, Hoc=Hoc, lens=lens, image=image, fourcc=fcc)])
    engine.run()
    want = engine.fetch_pinned()[0]
    fetched = engine.fetch()[0]
    raw = native.Result()
    native.hip_check(lib.vmhip_batch_fetch_held(engine.native_batch(), C.byref(raw)))
    assert raw.n_visible == V
    for key, pointer in (("px", raw.pixel_coordinates), ("nb", raw.neighbourhood), ("gidx", raw.global_indices), ("cls", raw.classifications)):
        assert np.array_equal(np.ctypeslib.as_array(pointer, (want[key].size,)), want[key].reshape(-1)), key
        assert np.array_equal(c[key], want[key]) and np.array_equal(fetched[key], want[key]), key
        if key != "cls":
            assert np.array_equal(p[key], want[key]), key
    p, c = engine.project(small, Hoc, lens), engine(small, Hoc, lens, image, fcc)
    engine.stage([dict(mesh=small, Hoc=Hoc, lens=lens, image=image, fourcc=fcc)])
    engine.run()
    want = engine.fetch_pinned()[0]
    assert 0 < len(want["gidx"]) * 44 < 8 * MB
    for key in want:
        assert np.array_equal(c[key], want[key]) and (key == "cls" or np.array_equal(p[key], want[key])), key
