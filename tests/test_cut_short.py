"""A pass that could not be launched to its end leaves nothing that the next one works with: run stamps, counts, lists of tiles."""
import math

import numpy as np
import pytest

from visualmesh_amd import engine as eng
from visualmesh_amd import native
from visualmesh_amd import workloads as wl

pytestmark = pytest.mark.gpu


def _frames(rng, n, k, pitch):
    mesh, lens = eng.Mesh(wl.RING6, wl.SPHERE, 0.0949, 1.0, k, 8.0), native.make_lens(160, 120, wl.EQUISOLID, 52.0, math.pi)
    return [dict(mesh=mesh, Hoc=wl.make_hoc(1.0, math.radians(pitch), 0.0, rng.uniform(-3, 3)), lens=lens, image=wl.random_image(rng, 160, 120, 4), fourcc=wl.fourcc("RGBA"))
            for _ in range(n)]


@pytest.mark.parametrize("early", [False, True], ids=["whole", "in two pieces"])
@pytest.mark.parametrize("widths,precision", [([3, 16, 32, 32, 4], native.FP32), ([3, 64, 64, 4], native.FP32), ([3, 64, 64, 4], native.SPLIT)], ids=["tiles", "half tiles", "pairs"])
def test_the_run_after_a_failed_one(widths, precision, early, monkeypatch):
    """With few halo slots nearly every tile of the failed pass, three dense frames, is on the list of those computed from memory; the
    batch staged then is smaller, on the same mesh."""
    monkeypatch.setenv("VMHIP_HALO_CAP", "8")
    rng, lib = np.random.default_rng(5), native.hip()
    network = wl.glorot_network(np.random.default_rng(3), widths, 6, wl.SELU)
    engine, fresh = eng.Engine(network, wl.RING6, precision), eng.Engine(network, wl.RING6, precision)
    large, small = _frames(rng, 3, 2.5, 40.0), _frames(rng, 1, 2.5, 5.0)
    engine.stage(large)
    if early:
        for _ in range(4):
            engine.run()
            engine.fetch_packed()
    native.hip_check(lib.vmhip_debug_set(native.DEBUG_CUT_SHORT, 1.0))
    try:
        with pytest.raises(native.VisualMeshError, match="cut short"):
            engine.run()
        with pytest.raises(native.VisualMeshError):
            engine.fetch()
    finally:
        native.hip_check(lib.vmhip_debug_set(native.DEBUG_CUT_SHORT, 0.0))
    for frames in (small, large):
        fresh.stage(frames)
        fresh.run()
        want = fresh.fetch()
        engine.stage(frames)
        for _ in range(3):
            engine.run()
            for got, w in zip(engine.fetch(), want):
                for key in w:
                    assert np.array_equal(got[key], w[key]), key
