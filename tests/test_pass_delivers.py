"""What a pass brings home itself: classifications stored behind the verdict, gathered on the device where they are many, and the whole result of a call."""
import math

import numpy as np
import pytest

from visualmesh_amd import engine as eng
from visualmesh_amd import native
from visualmesh_amd import workloads as wl

pytestmark = pytest.mark.gpu


def _frames(rng, ks, model=wl.RING6, blind=()):
    shape, radius = (wl.SPHERE, 0.0949) if model == wl.RING6 else (wl.CIRCLE, 0.05)
    lens, sky, image = native.make_lens(320, 240, wl.EQUISOLID, 105.0, math.pi), native.make_lens(320, 240, wl.RECTILINEAR, 176.0, math.pi / 2), wl.random_image(rng, 320, 240, 4)
    return [dict(mesh=eng.Mesh(model, shape, radius, 1.0, k, 6.0), Hoc=wl.make_hoc(1.0, math.radians(-80.0 if i in blind else rng.uniform(20, 60)), 0.0, rng.uniform(-3, 3)),
                 lens=sky if i in blind else lens, image=image, fourcc=wl.fourcc("RGBA")) for i, k in enumerate(ks)]


def _same(got, want):
    for g, w in zip(got, want):
        for key in w:
            assert g[key].shape == w[key].shape and np.array_equal(g[key], w[key]), key


# few rows; ragged frames of one to some hundred tiles; a blind frame between others; nothing but blind ones; eight neighbours; more classifications than are stored directly
@pytest.mark.parametrize("ks,classes,model,blind", [((0.5,), 1, wl.RING6, ()), ((1.0, 2.3, 4.1, 0.7), 3, wl.RING6, ()), ((2.0, 2.0, 1.7), 5, wl.RING6, (1,)), ((2.0, 2.0), 4, wl.RING6, (0, 1)),
                                                    ((1.5, 2.2), 4, wl.NMGRID8, ()), ((3.0, 5.0, 4.0), 100, wl.RING6, ()), ((3.0, 5.5, 5.0), 100, wl.RING6, (0,))])
def test_the_same_bytes_as_array_by_array(ks, classes, model, blind):
    rng = np.random.default_rng(7)
    net = wl.glorot_network(np.random.default_rng(3), [3, 16, classes], wl.N_NEIGHBOURS[model], wl.SELU)
    engine, frames = eng.Engine(net, model), _frames(rng, ks, model, blind)
    engine.stage(frames)
    most = 4 * classes * sum(int((r[:, 1] - r[:, 0]).sum()) for r in (engine.staged_ranges(i) for i in range(len(frames))))
    assert (most > 8 << 20) == (classes == 100)
    for turn in range(5):
        engine.run() if turn != 3 else (engine.run_async(), engine.wait())
        assert bool(native.hip().vmhip_batch_delivered(engine.native_batch())) == (turn > 1 and len(blind) < len(ks))
        got = engine.fetch_packed()
        _same(got, engine.fetch_pinned())
    want = engine.fetch_pinned()
    want = [{key: a.copy() for key, a in w.items()} for w in want]
    for f, w in zip(frames, want):  # the calls of one frame, whose candidates are not tested by the host
        _same([engine(f["mesh"], f["Hoc"], f["lens"], f["image"], f["fourcc"])], [w])
        if len(w["gidx"]):
            _same([engine.project(f["mesh"], f["Hoc"], f["lens"])], [{key: w[key] for key in ("px", "nb", "gidx")}])


@pytest.mark.parametrize("precision", [native.FP32, native.BF16, native.SPLIT], ids=["fp32", "bf16", "split"])
@pytest.mark.parametrize("frames,blind,halo_cap", [(10, (), None), (10, (0, 4, 5, 9), None), (12, (1,), 20), (1, (), None)], ids=["four groups", "blind frames", "far neighbours", "one frame"])
def test_the_last_two_layers_by_groups_of_frames(precision, frames, blind, halo_cap, monkeypatch):
    """More than 8 MB of classifications behind 64-wide layers: the same bits as with all frames at once, which the first passes and every other fetch have."""
    if halo_cap is not None:
        monkeypatch.setenv("VMHIP_HALO_CAP", str(halo_cap))
    rng = np.random.default_rng(7)
    lens, sky = native.make_lens(1280, 1024, wl.EQUISOLID, 420.0, math.pi), native.make_lens(1280, 1024, wl.RECTILINEAR, 700.0, math.pi / 2)
    mesh, image = eng.Mesh(wl.RING6, wl.SPHERE, 0.0949, 1.2, 24.5 if frames == 1 else 7.6, 20.0), wl.random_image(rng, 1280, 1024, 4)
    batch = [dict(mesh=mesh, Hoc=wl.make_hoc(1.2, math.radians(-80.0 if i in blind else rng.uniform(20, 50)), 0.0, rng.uniform(-3, 3)), lens=sky if i in blind else lens, image=image,
                  fourcc=wl.fourcc("RGBA")) for i in range(frames)]
    engine = eng.Engine(wl.glorot_network(np.random.default_rng(3), [3, 64, 64, 64, 4], 6, wl.SELU), wl.RING6, precision)
    engine.stage(batch)
    assert sum(16 * int((r[:, 1] - r[:, 0]).sum()) for r in (engine.staged_ranges(i) for i in range(frames))) > 8 << 20
    want = None
    for turn in range(5):
        engine.run()
        got = engine.fetch_packed()
        if want is None:
            want = [{key: a.copy() for key, a in g.items()} for g in got]
        _same(got, want)
    _same(engine.fetch_pinned(), want)


def test_no_groups_where_the_class_layer_could_not_be_launched_for_some_frames():
    """Batches whose 64-wide rows reach 4 GiB, which the sliced class layer's 32-bit offsets do not: all frames at once. A first group that has fewer rows than the classifications of
    the whole batch cover of the matrix beneath them would have the next one read rows that are no longer there."""
    rng = np.random.default_rng(7)
    small, lens, image = native.make_lens(320, 240, wl.EQUISOLID, 105.0, math.pi), native.make_lens(1280, 1280, wl.EQUIDISTANT, 400.0, math.pi), wl.random_image(rng, 1280, 1280, 4)
    mesh, few = eng.Mesh(wl.RING6, wl.SPHERE, 0.0949, 1.0, 56.5, 20.0), eng.Mesh(wl.RING6, wl.SPHERE, 0.0949, 1.0, 2.0, 6.0)
    batch = [dict(mesh=few, Hoc=wl.make_hoc(1.0, math.radians(30.0), 0.0, 0.0), lens=small, image=image[:240, :320].copy(), fourcc=wl.fourcc("RGBA"))]
    batch += [dict(mesh=mesh, Hoc=wl.make_hoc(1.0, math.radians(90.0), 0.0, turn), lens=lens, image=image, fourcc=wl.fourcc("RGBA")) for turn in (0.3, 1.1)]
    engine = eng.Engine(wl.glorot_network(np.random.default_rng(3), [3, 64, 64, 4], 6, wl.SELU), wl.RING6, native.BF16)
    engine.stage(batch)
    rows = [int((r[:, 1] - r[:, 0]).sum()) for r in (engine.staged_ranges(i) for i in range(3))]
    assert sum(rows) * 64 * 4 > 1 << 32 and rows[0] * 8 < sum(rows) and rows[0] + rows[1] / 2 >= sum(rows) / 4
    want = None
    for turn in range(3):
        engine.run()
        got = engine.fetch_packed()
        if want is None:
            want = [{key: a.copy() for key, a in g.items()} for g in got]
    _same(got, want)
