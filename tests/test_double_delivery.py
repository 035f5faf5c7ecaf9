"""The double engine's results through its page-locked block, and past it (64 MB), in calls of changing size."""
import math

import numpy as np
import pytest

from visualmesh_amd import engine as eng
from visualmesh_amd import native
from visualmesh_amd import workloads as wl

pytestmark = pytest.mark.gpu


def test_sizes_in_turn():
    """One tile's rows, a frame, more than the block holds, one tile's again: neighbourhoods as the mesh and the indices say, pixels on screen, a classification's geometry the
    projection's, every row's probabilities a distribution."""
    lens, Hoc = native.make_lens64(1280, 1024, wl.EQUIDISTANT, 310.0, math.pi), wl.make_hoc(1.0, math.radians(90.0), 0.0, 0.3, np.float64)
    groups = [[(w.astype(np.float64), b.astype(np.float64), a) for w, b, a in g] for g in wl.glorot_network(np.random.default_rng(5), [3, 8, 3], 8, wl.SELU)]
    engine, image = eng.Engine64(groups, wl.NMGRID8), wl.random_image(np.random.default_rng(6), 1280, 1024, 4)
    for k in (0.3, 3.0, 14.0, 0.3):
        mesh = eng.Mesh64(wl.NMGRID8, wl.CIRCLE, 0.05, 1.0, k, 5.0)
        p, c = engine.project(mesh, Hoc, lens), engine(mesh, Hoc, lens, image, wl.fourcc("RGBA"))
        V = len(p["gidx"])
        assert V > 0 and (V * 52 > 64 << 20) == (k == 14.0)
        for key in ("px", "nb", "gidx"):
            assert np.array_equal(p[key], c[key]), key
        row = np.full(mesh.n_nodes + 1, V, np.int32)
        row[p["gidx"]] = np.arange(V)
        assert np.all(np.diff(p["gidx"]) > 0)
        assert np.array_equal(p["nb"][:V], row[mesh.arrays()[1][p["gidx"]]]) and np.all(p["nb"][V] == V)
        assert np.all((p["px"] >= 0) & (p["px"] + 1 < [1280, 1024]))
        assert c["cls"].shape == (V + 1, 3) and np.abs(c["cls"].sum(1) - 1).max() < 1e-12
