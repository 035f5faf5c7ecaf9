"""The C++ engine's calls that return their results by value (what a caller of the reference's interface uses), against the oracle."""
import ctypes as C
import math

import numpy as np
import pytest

from helpers import PROB_TOL, assert_classification_parity, assert_projection_parity
from oracle import vmo
from visualmesh_amd import engine as eng
from visualmesh_amd import native
from visualmesh_amd import workloads as wl

pytestmark = pytest.mark.gpu


def _fp(a):
    return a.ctypes.data_as(C.POINTER(C.c_float))


def _ip(a):
    return a.ctypes.data_as(C.POINTER(C.c_int32))


@pytest.mark.parametrize("model", ["ring6", "nmgrid8"])
def test_projection_and_classification_by_value(oracle, model):
    """Every array of both calls, and the table of a camera that sees nothing: its null row alone."""
    model_id, shape, radius, nn = {"ring6": (wl.RING6, wl.SPHERE, 0.0949, 6), "nmgrid8": (wl.NMGRID8, wl.CIRCLE, 0.05, 8)}[model]
    net = wl.glorot_network(np.random.default_rng(5), [3, 16, 3], nn, wl.SELU)
    args, lens = (model_id, shape, radius, 1.0, 4.0, 5.0), (320, 256, wl.RECTILINEAR, 175.0, math.pi / 2)
    mesh, o_mesh, e_lens, o_lens = eng.Mesh(*args), oracle.mesh(*args), native.make_lens(*lens), vmo.make_lens(*lens)
    image, fcc, lib = wl.random_image(np.random.default_rng(6), 320, 256, 4), wl.fourcc("RGBA"), native.host()
    engine = eng.Engine(net, model_id)
    for pitch in (50.0, -80.0, 30.0):
        Hoc = np.ascontiguousarray(wl.make_hoc(1.0, math.radians(pitch), 0.02, 0.3), dtype=np.float32)
        cap = mesh.n_nodes
        px, nb, gidx, cls = np.zeros((cap, 2), np.float32), np.full((cap + 1, nn), -7, np.int32), np.zeros(cap, np.int32), np.zeros((cap + 1, 3), np.float32)
        V = native.host_check(lib.vmh_engine_project(engine.ptr, mesh.ptr, _fp(Hoc), C.byref(e_lens), cap, _fp(px), _ip(nb), _ip(gidx)))
        want = o_mesh.project(Hoc, o_lens)
        assert (V == 0) == (pitch < 0)
        assert_projection_parity(dict(px=px[:V], nb=nb[:V + 1], gidx=gidx[:V]), want, "projection at %g degrees" % pitch)
        assert (nb[V + 1:] == -7).all()
        V = native.host_check(lib.vmh_engine_classify(engine.ptr, mesh.ptr, _fp(Hoc), C.byref(e_lens), image.ctypes.data, fcc, cap, _fp(px), _ip(nb), _ip(gidx), _fp(cls)))
        if pitch < 0:
            assert V == 0
            continue
        want = o_mesh.classify(Hoc, o_lens, image, fcc, vmo.Network(net))
        assert_classification_parity(dict(px=px[:V], nb=nb[:V + 1], gidx=gidx[:V], cls=cls[:V + 1]), want, PROB_TOL, "classification at %g degrees" % pitch)
