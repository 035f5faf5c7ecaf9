"""The class layer of wide rows (conv_narrow.hip) in four-neighbour meshes: five gather slots, an 8-byte row of the neighbour table."""
import ctypes as C
import math

import numpy as np
import pytest

from helpers import PROB_TOL
from visualmesh_amd import engine as eng
from visualmesh_amd import native
from visualmesh_amd import workloads as wl

pytestmark = pytest.mark.gpu


def _fp(a):
    return a.ctypes.data_as(C.POINTER(C.c_float))


def _ip(a):
    return a.ctypes.data_as(C.POINTER(C.c_int32))


# every width; a mesh of one tile, several, with all neighbours staged and with most of the halo read from global memory
@pytest.mark.parametrize("c_in,c_out,k,max_distance,halo_cap", [(64, 3, 4.0, 8.0, None), (64, 4, 4.0, 8.0, "8"), (48, 4, 4.0, 8.0, None), (32, 2, 1.5, 2.0, None),
                                                                 (32, 1, 6.0, 20.0, "8")])
def test_class_layer_with_five_slots(oracle, monkeypatch, c_in, c_out, k, max_distance, halo_cap):
    """The first four neighbours of a Ring6 mesh through the C ABI, against the definition of the layers in float64 on the returned
    neighbourhood and on the oracle's samples at the returned pixels (fp32's parity bar); one output channel uses tanh."""
    if halo_cap:
        monkeypatch.setenv("VMHIP_HALO_CAP", halo_cap)
    lib, nn, W, H = native.hip(), 4, 640, 512
    rng = np.random.default_rng(44)
    mesh = eng.Mesh(wl.RING6, wl.SPHERE, 0.0949, 1.0, k, max_distance)
    rays, nbr = mesh.arrays()
    nbr = np.ascontiguousarray(nbr[:, :nn])
    lens = native.make_lens(W, H, wl.EQUISOLID, 210.0, math.pi)
    Hoc = np.ascontiguousarray(wl.make_hoc(1.0, math.radians(40.0), 0.02, 0.3), dtype=np.float32)
    ranges, image = np.ascontiguousarray(mesh.lookup(Hoc, lens), dtype=np.int32), wl.random_image(rng, W, H, 4)
    groups = wl.glorot_network(rng, [3, 16, c_in, c_out], nn, wl.SELU)
    if c_out == 1:
        groups[-1] = [(w, b, wl.TANH) for w, b, _ in groups[-1]]
    net, engine, handle, batch = native.Network(groups), C.c_void_p(), C.c_void_p(), C.c_void_p()
    native.hip_check(lib.vmhip_engine_create(C.byref(net.c), nn, native.FP32, C.byref(engine)))
    native.hip_check(lib.vmhip_mesh_upload(_fp(rays), _ip(nbr), mesh.n_nodes, nn, C.byref(handle)))
    Rco = np.ascontiguousarray(Hoc[:3, :3].T)
    frame = native.Frame(handle, (C.c_float * 9)(*Rco.ravel()), lens, _ip(ranges), len(ranges), image.ctypes.data, wl.fourcc("RGBA"), None)
    native.hip_check(lib.vmhip_batch_create(engine, C.byref(batch)))
    native.hip_check(lib.vmhip_batch_stage(batch, C.byref(frame), 1, 1))
    native.hip_check(lib.vmhip_batch_profile(batch, 1))
    native.hip_check(lib.vmhip_batch_run(batch))
    names = [n for n, _, _ in native.profile_read(batch)]
    n_cand = int((ranges[:, 1] - ranges[:, 0]).sum())
    px, gidx, nb, cls = np.zeros((n_cand, 2), np.float32), np.zeros(n_cand, np.int32), np.zeros((n_cand + 1, nn), np.int32), np.zeros((n_cand + 1, c_out), np.float32)
    result = native.Result(n_cand, 0, _fp(px), _ip(gidx), _ip(nb), _fp(cls))
    native.hip_check(lib.vmhip_batch_fetch(batch, C.byref(result)))
    lib.vmhip_batch_destroy(batch)
    lib.vmhip_mesh_release(handle)
    lib.vmhip_engine_destroy(engine)
    assert [n for n in names if n.startswith("conv_narrow")] == ["conv_narrow_%dx%ds5" % (c_in, c_out)], names
    V = result.n_visible
    assert V > 200
    row_of = np.full(mesh.n_nodes + 1, V, np.int32)
    row_of[gidx[:V]] = np.arange(V, dtype=np.int32)
    table = np.concatenate([row_of[nbr[gidx[:V]]], np.full((1, nn), V, np.int32)])
    assert np.array_equal(nb[:V + 1], table)
    x = np.concatenate([np.stack([oracle.fn_interpolate(px[i], image, W, H, wl.fourcc("RGBA")) for i in range(V)]), -np.ones((1, 4), np.float32)]).astype(np.float64)
    alpha, scale = 1.6732632423543772848170429916717, 1.0507009873554804934193349852946
    for (w, b, act), in groups:
        x = np.concatenate([x] + [x[table[:, j]] for j in range(nn)], axis=1) @ w.astype(np.float64) + b.astype(np.float64)
        if act == wl.SELU:
            x = scale * np.where(x >= 0, x, alpha * np.exp(np.minimum(x, 0)) - alpha)
        else:
            x = np.tanh(x) if act == wl.TANH else np.exp(x) / np.exp(x).sum(axis=1, keepdims=True)
    worst = float(np.abs(cls[:V + 1] - x).max())
    print("%d -> %d: V = %d, worst %.3e" % (c_in, c_out, V, worst), flush=True)
    assert worst <= PROB_TOL
