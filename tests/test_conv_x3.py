"""fp32 layers on the bf16 matrix instructions with every factor in three parts (conv_x3.hip, conv_x3_tile.hip)."""
import math
import os
import re

import numpy as np
import pytest

from visualmesh_amd import engine as eng
from visualmesh_amd import native
from visualmesh_amd import workloads as wl

# widths, the kernels of the layers behind the first, and of the same layers as fp32 products
NETWORKS = {"64": ([3, 64, 64, 64, 64, 4], ["conv_x3_64x64s7"] * 3, ["conv_mfma_64x64s7"] * 3),
            "32": ([3, 16, 32, 32, 32, 4], ["conv_x3_tile_16x32s7"] + ["conv_x3_tile_32x32s7"] * 2, ["conv_mfma_16x32s7"] + ["conv_mfma_32x32s7"] * 2),
            "uniform 32": ([3, 32, 32, 32, 32, 4], ["conv_x3_tile_32x32s7"] * 3, ["conv_mfma_32x32s7"] * 3)}


@pytest.mark.parametrize("file,kernels", [("conv_x3.hip", 2), ("conv_x3_tile.hip", 4)])
def test_kernels_do_not_spill(tmp_path, file, kernels):
    """Weights live in registers as in conv_bf16.hip, and the waits are counted by hand: no kernel may touch scratch memory."""
    import subprocess
    from visualmesh_amd import build as vm_build
    out = tmp_path / "kernels.s"
    flags = [f for f in vm_build.HIP_FLAGS if f != "-fPIC"]
    subprocess.run([vm_build.HIPCC] + flags + ["-S", "--cuda-device-only", "-o", str(out), os.path.join(vm_build.CSRC, file)],
                   check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    text = out.read_text()
    sizes = [int(x) for x in re.findall(r"\.private_segment_fixed_size:\s+(\d+)", text)]
    assert len(sizes) == kernels and not any(sizes), sizes
    assert "scratch_" not in text


def _network(widths, activation=wl.SELU, seed=3):
    return wl.glorot_network(np.random.default_rng(seed), list(widths), 6, activation)


def _frames(n, k, seed=5, blind=()):
    rng = np.random.default_rng(seed)
    mesh, lens, fcc = eng.Mesh(wl.RING6, wl.SPHERE, 0.0949, 1.0, k, 8.0), native.make_lens(320, 256, wl.EQUISOLID, 105.0, math.pi), wl.fourcc("RGBA")
    sky = native.make_lens(320, 256, wl.RECTILINEAR, 176.0, math.pi / 2)
    image = wl.random_image(rng, 320, 256, 4)
    return [dict(mesh=mesh, Hoc=wl.make_hoc(1.0, math.radians(-80.0 if i in blind else rng.uniform(20, 60)), rng.uniform(-0.1, 0.1), rng.uniform(-3, 3)),
                 lens=sky if i in blind else lens, image=image, fourcc=fcc) for i in range(n)]


def _run(engine, frames):
    """(results, names of the layers' kernels)"""
    engine.stage(frames)
    engine.run()
    out = engine.fetch()
    engine.profile(1)
    engine.run()
    names = [n for n, _, _ in engine.profile_read() if n.startswith("conv")]
    engine.profile(0)
    return out, names


def _float64(network, frames, results):
    """the network on the engine's own neighbourhoods and the oracle's sampled inputs, in float64 (selu with the exact exponential)"""
    from oracle import vmo
    O, out = vmo.load("oracle"), []
    for f, r in zip(frames, results):
        if not len(r["gidx"]):
            out.append(np.zeros((0, network[-1][-1][0].shape[1])))
            continue
        x = np.array([O.fn_interpolate(p, f["image"], f["lens"].width, f["lens"].height, f["fourcc"]) for p in r["px"]], np.float64)
        x = np.concatenate([x, np.full((1, 4), -1.0)])
        for (w, b, a), in network:
            y = np.concatenate([x[:, None, :], x[r["nb"]]], axis=1).reshape(len(x), -1) @ w.astype(np.float64) + b.astype(np.float64)
            if a == wl.SELU:
                x = 1.0507009873554804934193349852946 * np.where(y >= 0, y, 1.6732632423543772848170429916717 * np.expm1(np.minimum(y, 0)))
            elif a == wl.RELU:
                x = np.maximum(y, 0)
            else:
                e = np.exp(y)
                x = e / e.sum(1, keepdims=True)
        out.append(x)
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("activation", [wl.SELU, wl.RELU], ids=["selu", "relu"])
@pytest.mark.parametrize("n,k,blind", [(1, 0.6, ()), (1, 1.0, ()), (3, 1.4, (1,)), (2, 3.0, ()), (16, 1.2, (0, 7)), (1, 5.0, ()), (6, 6.0, ())])
@pytest.mark.parametrize("width", sorted(NETWORKS))
def test_against_the_chain_of_fp32_products(width, n, k, blind, activation, monkeypatch):
    """Frames of a few rows up to more tiles than blocks, with and without frames that see nothing: within what two orders of fp32 sums
    differ by. A sum of 448 products carries about sqrt(448) 2^-24 = 1.3e-6 of its size whatever the order; four such layers in a row and
    a factor of two for the largest of many rows: 1e-5 of a probability."""
    widths, kernels, fp32_kernels = NETWORKS[width]
    network, frames = _network(widths, activation), _frames(n, k, blind=blind)
    got, names = _run(eng.Engine(network, wl.RING6), frames)
    assert names[-4:-1] == kernels, names
    monkeypatch.setenv("VMHIP_CONV_KERNEL", "mfma")
    want, names = _run(eng.Engine(network, wl.RING6), frames)
    assert names[-4:-1] == fp32_kernels, names
    assert sum(len(w["gidx"]) for w in want) > 0
    for g, w in zip(got, want):
        assert np.array_equal(g["gidx"], w["gidx"]) and np.array_equal(g["nb"], w["nb"])
        assert g["cls"].shape == w["cls"].shape
        if len(w["gidx"]):
            assert np.abs(g["cls"] - w["cls"]).max() <= 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("width", sorted(NETWORKS))
def test_rows_that_are_not_staged_give_the_same_bits(width, monkeypatch):
    """With few halo slots most tiles are computed from memory: the same parts multiplied in the same order."""
    widths, kernels, _ = NETWORKS[width]
    network, frames = _network(widths), _frames(3, 3.0)
    want, _ = _run(eng.Engine(network, wl.RING6), frames)
    for cap in (0, 8, 60, 128, 200):
        monkeypatch.setenv("VMHIP_HALO_CAP", str(cap))
        got, names = _run(eng.Engine(network, wl.RING6), frames)
        assert names[-4:-1] == kernels, names
        for g, w in zip(got, want):
            assert np.array_equal(g["cls"], w["cls"]), cap


@pytest.mark.gpu
@pytest.mark.parametrize("width", sorted(NETWORKS))
def test_a_frame_alone_and_among_others(width):
    """A few tiles (two blocks to each) and many: the same bits, pass after pass."""
    network, frames = _network(NETWORKS[width][0]), _frames(12, 4.0)
    engine = eng.Engine(network, wl.RING6)
    together, _ = _run(engine, frames)
    assert sum(len(r["gidx"]) for r in together) > 40000
    for i in (0, 5, 11):
        alone, _ = _run(engine, frames[i:i + 1])
        assert np.array_equal(alone[0]["cls"], together[i]["cls"])
    engine.stage(frames)
    for _ in range(4):
        engine.run()
        for a, b in zip(engine.fetch(), together):
            assert np.array_equal(a["cls"], b["cls"])


@pytest.mark.gpu
def test_networks_whose_activations_could_leave_the_range():
    """Weights by which a sum could reach 1e30, infinite ones and such that are no numbers, whichever channel they belong to, and activations
    without this kernel: the fp32 instructions, as ever."""
    frames = _frames(1, 1.5)
    for change in ("large", "infinite", "nan", "infinite, then nan", "nan bias", "tanh", "none"):
        network = _network([3, 64, 64, 64, 4], wl.TANH if change == "tanh" else wl.SELU)
        if change == "large":
            network = [[(w * (1e14 if i in (0, 1) else 1), b, a) for w, b, a in g] for i, g in enumerate(network)]
        if change.startswith("infinite"):
            network[1][0][0][5, 7] = np.inf
        if change.endswith("nan"):  # channels with finite sums follow
            network[1][0][0][9, 8] = np.nan
        if change == "nan bias":
            network[1][0][1][30] = np.nan
        _, names = _run(eng.Engine(network, wl.RING6), frames)
        assert names.count("conv_x3_64x64s7") == (2 if change == "none" else 0), (change, names)


@pytest.mark.gpu
@pytest.mark.parametrize("widths", [[3] + [64] * 6 + [4], [3, 16, 32, 32, 32, 32, 32, 16, 3], [3, 32, 32, 32, 32, 3]], ids=["64", "32", "uniform 32"])
def test_sums_are_closer_to_float64_than_those_of_fp32_products(widths, monkeypatch):
    """The distance of the probabilities from float64 is no larger than that of the chain of fp32 products (about half of it where
    measured: 1.6e-7 against 3.9e-7, 2.1e-7 against 4.0e-7, 1.1e-7 against 2.2e-7)."""
    network, frames = _network(widths, seed=20), _frames(1, 2.0)
    got, names = _run(eng.Engine(network, wl.RING6), frames)
    assert any(n.startswith("conv_x3") for n in names), names
    monkeypatch.setenv("VMHIP_CONV_KERNEL", "mfma")
    plain, _ = _run(eng.Engine(network, wl.RING6), frames)
    want = _float64(network, frames, got)
    error = [np.sqrt(np.mean((r[0]["cls"] - want[0]) ** 2)) for r in (got, plain)]
    print("rms error: %.3g, of fp32 products %.3g" % tuple(error), flush=True)
    assert error[0] <= error[1]
