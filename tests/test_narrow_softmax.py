"""The class layers of conv_narrow.hip: the precision and the range of their softmax."""
import math

import numpy as np
import pytest

from visualmesh_amd import engine as eng
from visualmesh_amd import native
from visualmesh_amd import workloads as wl

pytestmark = pytest.mark.gpu

# e^x below the smallest normal number for every class; a sum whose reciprocal is below it; large logits that lie close together and
# ones far apart; one class
LOGITS = [(-95.3, -96.1, -97.7, -95.9), (-98.9, -97.2, -99.4), (87.9, 3.0, -2.0, 80.0), (88.6, -60.0), (79.93, 79.17, 78.71, 77.39), (-71.3, -70.9, -70.1),
          (41.7, 40.3, 38.9, 37.7), (15.3, -14.9, 2.6, 0.7), (-88.9,)]


def _probabilities(model, c_in, logits):
    """(the class layer's rows, its kernel's name) with weights of zero and the logits as biases: the softmax alone"""
    model_id, shape, radius, nn = {"ring6": (wl.RING6, wl.SPHERE, 0.0949, 6), "nmgrid8": (wl.NMGRID8, wl.CIRCLE, 0.05, 8)}[model]
    rng = np.random.default_rng(6)
    mesh, lens, image = eng.Mesh(model_id, shape, radius, 1.0, 4.0, 5.0), native.make_lens(640, 512, wl.EQUISOLID, 210.0, math.pi), wl.random_image(rng, 640, 512, 4)
    net = wl.glorot_network(rng, [3, 16, c_in, len(logits)], nn, wl.SELU)
    w, _, activation = net[-1][-1]
    net[-1][-1] = (np.zeros_like(w), np.asarray(logits, np.float32), activation)
    engine = eng.Engine(net, model_id)
    engine.stage([dict(mesh=mesh, Hoc=wl.make_hoc(1.0, math.radians(30.0), 0.05, 0.3), lens=lens, image=image, fourcc=wl.fourcc("RGBA"))])
    engine.run()
    got = engine.fetch_packed()[0]["cls"].copy()
    engine.profile(True)
    engine.run()
    assert len(got) > 1000
    return got, engine.profile_read()[-1][0]


def _check(got, logits, relative):
    """Within `relative` of the double value. Where some e^x is denormal, each of them is off by up to 2 of its units of 2^-149 instead:
    that for the term and for every term of the sum, over the sum."""
    e = np.exp(np.asarray(logits, np.float32).astype(np.float64))
    want = e / e.sum()
    denormal = (len(e) + 1) * 2.0 ** -148 / e.sum() if e.min() < 2.0 ** -126 else 2.0 ** -149
    assert (np.abs(got - want) <= relative * want + denormal).all(), (logits, got[0], want, np.abs(got / want - 1.0).max())


@pytest.mark.parametrize("c_in,model", [(32, "ring6"), (48, "nmgrid8"), (64, "ring6")])
def test_softmax_of_logits_near_the_ends_of_the_range(c_in, model):
    """Within 5e-7: an ulp (1.2e-7) for e^x, the same for its sum and 3 roundings of 6e-8, one for the division."""
    for logits in LOGITS:
        got, name = _probabilities(model, c_in, logits)
        assert name.startswith("conv_narrow_%dx%d" % (c_in, len(logits)))
        _check(got, logits, 5e-7)


@pytest.mark.parametrize("c_in,c_out,model", [(16, 2, "ring6"), (16, 3, "ring6"), (24, 4, "nmgrid8")])
def test_softmax_of_thin_rows(c_in, c_out, model):
    """The hardware's exponential up to logits of 85: |x| 1e-7 more for e^x and for its sum. The library's beyond."""
    more = {2: [(85.9, 86.3), (-99.1, -98.3)], 3: [(86.3, 86.9, 87.0), (12.9, -86.0, 13.1)], 4: [(86.0, 86.2, 86.4, 86.1)]}[c_out]
    for logits in [x for x in LOGITS if len(x) == c_out] + more:
        got, name = _probabilities(model, c_in, logits)
        assert name.startswith("conv_narrow_%dx%d" % (c_in, c_out))
        far = max(abs(x) for x in logits)
        _check(got, logits, 5e-7 + (2e-7 * far if far <= 85.0 else 0.0))
