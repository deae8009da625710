"""The inference's selection around the bounds of its two ways through layer
4: logits of the largest size that four keys at a time may meet, activations
around their bound, and logits that are not finite (whose choice must not
depend on the launch)."""
from __future__ import annotations

import numpy as np
import pytest

import rta_amd
from rta_amd import predictor as P
from rta_amd.device import DeviceBuffer

from test_predictor import HI, LO, _random_rays, keyed_top4

RAYS = 77
MANY = 32 * (4 * 256) + 33     # more than one wave a SIMD


def infer(pred, o, d, top_k, with_logits):
    n = len(o) // 3
    logits = DeviceBuffer(4160 * n) if with_logits else None
    top = DeviceBuffer(16 * n)
    pred.infer(DeviceBuffer.from_array(o), DeviceBuffer.from_array(d), n, top=top, logits=logits,
               top_k=top_k)
    rta_amd.synchronize()
    got = top.download(np.int32, 4 * n).reshape(n, 4)
    return got, logits.download(np.float32, 1040 * n).reshape(n, 1040) if with_logits else None


def network(w4_scale, b4_scale, h3_scale):
    """Weights whose layer 4 and whose last hidden layer have the given sizes."""
    pred = P.HitPredictor(1024, seed=5, scene_min=LO, scene_max=HI)
    params = pred.params()
    rng = np.random.default_rng(31)
    w4, b4, w3 = P.LAYOUT["W4"][0], P.LAYOUT["b4"][0], P.LAYOUT["W3"][0]
    params[w4:w4 + 1024 * 64] = rng.uniform(-w4_scale, w4_scale, 1024 * 64).astype(np.float32)
    params[b4:b4 + 1024] = rng.uniform(-b4_scale, b4_scale, 1024).astype(np.float32)
    params[w3:w3 + 64 * 64] *= np.float32(h3_scale)
    pred.set_params(params)
    return pred


def tiled(a, n):
    return np.ascontiguousarray(a.reshape(RAYS, 3)[np.arange(n) % RAYS]).reshape(-1)


# weights just below 2^34 and biases just below 2^66; activations far below,
# around and above 2^66
@pytest.mark.gpu
@pytest.mark.parametrize("top_k", [1, 4])
@pytest.mark.parametrize("h3_scale", [1.0, 2.0 ** 60, 2.0 ** 64, 2.0 ** 66, 2.0 ** 68])
def test_largest_logits(gpu, h3_scale, top_k):
    pred = network(0.99 * 2.0 ** 34, 0.99 * 2.0 ** 66, h3_scale)
    o, d = _random_rays(RAYS, 29)
    got, logits = infer(pred, o, d, top_k, True)
    assert np.isfinite(logits).all() and np.abs(logits).max() > 2.0 ** 34 * h3_scale / 2.0 ** 8
    exp = keyed_top4(logits)
    if top_k == 1:
        exp[:, 1:] = -1
    assert np.array_equal(got, exp)
    for with_logits in (False, True):
        got, _ = infer(pred, tiled(o, MANY), tiled(d, MANY), top_k, with_logits)
        assert np.array_equal(got, exp[np.arange(MANY) % RAYS])


@pytest.mark.gpu
@pytest.mark.parametrize("top_k", [1, 4])
def test_logits_that_are_not_finite(gpu, top_k):
    """Sums that overflow: the launch's size and the logits output do not
    change a ray's choice."""
    pred = network(2.0 ** 70, 2.0 ** 70, 2.0 ** 60)
    o, d = _random_rays(RAYS, 29)
    exp, logits = infer(pred, o, d, top_k, True)
    assert not np.isfinite(logits).all()
    for n in (RAYS, MANY):
        for with_logits in (False, True):
            got, _ = infer(pred, tiled(o, n), tiled(d, n), top_k, with_logits)
            assert np.array_equal(got, exp[np.arange(n) % RAYS])
