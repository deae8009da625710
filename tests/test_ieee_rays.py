"""Rays that take the reference's IEEE box test (a zero direction component,
or any ray of a scene whose boxes are outside the division-free range) in the
persistent traversal, against the oracle: alone in their waves and beside
other rays, where a wave gathers its nodes (neighbouring rays) and where it
stages them (rays in no order; waves of 64 rays, as only those reach the
stage)."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from rta_amd import scenes
from rta_amd.device import DeviceBuffer

from test_short_stack import Packed, same_records

BASE = 4096
WHOLE_WAVES = 200001      # more than 24 waves on each of 256 CUs take by halves


def mesh(flagged: bool):
    tris = scenes.heightfield(40, 40, seed=3)
    if flagged:
        tris["a"][11, 0] = 1e-30      # below the range of exact quotients
    return oracle.lbvh_build(tris)


def rays(zero_every: int, ordered: bool):
    rng = np.random.default_rng(7)
    if ordered:
        at = np.arange(BASE)
        o = np.stack([(at % 64 + 0.5) / 64, (at // 64 + 0.5) / 64, np.full(BASE, 2.0)], axis=1)
        d = np.tile([1e-3, 2e-3, -1.0], (BASE, 1))
        d[::zero_every, :2] = 0.0
    else:
        o = rng.uniform(0.0, 1.0, (BASE, 3))
        d = rng.normal(size=(BASE, 3))
        d[::zero_every, 0] = 0.0
        d[::2 * zero_every, 1] = 0.0
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    t = np.full(BASE, np.finfo(np.float32).max, np.float32)
    return o.astype(np.float32).reshape(-1), d.astype(np.float32).reshape(-1), t


@pytest.mark.gpu
@pytest.mark.parametrize("flagged", [False, True])
@pytest.mark.parametrize("ordered", [False, True])
@pytest.mark.parametrize("zero_every", [1, 2, 16])
@pytest.mark.parametrize("n", [BASE, WHOLE_WAVES])
def test_ieee_rays(gpu, n, zero_every, ordered, flagged):
    ref = mesh(flagged)
    o, d, t = rays(zero_every, ordered)
    at = np.arange(n) % BASE
    many = [DeviceBuffer.from_array(np.ascontiguousarray(a.reshape(BASE, -1)[at]).reshape(-1))
            for a in (o, d, t)]
    pk = Packed(ref["tris"], ref["nodes"])
    assert int(pk.flags.download(np.uint32, 1)[0]) == int(flagged)
    for shadow in (False, True):
        exp, _ = oracle.trace_kernel(ref["tris"], ref["nodes"], o, d, t, any_hit=shadow)
        assert (exp["t"] != t).any()
        got = pk.trace(*many, n, 32, shadow=shadow)
        assert same_records(got, exp[at])
