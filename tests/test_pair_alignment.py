"""Pair records at an address that is 16-byte but not 64-byte aligned: the
entry points take any device pointer that float4 loads can read, so the
persistent traversal gives the oracle's records there too, also for rays in no
order in waves of 64 rays (which stage aligned records through LDS)."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from rta_amd import scenes
from rta_amd.abi import call, ptr
from rta_amd.device import DeviceBuffer, DeviceView

from test_ieee_rays import BASE, WHOLE_WAVES
from test_short_stack import Packed, same_records


def rays():
    rng = np.random.default_rng(12)
    o = rng.uniform(0.0, 1.0, (BASE, 3))
    d = rng.normal(size=(BASE, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    t = np.full(BASE, np.finfo(np.float32).max, np.float32)
    return o.astype(np.float32).reshape(-1), d.astype(np.float32).reshape(-1), t


def shifted(buf: DeviceBuffer, offset: int) -> DeviceView:
    """A copy of the buffer that starts `offset` bytes into an allocation."""
    view = DeviceView(DeviceBuffer(buf.nbytes + 64), offset, buf.nbytes)
    call("rta_hip_memcpy_dtod", ptr(view), ptr(buf), buf.nbytes, None)
    return view


@pytest.mark.gpu
@pytest.mark.parametrize("offset", [0, 16, 32, 48])
@pytest.mark.parametrize("block", [64, 256])
def test_shifted_pairs(gpu, offset, block):
    ref = oracle.lbvh_build(scenes.heightfield(40, 40, seed=3))
    o, d, t = rays()
    at = np.arange(WHOLE_WAVES) % BASE
    many = [DeviceBuffer.from_array(np.ascontiguousarray(a.reshape(BASE, -1)[at]).reshape(-1))
            for a in (o, d, t)]
    pk = Packed(ref["tris"], ref["nodes"])
    pk.pairs = shifted(pk.pairs, offset)
    assert pk.pairs.ptr % 64 == offset
    for shadow in (False, True):
        exp, _ = oracle.trace_kernel(ref["tris"], ref["nodes"], o, d, t, any_hit=shadow)
        assert same_records(pk.trace(*many, WHOLE_WAVES, 32, shadow=shadow, block=block), exp[at])
