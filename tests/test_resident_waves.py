"""Launches at the sizes where 32 or 64 rays a wave just fit the waves that 256
CUs hold, 21 each, and one ray beyond: rays of every stack depth in no order
against the oracle."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from rta_amd.device import DeviceBuffer

from test_short_stack import Packed, same_records
from test_traversal_paths import forest, forest_rays


@pytest.mark.gpu
@pytest.mark.parametrize("n", [21 * 256 * 32, 21 * 256 * 32 + 1, 21 * 256 * 64, 21 * 256 * 64 + 1])
def test_rays_of_resident_waves(gpu, n):
    tris, nodes = forest()
    o, d, t = forest_rays(True)
    at = np.arange(n) % len(t)
    many = [DeviceBuffer.from_array(np.ascontiguousarray(a.reshape(len(t), -1)[at]).reshape(-1))
            for a in (o, d, t)]
    pk = Packed(tris, nodes)
    for shadow in (False, True):
        exp, _ = oracle.trace_kernel(tris, nodes, o, d, t, any_hit=shadow)
        assert same_records(pk.trace(*many, n, 32, shadow=shadow), exp[at])
