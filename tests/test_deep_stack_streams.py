"""Spilled stack entries of traversals that run at once: the waves of both
streams take their slots from one pool, and every slot comes back.  The
launches together claim many times the pool's 8,192 slots, so one that were
kept would end in counted stack overflows."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import oracle
import rta_amd
from rta_amd.abi import HIT_DTYPE, TraceConfig, call, ptr
from rta_amd.device import DeviceBuffer, Stream

from test_short_stack import Packed, same_records
from test_traversal_paths import forest, forest_rays

ROUNDS = 12
RAYS = 200001            # 64 a wave: 3,126 waves, nearly all with deep rays


@pytest.mark.gpu
def test_two_streams_spill_at_once(gpu):
    tris, nodes = forest()
    o, d, t = forest_rays(True)
    at = np.arange(RAYS) % len(t)
    ro, rd, rt = (DeviceBuffer.from_array(np.ascontiguousarray(a.reshape(len(t), -1)[at]).reshape(-1))
                  for a in (o, d, t))
    pk = Packed(tris, nodes)
    cfg = TraceConfig(64, 16, 32, 0, 10, 32)
    lanes = []
    for shadow in (False, True):
        hits, err, queue = DeviceBuffer(16 * RAYS), DeviceBuffer(4), DeviceBuffer(4)
        call("rta_reset_intersections", ptr(hits), RAYS, 1, None)
        err.fill_u32(0)
        lanes.append((shadow, Stream(), hits, err, queue))
    rta_amd.synchronize()
    for _ in range(ROUNDS):
        for shadow, stream, hits, err, queue in lanes:
            call("rta_trace_shadow_cis_persistent" if shadow else "rta_trace_cis_persistent",
                 ptr(pk.tri4), ptr(pk.pairs), ptr(pk.flags), pk.root[0], pk.root[1], ptr(ro), ptr(rd),
                 ptr(rt), RAYS, None, ptr(hits), ptr(err), ptr(queue), C.byref(cfg), ptr(stream))
    rta_amd.synchronize()
    for shadow, _, hits, err, _ in lanes:
        exp, _ = oracle.trace_kernel(tris, nodes, o, d, t, any_hit=shadow)
        assert int(err.download(np.uint32, 1)[0]) == 0
        assert same_records(hits.download(HIT_DTYPE, RAYS), exp[at])
