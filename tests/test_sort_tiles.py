"""The radix sort at the edges of its tiles (2,048 and 4,096 keys), of the
rule that lets the scatter sum the histograms itself (24 tiles) and of the
rule for larger tiles (2^19 keys): whole builds' codes order and the 32-bit
entry point against numpy's stable argsort."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import rta_amd
from rta_amd import scenes
from rta_amd.abi import call, ptr
from rta_amd.device import DeviceBuffer

SIZES = (1, 2047, 2048, 2049, 24 * 2048, 24 * 2048 + 1, 25 * 2048 + 7, 65 * 2048 + 3, 1 << 19,
         (1 << 19) + 1, (1 << 19) + 4095, 700_001)


@pytest.mark.gpu
@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("kind", ["random", "few"])
def test_sort_is_stable(gpu, n, kind):
    rng = np.random.default_rng(n)
    keys = (rng.integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32) if kind == "random"
            else rng.integers(0, 5, n).astype(np.uint32) * np.uint32(0x11000401))
    vals = np.arange(n, dtype=np.uint32)
    size = C.c_size_t(0)
    call("rta_lbvh_sort_work_bytes", n, C.byref(size))
    k, v, w = DeviceBuffer.from_array(keys), DeviceBuffer.from_array(vals), DeviceBuffer(size.value)
    call("rta_lbvh_sort", ptr(k), ptr(v), n, ptr(w), size, None)
    rta_amd.synchronize()
    order = np.argsort(keys, kind="stable")
    assert np.array_equal(k.download(np.uint32, n), keys[order])
    assert np.array_equal(v.download(np.uint32, n), vals[order])


@pytest.mark.gpu
@pytest.mark.parametrize("n", [12289, 24 * 2048, 24 * 2048 + 1, (1 << 19) + 1])
def test_build_orders_by_code(gpu, n):
    """The build's own passes (10-bit digits, three of them)."""
    g = int(np.ceil(np.sqrt(n / 2)))
    tris = np.random.default_rng(3).permutation(scenes.heightfield(g, g, seed=5)[:n])
    c = ((tris["a"] + tris["b"]) + tris["c"]) / np.float32(3.0)
    lo = np.minimum(np.minimum(tris["a"], tris["b"]), tris["c"]).min(axis=0)
    hi = np.maximum(np.maximum(tris["a"], tris["b"]), tris["c"]).max(axis=0)
    q = ((c - lo) * (np.float32(1024.0) / (hi - lo))).astype(np.uint32) & 0x3FF
    code = np.zeros(n, np.uint32)
    for bit in range(10):
        for axis in range(3):
            code |= ((q[:, axis] >> bit) & 1) << np.uint32(3 * bit + axis)
    bvh = rta_amd.LbvhConstructor().build(DeviceBuffer.from_array(tris), n)
    assert np.array_equal(bvh.indices(), np.argsort(code, kind="stable").astype(np.uint32))


def test_workspace_never_shrinks_with_n():
    """A workspace for n triangles serves every smaller mesh."""
    size, last = C.c_size_t(0), 0
    for n in sorted({1, 2, 2048, 2049, 12288, 12289, (1 << 19) - 1, 1 << 19, (1 << 19) + 1, 1 << 20}):
        call("rta_lbvh_workspace_bytes", n, C.byref(size))
        assert size.value >= last
        last = size.value
