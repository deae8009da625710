"""The one-workgroup scene box, codes and sort of small meshes: sizes at the
edges of its items per thread and of the rule that picks it, against the
oracle's build, with duplicate codes and a code of 0 among them."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
import rta_amd
from rta_amd import scenes
from rta_amd.device import DeviceBuffer

SIZES = (1, 2, 63, 64, 65, 1023, 1024, 1025, 2048, 2049, 4096, 4097, 6144, 6145, 8193, 10240, 10241,
         12287, 12288, 12289)


@pytest.mark.gpu
@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("shape", ["surface", "crowded"])
def test_small_build_equals_the_oracle(gpu, n, shape):
    if shape == "surface":
        g = int(np.ceil(np.sqrt(n / 2)))
        tris = scenes.heightfield(g, g, seed=n)[:n]
    else:
        # many triangles in few Morton cells, and one at the box's corner
        rng = np.random.default_rng(n)
        tris = scenes.random_triangles(n, seed=n, edge_min=1e-5, edge_max=1e-4)
        for f in ("a", "b", "c"):
            tris[f] = tris[f] * np.float32(0.002) + np.round(rng.random((n, 1)) * 4).astype(np.float32)
    tris = np.random.default_rng(1).permutation(tris)
    ref = oracle.lbvh_build(tris)
    dev = DeviceBuffer.from_array(tris)
    ctor = rta_amd.LbvhConstructor()
    bvh = ctor.build(dev, n)
    assert np.array_equal(bvh.indices(), ref["indices"])
    assert bvh.canonical_triangle_ptr().tobytes() == ref["tris"].tobytes()
    got = bvh.nodes()
    for f in ("type_left_elems", "right_tris", "min", "max"):
        assert np.array_equal(got[f], ref["nodes"][f]), f
