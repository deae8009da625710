"""The persistent traversal's two ways to fetch a node (each lane its own
record, or a quad of lanes one record after another through LDS) and its
spilled stack entries, against the oracle: a forest of chain trees
(test_stack_depth) under a balanced top, one chain per stack depth from 1 to
32 entries, whose rays in shuffled order stand at different nodes (the
staged fetch) and in chain order at the same ones; and boxes with min > max,
which only the IEEE test orders as the reference does."""
from __future__ import annotations


import numpy as np
import pytest

import oracle
from rta_amd import scenes
from rta_amd.abi import NODE_DTYPE
from rta_amd.device import DeviceBuffer

from test_short_stack import Packed, same_records
from test_stack_depth import chain_rays, chain_tree

FOREST = 64
GAP = 20.0


def forest():
    """(triangles, nodes): chain j (1 + j % 32 pushes) moved by j * GAP
    along y, below FOREST - 1 top nodes in heap order."""
    tris, nodes = [], []
    top = np.zeros(FOREST - 1, NODE_DTYPE)
    root, lo, hi = [0] * FOREST, [None] * (2 * FOREST - 1), [None] * (2 * FOREST - 1)
    node_at, tri_at = FOREST - 1, 0
    for j in range(FOREST):
        t, nd = chain_tree(1 + j % 32)
        for f in ("a", "b", "c"):
            t[f][:, 1] += GAP * j
        for f in ("min", "max"):
            nd[f][:, 1] += GAP * j
        inner = (nd["type_left_elems"] & 1) == 1
        nd["type_left_elems"][inner] += 2 * node_at
        nd["right_tris"][inner] += node_at
        nd["right_tris"][~inner] += tri_at
        root[j] = node_at
        lo[FOREST - 1 + j], hi[FOREST - 1 + j] = nd["min"][0], nd["max"][0]
        tris.append(t)
        nodes.append(nd)
        node_at += len(nd)
        tri_at += len(t)
    ident = lambda i: i if i < FOREST - 1 else root[i - (FOREST - 1)]   # noqa: E731
    for i in reversed(range(FOREST - 1)):
        left, right = 2 * i + 1, 2 * i + 2
        lo[i], hi[i] = np.minimum(lo[left], lo[right]), np.maximum(hi[left], hi[right])
        top[i]["type_left_elems"] = (ident(left) << 1) | 1
        top[i]["right_tris"] = ident(right)
        top[i]["min"], top[i]["max"] = lo[i], hi[i]
    return np.concatenate(tris), np.concatenate([top] + nodes)


def forest_rays(shuffled: bool):
    """chain_rays of every chain, moved with it; in chain order or shuffled."""
    o, d, t = chain_rays(61)
    n = len(t)
    ro = np.concatenate([o.reshape(-1, 3) + np.float32([0, GAP * j, 0]) for j in range(FOREST)])
    rd = np.tile(d.reshape(-1, 3), (FOREST, 1))
    rt = np.tile(t, FOREST)
    assert len(rt) == n * FOREST
    if shuffled:
        p = np.random.default_rng(9).permutation(len(rt))
        ro, rd, rt = ro[p], rd[p], rt[p]
    return (np.ascontiguousarray(ro, np.float32).reshape(-1),
            np.ascontiguousarray(rd, np.float32).reshape(-1), rt)


def test_forest_reaches_every_depth():
    tris, nodes = forest()
    o, d, t = forest_rays(False)
    hits, deep, depth = oracle.trace_kernel(tris, nodes, o, d, t, depth=True)
    assert deep == 0 and (hits["t"] != np.float32(np.finfo(np.float32).max)).all()
    assert set(np.unique(depth)) == set(range(1, 33))


@pytest.mark.gpu
@pytest.mark.parametrize("shuffled", [False, True])
@pytest.mark.parametrize("shadow", [False, True])
@pytest.mark.parametrize("stack", [16, 24, 32])
@pytest.mark.parametrize("block", [64, 256])
def test_every_stack_depth(gpu, shuffled, shadow, stack, block):
    tris, nodes = forest()
    o, d, t = forest_rays(shuffled)
    exp, _ = oracle.trace_kernel(tris, nodes, o, d, t, any_hit=shadow)
    pk = Packed(tris, nodes)
    ovf = DeviceBuffer(4 * (len(t) + 1)) if stack < 32 else None
    got = pk.trace(DeviceBuffer.from_array(o), DeviceBuffer.from_array(d),
                   DeviceBuffer.from_array(t), len(t), stack, shadow=shadow, ovf=ovf, block=block)
    assert same_records(got, exp)
    if ovf is not None:
        _, _, depth = oracle.trace_kernel(tris, nodes, o, d, t, depth=True, any_hit=shadow)
        assert int(ovf.download(np.uint32, 1)[0]) == int((depth > stack).sum())


# 16, 32 or 64 rays a wave without a queue, or waves that share one: the
# largest launch of each and the next, on a chip of 256 CUs with 20 waves each
@pytest.mark.gpu
@pytest.mark.parametrize("shadow", [False, True])
@pytest.mark.parametrize("n", [1, 17, 16384, 16385, 163840, 163841, 327680, 327681])
def test_rays_per_wave(gpu, n, shadow):
    tris, nodes = forest()
    o, d, t = forest_rays(True)
    exp, _ = oracle.trace_kernel(tris, nodes, o, d, t, any_hit=shadow)
    at = np.arange(n) % len(t)
    o, d = (np.ascontiguousarray(a.reshape(-1, 3)[at]).reshape(-1) for a in (o, d))
    got = Packed(tris, nodes).trace(DeviceBuffer.from_array(o), DeviceBuffer.from_array(d),
                                    DeviceBuffer.from_array(t[at]), n, 32, shadow=shadow)
    assert same_records(got, exp[at])


@pytest.mark.gpu
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_boxes_with_min_above_max(gpu, axis):
    """Nodes whose box has min > max on one axis: the reference swaps the two
    quotients, so such a box is tested like the ordered one."""
    mesh = scenes.heightfield(40, 40, seed=3)
    ref = oracle.lbvh_build(mesh)
    nodes = ref["nodes"].copy()
    lo = nodes["min"][5::7, axis].copy()
    nodes["min"][5::7, axis] = nodes["max"][5::7, axis]
    nodes["max"][5::7, axis] = lo
    rng = np.random.default_rng(2)
    n = 5000
    o = rng.uniform(0.0, 1.0, (n, 3)).astype(np.float32).reshape(-1)
    d = rng.normal(size=(n, 3))
    d = (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32).reshape(-1)
    t = np.full(n, np.finfo(np.float32).max, np.float32)
    exp, _ = oracle.trace_kernel(ref["tris"], nodes, o, d, t)
    got = Packed(ref["tris"], nodes).trace(DeviceBuffer.from_array(o), DeviceBuffer.from_array(d),
                                           DeviceBuffer.from_array(t), n, 32)
    assert same_records(got, exp)
