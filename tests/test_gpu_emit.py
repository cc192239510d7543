"""The one-launch emission of a pass's outputs where its parts meet: meshes
that begin inside a row of 512 nodes and off every 16-byte boundary, rows that
hold several meshes and levels, segment tables of at most 64 entries, above
64 and above 4096 (the lookup takes one, two and three steps), and 64-bit codes
from 32-bit keys.  Every field equals the oracle's, bit for bit."""
import numpy as np
import pytest

import pyoracle as po
from parity import compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 9, 70, 900])
@pytest.mark.parametrize("key_bits,flags", [(0, 0), (64, 0), (0, 1)])
def test_small_meshes_end_to_end(gpu_ctx, n, key_bits, flags):
    rng = np.random.default_rng(n)
    meshes = []
    for i in range(n):
        pts = rng.normal(size=(3 + i % 5, 3)).astype(np.float32)
        tri = np.stack([np.arange(k, k + 3) for k in range(len(pts) - 2)]).astype(np.int32)
        meshes.append((pts, tri, int(rng.integers(1, 33))))
    trees, st = gpu_ctx.build_batch(meshes, key_bits=key_bits, flags=flags)
    assert not any(st), st
    step = max(1, n // 60)
    for (p, t, res), tree in list(zip(meshes, trees))[::step]:
        ref = po.build(p, t, res, key_bits=key_bits or 32)
        fields = None if not flags else ["voxels", "code", "is_leaf", "origin", "width", "parent",
                                         "childs", "neighbors", "level_nodes"]
        compare(tree, ref, fields=fields, check_aos=not key_bits and not flags)


@pytest.mark.parametrize("n", [1, 9, 70, 900])
@pytest.mark.parametrize("flags", [0, 1])
def test_small_meshes_intended(gpu_ctx, n, flags):
    """Intended neighbors and kept records of meshes whose rows and record
    runs begin off every 16-byte boundary, with levels of 1, 2, ... 33 and
    more groups (a workgroup writes 32) and roots without children."""
    rng = np.random.default_rng(n + 1)
    meshes = []
    for i in range(n):
        pts = rng.normal(size=(3 + i % 7, 3)).astype(np.float32)
        tri = np.stack([np.arange(k, k + 3) for k in range(len(pts) - 2)]).astype(np.int32)
        meshes.append((pts, tri, int(rng.integers(1, 33))))
    trees, st = gpu_ctx.build_batch(meshes, semantics=1, flags=flags)
    assert not any(st), st
    for (p, t, res), tree in list(zip(meshes, trees))[::max(1, n // 60)]:
        ref = po.build(p, t, res, semantics=1)
        compare(tree, ref, fields=["voxels", "code", "parent", "childs", "neighbors"] if flags
                else None, check_aos=not flags)


def test_intended_records_over_many_blocks(gpu_ctx):
    """More than 1024 blocks of 512 nodes: the block scan carries over."""
    from svo_amd import meshgen
    p, t = meshgen.noisy_icosphere(4, seed=3)
    tree = gpu_ctx.build(p, t, 256, semantics=1)
    assert tree.info.n_nodes > 1024 * 512
    compare(tree, po.build(p, t, 256, semantics=1))
