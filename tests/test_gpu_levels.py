"""The passes above the first level at the edges of their tiles: levels of a
tile of 1024 or 4096 elements, one less and one more, at the point where the
one-workgroup tail takes over and where the tile size changes, groups that go
on over a thread's and a tile's end, and the same for several meshes in one
batch.  Every field equals the oracle's."""
import numpy as np
import pytest

import pyoracle as po
import svo_amd
from parity import compare

pytestmark = pytest.mark.gpu

FIELDS = ["voxels", "code", "is_leaf", "origin", "width", "parent", "childs", "neighbors",
          "level_nodes"]


def _cells(rng, n, side, shape):
    """n tiny triangles, one to a group of the first level (a cell of 2 x 2 x 2),
    in a grid of 2 * side cells: `dense` fills the groups in Morton order, so
    that the next level's groups have eight members each; `loose` draws them."""
    if shape == "dense":
        k = np.arange(n, dtype=np.int64)
    else:
        k = np.sort(rng.choice(side ** 3, n, replace=False))
        k[0], k[-1] = 0, side ** 3 - 1
    xyz = np.zeros((n, 3), np.int64)
    for b in range(10):
        for d in range(3):
            xyz[:, d] |= ((k >> (3 * b + d)) & 1) << b
    c = (2 * xyz + 0.5).astype(np.float32)
    p = np.repeat(c[:, None], 3, axis=1)
    p[:, 1, 0] += 0.25
    p[:, 2, 1] += 0.25
    corner = np.array([[[0, 0, 0]] * 3, [[2 * side] * 3] * 3], np.float32)
    p = np.concatenate([p, corner])  # the box is the grid: cells of size 1
    return p.reshape(-1, 3), np.arange(3 * (n + 2), dtype=np.int32).reshape(-1, 3)


@pytest.mark.parametrize("path", [1, 2])
@pytest.mark.parametrize("shape", ["dense", "loose"])
@pytest.mark.parametrize("n", [1, 7, 8, 9, 1020, 1023, 1024, 1025, 4092, 4095, 4096, 4097, 20000])
def test_level_edges(gpu_ctx, n, shape, path):
    p, t = _cells(np.random.default_rng(n), n, 32 if n > 1 else 2, shape)
    res = 64 if n > 1 else 4
    gpu_ctx.set_option("dedup_path", path)
    try:
        trees, st = gpu_ctx.build_batch([(p, t, res), (p[: 3 * max(n // 2, 1)], t[: max(n // 2, 1)], res),
                                         (p, t, res)], flags=svo_amd.BUILD_NO_VERTEX_EDGE)
    finally:
        gpu_ctx.set_option("dedup_path", 0)
    assert not any(st), st
    want = po.build(p, t, res)
    for tree in (trees[0], trees[2]):
        compare(tree, want, fields=FIELDS, check_aos=False)
    m = max(n // 2, 1)
    compare(trees[1], po.build(p[: 3 * m], t[:m], res), fields=FIELDS, check_aos=False)


def _links(v):
    """Codes, parents and children of the tree over the sorted voxel codes."""
    none = 0xFFFFFFFF
    lv, e = [], v.astype(np.int64)
    while len(e) > 1:
        e = np.unique(e >> 3)
        lv.append((e[:, None] * 8 + np.arange(8)).ravel())
    lv.append(e)
    base = np.concatenate([[0], np.cumsum([len(x) for x in lv])])
    parent = np.full(base[-1], none, np.int64)
    childs = np.full((base[-1], 8), none, np.int64)
    for i in range(len(lv) - 1):
        j = base[i + 1] + np.searchsorted(lv[i + 1], lv[i][::8] >> 3)
        parent[base[i]:base[i + 1]] = np.repeat(j, 8)
        childs[j] = base[i] + np.arange(len(lv[i])).reshape(-1, 8)
    return np.concatenate(lv), parent, childs


@pytest.mark.parametrize("path", [1, 2])
@pytest.mark.parametrize("n", [1 << 20, (1 << 20) + 1])
def test_tile_size_changes(gpu_ctx, n, path):
    """A level 2 of 2^20 elements and of one more."""
    p, t = _cells(np.random.default_rng(1), n, 128, "loose")
    gpu_ctx.set_option("dedup_path", path)
    try:
        tree = gpu_ctx.build(p, t, 256, flags=svo_amd.BUILD_NO_VERTEX_EDGE)
    finally:
        gpu_ctx.set_option("dedup_path", 0)
    v = tree.field("voxels")
    assert len(np.unique(v >> 3)) == n
    code, parent, childs = _links(v)
    assert np.array_equal(tree.field("code"), code)
    assert np.array_equal(tree.field("parent"), parent)
    assert np.array_equal(tree.field("childs").reshape(-1, 8), childs)


def test_tile_sums(gpu_ctx):
    """Bitmaps of 2048 tiles, whose emission adds the tile counts up itself, and
    of one tile more, which a scan of their own adds up; each mesh's span ends
    at the next mesh's first tile, a single voxel's as well."""
    from svo_amd import meshgen
    p, t = meshgen.icosphere(3)
    big, small = (p, t, 512), (p, t, 9)
    one = (p[:3], np.array([[0, 1, 2]], np.int32), 1)
    want = {id(m): po.build(*m) for m in (big, small, one)}
    for batch in ([big], [big, one], [small, big], [one, small, one, one, small]):
        trees, st = gpu_ctx.build_batch(batch)
        assert not any(st)
        for m, tree in zip(batch, trees):
            compare(tree, want[id(m)], fields=FIELDS, check_aos=False)
            tree.free()
