"""Row-interval voxelization against the oracle's cell-by-cell tests: the raw
hits (duplicates counted) of triangles whose rows, intervals and rounding the
interval arithmetic has to get right.  Families: triangles of every size from
below a cell to the whole grid (also past the size limit, in queued items of
512 rows), slivers, triangles in and parallel to the grid's planes (slope zero
in one or more tests), vertices on cell boundaries, boxes far from the origin,
and coordinates so small or large that the tests' products leave the range in
which intervals hold."""
import numpy as np
import pytest

import pyoracle as po
import svo_amd

pytestmark = pytest.mark.gpu


def _soup(rng, n, size):
    c = rng.random((n, 1, 3))
    return (c + size * rng.normal(size=(n, 3, 3))).reshape(-1, 3)


def _family(name, rng):
    n = 600
    if name == "sizes":
        return _soup(rng, n, np.repeat(10.0 ** rng.uniform(-4, 0, (n, 1, 1)), 3, axis=1))
    if name == "slivers":
        p = _soup(rng, n, 0.1).reshape(n, 3, 3)
        p[:, 2] = p[:, 0] + (p[:, 1] - p[:, 0]) * rng.random((n, 1)) + 1e-7 * rng.normal(size=(n, 3))
        return p.reshape(-1, 3)
    if name == "axis":  # one axis constant, or two corners sharing coordinates
        p = _soup(rng, n, 0.1).reshape(n, 3, 3)
        k = rng.integers(0, 3, n)
        for i in range(n):
            p[i, :, k[i]] = p[i, 0, k[i]]
            if i % 3 == 0:
                p[i, 1, (k[i] + 1) % 3] = p[i, 0, (k[i] + 1) % 3]
        return p.reshape(-1, 3)
    if name == "lattice":  # corners on a coarse lattice: many ties with cell boundaries
        return np.round(_soup(rng, n, 0.15) * 16) / 16
    if name == "degenerate":
        p = _soup(rng, n, 0.1).reshape(n, 3, 3)
        p[: n // 2, 1] = p[: n // 2, 0]
        p[: n // 4, 2] = p[: n // 4, 0]
        return p.reshape(-1, 3)
    raise ValueError(name)


CASES = [("sizes", 1.0, 0.0), ("slivers", 1.0, 0.0), ("axis", 1.0, 0.0), ("lattice", 1.0, 0.0),
         ("degenerate", 1.0, 0.0), ("sizes", 1.0, 300.0), ("sizes", 1e-14, 0.0),
         ("sizes", 1e-18, 0.0), ("axis", 1e-20, 0.0), ("sizes", 1e9, 0.0), ("sizes", 1e15, 0.0),
         ("slivers", 1e18, 0.0)]


@pytest.mark.parametrize("name,scale,offset", CASES)
@pytest.mark.parametrize("res,kb", [((64, 64, 64), 32), ((101, 33, 250), 32), ((700, 1100, 900), 64)])
def test_hits_equal_oracle(name, scale, offset, res, kb):
    rng = np.random.default_rng(7)
    pts = ((_family(name, rng) + offset) * scale).astype(np.float32)
    tri = np.arange(len(pts), dtype=np.int32).reshape(-1, 3)
    if max(res) > 512:
        tri = tri[:200]
    st, want = po.voxelize(pts, tri, res, key_bits=kb)
    assert st == 0
    got, n = svo_amd.k_voxelize(pts, tri, res, key_bits=kb)
    print(f"{name} scale {scale} offset {offset} res {res}: {n} hits", flush=True)
    assert np.array_equal(np.unique(got.astype(np.uint64)), np.unique(want.astype(np.uint64)))


@pytest.mark.parametrize("limit", [1, 40, 1024, 1 << 20])
@pytest.mark.parametrize("path", [1, 2])
@pytest.mark.parametrize("n", [1, 3, 4, 5, 31, 32, 33, 127, 600])
def test_split_does_not_change_hits(gpu_ctx, limit, path, n):
    """The runs of triangles per wave, the size limit and the output path change
    neither the voxels nor the number of raw hits."""
    rng = np.random.default_rng(n)
    pts = _family("sizes", rng)[: 3 * n].astype(np.float32)
    tri = np.arange(3 * n, dtype=np.int32).reshape(-1, 3)
    st, want = po.voxelize(pts, tri, 90)
    assert st == 0
    gpu_ctx.set_option("small_max_cells", limit)
    gpu_ctx.set_option("dedup_path", path)
    try:
        tree = gpu_ctx.build(pts, tri, 90, flags=svo_amd.BUILD_NO_VERTEX_EDGE)
    finally:
        gpu_ctx.set_option("small_max_cells", 1024)
        gpu_ctx.set_option("dedup_path", 0)
    assert np.array_equal(tree.field("voxels"), np.unique(want).astype(np.uint32))
    _, hits = svo_amd.k_voxelize(pts, tri, 90)
    assert tree.info.n_hits == hits
