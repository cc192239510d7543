"""Raw voxelization hits, triangle by triangle: the GPU's codes of a mesh, as a
multiset, are the sum of the oracle's sets of its triangles one at a time (a
triangle hits a cell at most once; the grid stays, as all points stay).  So a
cell missed, added or emitted twice for one triangle shows also where other
triangles cover it.  The same sum is the hit count of a build, for each
de-duplication path and size limit.  The triangles are those of
test_gpu_vox_rows."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

import pyoracle as po
import svo_amd
from test_gpu_vox_rows import CASES, _family

pytestmark = pytest.mark.gpu


def _per_triangle(pts, tri, res, kb):
    with ThreadPoolExecutor(8) as ex:
        sets = list(ex.map(lambda t: po.voxelize(pts, t[None], res, key_bits=kb, threads=1)[1],
                           tri))
    return np.sort(np.concatenate(sets))


@pytest.mark.parametrize("name,scale,offset", CASES)
@pytest.mark.parametrize("res,kb", [((64, 64, 64), 32), ((101, 33, 250), 32),
                                    ((300, 1100, 200), 64)])
def test_hits_are_the_triangles_sum(name, scale, offset, res, kb):
    pts = ((_family(name, np.random.default_rng(8)) + offset) * scale).astype(np.float32)
    tri = np.arange(len(pts), dtype=np.int32).reshape(-1, 3)
    if max(res) > 512:
        tri = tri[:200]
    want = _per_triangle(pts, tri, res, kb)
    got, n = svo_amd.k_voxelize(pts, tri, res, key_bits=kb)
    print(f"{name} scale {scale} offset {offset} res {res}: {n} hits, {len(np.unique(want))} cells",
          flush=True)
    assert n == len(want) == len(got)
    assert np.array_equal(np.sort(got.astype(np.uint64)), want)


@pytest.mark.parametrize("limit", [1, 1024, 1 << 20])
@pytest.mark.parametrize("n", [1, 5, 33, 600])
def test_hit_count_of_builds(gpu_ctx, limit, n):
    pts = _family("sizes", np.random.default_rng(n))[: 3 * n].astype(np.float32)
    tri = np.arange(3 * n, dtype=np.int32).reshape(-1, 3)
    want = len(_per_triangle(pts, tri, (90, 90, 90), 32))
    for path in (1, 2):
        gpu_ctx.set_option("small_max_cells", limit)
        gpu_ctx.set_option("dedup_path", path)
        try:
            tree = gpu_ctx.build(pts, tri, 90, flags=svo_amd.BUILD_NO_VERTEX_EDGE)
        finally:
            gpu_ctx.set_option("small_max_cells", 1024)
            gpu_ctx.set_option("dedup_path", 0)
        assert tree.info.n_hits == want, path
        tree.free()
