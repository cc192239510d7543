"""Level 1 from the flagged lines of a large bitmap (one mesh, 256 MB and
more): scattered triangles, which leave most lines empty, triangles packed
into a few lines and tiles that are full, and flags in the first and the last
line.  Every field equals the oracle's and the sort path's, also on a second
build, which finds the bitmap as the first one left it."""
import numpy as np
import pytest

import pyoracle as po
import svo_amd
from parity import compare

pytestmark = pytest.mark.gpu

FIELDS = ["voxels", "code", "is_leaf", "origin", "width", "parent", "childs", "level_nodes"]


def _mesh(rng, shape, res):
    h = max(res)
    corner = np.array([[[0, 0, 0]] * 3, [res] * 3], np.float64)  # first and last cell
    if shape == "scattered":  # about 30 cells an axis, flat: most cells missed
        p = rng.random((160, 1, 3)) * res + 15 * rng.normal(size=(160, 3, 3))
    elif shape == "one":  # a triangle across the grid
        p = np.array([[[0, 0, 0], [h, 0.3 * h, 0], [0, 0.2 * h, 0.7 * h]]])
    else:  # a block of 64^3 cells, nearly every one of them hit
        z = (np.arange(192) + 0.5) / 3
        a = np.stack([np.zeros(192), np.zeros(192), z], 1)
        u, v = np.array([128.0, 0, 0]), np.array([0, 128.0, 0])
        p = np.stack([a, a + u, a + v], 1) + np.array([8.0, 16.0, 32.0])
    p = np.clip(p, 0, res)
    p = np.concatenate([p, corner + 0.1 * rng.random((2, 3, 3)) * np.array([1, -1])[:, None, None]])
    return (p.reshape(-1, 3).astype(np.float32), np.arange(3 * len(p), dtype=np.int32).reshape(-1, 3))


@pytest.mark.parametrize("shape", ["scattered", "one", "block"])
@pytest.mark.parametrize("res", [(1500, 1500, 1500), (2048, 2048, 2048), (1100, 300, 2000)])
def test_lines(gpu_ctx, shape, res):
    p, t = _mesh(np.random.default_rng(3), shape, res)
    want = po.build(p, t, res, key_bits=64)
    for path in (1, 1, 2):
        gpu_ctx.set_option("dedup_path", path)
        try:
            tree = gpu_ctx.build(p, t, res, flags=svo_amd.BUILD_NO_VERTEX_EDGE)
        finally:
            gpu_ctx.set_option("dedup_path", 0)
        print(shape, res, path, tree.info.n_voxels, flush=True)
        compare(tree, want, fields=FIELDS, check_aos=False)
        tree.free()
