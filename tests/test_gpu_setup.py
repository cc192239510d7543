"""The set-up kernels of a pass: boxes of point sets whose coordinates end
inside, at and past a workgroup's 3072 dwords, extremes in the last point, and the flags for a coordinate that is
not finite and an index out of range anywhere in the arrays, alone and beside
good meshes of one batch."""
import numpy as np
import pytest

import pyoracle as po
import svo_amd
from parity import compare

pytestmark = pytest.mark.gpu


def _mesh(rng, n_points):
    p = rng.random((n_points, 3)).astype(np.float32)
    p[-1] = [1.5, -0.25, 2.0]
    t = np.arange(n_points - n_points % 3, dtype=np.int32).reshape(-1, 3)
    return p, np.concatenate([t, [[n_points - 1, 0, 1]]]).astype(np.int32)


SIZES = [3, 5, 255, 256, 1023, 1024, 1025, 2049, 5000]


@pytest.mark.parametrize("n", SIZES)
def test_boxes(gpu_ctx, n):
    p, t = _mesh(np.random.default_rng(n), n)
    if n > 300:  # small triangles: the oracle walks every cell of a box
        p[3:-1] = p[0] + 0.02 * p[3:-1]
    tree = gpu_ctx.build(p, t, 24, flags=svo_amd.BUILD_NO_VERTEX_EDGE)
    compare(tree, po.build(p, t, 24), fields=["voxels", "origin", "width", "level_nodes"],
            check_aos=False)


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("what", ["nan", "inf", "negative", "past"])
def test_flags(gpu_ctx, n, what):
    """The bad mesh is refused, its neighbors in the batch are built."""
    rng = np.random.default_rng(n)
    meshes = []
    for at in (0, n // 2, n - 1):
        good = _mesh(rng, 5)
        p, t = _mesh(rng, n)
        if what in ("nan", "inf"):
            p[at, at % 3] = np.nan if what == "nan" else -np.inf
        else:
            t.reshape(-1)[at] = -1 if what == "negative" else n
        meshes += [(*good, 8), (p, t, 8)]
    trees, st = gpu_ctx.build_batch(meshes)
    assert [bool(s) for s in st] == [False, True] * 3
    for (p, t, res), tree in list(zip(meshes, trees))[::2]:
        compare(tree, po.build(p, t, res))
