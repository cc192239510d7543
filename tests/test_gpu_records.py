"""Reference-semantics vertex and edge records on the GPU at the sizes where
the record kernel's pieces meet: a workgroup holds 512 16-byte pieces, 21 edge
pieces or 8 vertex pieces per node, so nodes are cut across workgroups at 24.4
(edges) and 64 (vertices) nodes.  Expected values are the reference's formulas
(SVO.cu:567-584, 638-663) in float32, bit for bit: the zero offset keeps the
bare origin (a negative zero stays one), every other corner adds 0 or the
width."""
import numpy as np
import pytest

import svo_amd

pytestmark = pytest.mark.gpu

EDGES = [((0, 0, 0), (0, 1, 0)), ((0, 1, 0), (1, 1, 0)), ((1, 1, 0), (1, 0, 0)),
         ((1, 0, 0), (0, 0, 0)), ((0, 0, 1), (0, 1, 1)), ((0, 1, 1), (1, 1, 1)),
         ((1, 1, 1), (1, 0, 1)), ((1, 0, 1), (0, 0, 1)), ((0, 0, 0), (0, 0, 1)),
         ((0, 1, 0), (0, 1, 1)), ((1, 1, 0), (1, 1, 1)), ((1, 0, 0), (1, 0, 1))]


@pytest.mark.parametrize("n", [1, 2, 24, 25, 26, 63, 64, 65, 511, 512, 513, 12288, 100_003])
def test_reference_records(n):
    rng = np.random.default_rng(n)
    o = rng.normal(size=(n, 3)).astype(np.float32)
    o[rng.random((n, 3)) < 0.2] = np.float32(-0.0)
    w = (rng.random(n) + 0.01).astype(np.float32)
    verts, edges = svo_amd.k_ref_vertex_edge(o, w)
    owner = np.arange(n, dtype=np.uint32)
    assert np.array_equal(verts["owner"], np.repeat(owner, 8))
    assert np.array_equal(edges["owner"], np.repeat(owner, 12))
    v = verts["p"].reshape(n, 8, 3)
    for j in range(8):
        bits = np.array([j & 1, j >> 1 & 1, j >> 2 & 1], np.float32)
        assert np.array_equal(v[:, j].view(np.uint32), (w[:, None] * bits).view(np.uint32))
    for i, ends in enumerate(EDGES):
        for name, end in zip("ab", ends):
            add = np.where(np.array(end, bool)[None, :], w[:, None], np.float32(0.0))
            want = o if end == (0, 0, 0) else o + add
            got = edges[name].reshape(n, 12, 3)[:, i]
            assert np.array_equal(np.ascontiguousarray(got).view(np.uint32),
                                  np.ascontiguousarray(want, np.float32).view(np.uint32)), (i, name)
