"""Which builds read a bitmap by its flagged lines (the stage `line_flags` says
so), and a plan that does: one mesh on a grid whose bitmap is just the 256 MB
from which it is so, replayed as it was, over a mesh of other sizes, whose
replay must fall back, and over the first mesh again."""
import ctypes as C
import os
import sys

import numpy as np
import pytest

import pyoracle as po
import svo_amd
from parity import compare
from test_gpu_lines import FIELDS, _mesh

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402

pytestmark = pytest.mark.gpu

LEAST = (2048, 1024, 1024)  # 2^31 codes: 256 MB


def _takes_lines(ctx, meshes, path=1):
    ctx.set_timing(True)
    ctx.set_option("dedup_path", path)
    try:
        trees, st = ctx.build_batch(meshes, flags=svo_amd.BUILD_NO_VERTEX_EDGE)
        assert not any(st)
        return "line_flags" in ctx.stage_ms()
    finally:
        ctx.set_option("dedup_path", 0)
        ctx.set_timing(False)
        for t in trees:
            t.free()


@pytest.mark.parametrize("shape", ["scattered", "one", "block"])
@pytest.mark.parametrize("res", [(1500, 1500, 1500), (2048, 2048, 2048), (1100, 300, 2000), LEAST])
def test_large_bitmaps_take_them(gpu_ctx, shape, res):
    """Where the flags, a byte a line, have room in level 1's keys: 8 bytes for
    each candidate cell."""
    p, t = _mesh(np.random.default_rng(3), shape, res)
    took = _takes_lines(gpu_ctx, [(p, t, res)])
    stats = bench.pass_stats(gpu_ctx)
    print(shape, res, took, stats, flush=True)
    assert stats["bitmap_bytes"] >= 256 << 20 and stats["key_bytes"] == 8
    assert took == (stats["bitmap_bytes"] // 64 <= 8 * stats["box_cells"])
    assert took or res == (1100, 300, 2000) or res == LEAST
    assert not _takes_lines(gpu_ctx, [(p, t, res)], path=2)


@pytest.mark.parametrize("res", [(1100, 300, 2000), LEAST, (3000, 500, 700)])
def test_uneven_grids(gpu_ctx, res):
    """Uneven grids with enough triangles to take them, every field."""
    rng = np.random.default_rng(5)
    p = rng.random((2000, 1, 3)) * res + 40 * rng.normal(size=(2000, 3, 3))
    p = np.clip(p, 0, res).reshape(-1, 3).astype(np.float32)
    t = np.arange(len(p), dtype=np.int32).reshape(-1, 3)
    assert _takes_lines(gpu_ctx, [(p, t, res)])
    want = po.build(p, t, res, key_bits=64)
    for path in (1, 1, 2):
        gpu_ctx.set_option("dedup_path", path)
        try:
            tree = gpu_ctx.build(p, t, res, flags=svo_amd.BUILD_NO_VERTEX_EDGE)
        finally:
            gpu_ctx.set_option("dedup_path", 0)
        compare(tree, want, fields=FIELDS, check_aos=False)
        tree.free()


def test_others_do_not(gpu_ctx):
    p, t = _mesh(np.random.default_rng(3), "scattered", LEAST)
    assert not _takes_lines(gpu_ctx, [(p, t, (1024, 1024, 1024))])  # 128 MB
    assert not _takes_lines(gpu_ctx, [(p, t, LEAST), (p, t, 64)])   # two meshes



def test_plan(gpu_ctx):
    p, t = _mesh(np.random.default_rng(4), "scattered", LEAST)
    want = po.build(p, t, LEAST, key_bits=64)
    # the same triangles, flat: other voxels and nodes in the same box
    q = p.copy()
    q[:-6, 2] *= np.float32(0.1)
    other = po.build(q, t, LEAST, key_bits=64)
    assert other.info.n_nodes != want.info.n_nodes
    mesh = gpu_ctx.upload_mesh(p, t)

    def upload(pts):
        svo_amd._check(svo_amd.lib().svo_device_copy(
            gpu_ctx.handle, C.c_void_p(mesh.points_ptr), pts.ctypes.data, pts.nbytes, 0), "upload")

    plan = gpu_ctx.plan([mesh.desc(LEAST)], on_device=True, flags=svo_amd.BUILD_NO_VERTEX_EDGE)
    try:
        for pts, ref, same in ((p, want, True), (p, want, True), (q, other, False), (p, want, True),
                               (q, other, False), (p, want, True)):
            upload(np.ascontiguousarray(pts))
            trees, st, replayed = plan.run()
            print(f"replayed {replayed}", flush=True)
            assert st == [0] and replayed == same
            compare(trees[0], ref, fields=FIELDS, check_aos=False)
            trees[0].free()
            # the program's own work between replays
            gpu_ctx.build(p, t, 64, flags=svo_amd.BUILD_NO_VERTEX_EDGE).free()
    finally:
        plan.close()
        mesh.free()
