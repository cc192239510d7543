"""Large read-outs, which pass through a pinned ring in pieces of 512 KiB:
sizes around the least that does (1 MiB), around whole pieces and around the
ring's 8 MiB, to destinations off every alignment, from several threads at
once, against the same bytes read in small parts."""
import ctypes
import threading

import numpy as np
import pytest

import svo_amd
from svo_amd import meshgen

pytestmark = pytest.mark.gpu

FIELDS = ["neighbors", "childs", "vertices", "edges", "nodes_aos", "code"]


@pytest.fixture(scope="module")
def tree(gpu_ctx):
    p, t = meshgen.noisy_icosphere(4, seed=2)
    tree = gpu_ctx.build(p, t, 128)
    yield tree
    tree.free()


def _whole(tree, field, at=0):
    fid = svo_amd.FIELDS[field]
    n = int(svo_amd.lib().svo_tree_field_bytes(tree._h, fid))
    buf = np.full(n + at + 64, 0xAB, np.uint8)
    svo_amd._check(svo_amd.lib().svo_tree_copy_field(tree._h, fid, buf.ctypes.data + at, n), field)
    assert (buf[:at] == 0xAB).all() and (buf[at + n:] == 0xAB).all()
    return buf[at: at + n]


@pytest.mark.parametrize("field", FIELDS)
@pytest.mark.parametrize("at", [0, 1, 4, 31])
def test_alignment_and_parts(tree, field, at):
    got = _whole(tree, field, at)
    assert field == "code" or got.nbytes > 4 << 20
    if field == "nodes_aos":
        assert np.array_equal(got, _whole(tree, field))
        return
    whole = tree.field(field)
    assert np.array_equal(got, whole.reshape(-1).view(np.uint8))
    rows, step = whole.shape[0], 1000
    for start in list(range(0, rows, max(step, rows // 40))) + [max(0, rows - step)]:
        k = min(step, rows - start)  # far below 1 MiB: the plain path
        assert np.array_equal(tree.field_rows(field, start, k), whole[start: start + k])


def test_sizes(gpu_ctx):
    """Device bytes of every size around the limits, by the tree's width array
    of meshes whose node counts differ."""
    rng = np.random.default_rng(0)
    seen = set()
    for n in (1500, 2200, 3000, 6000, 12000):
        p = rng.random((n, 3)).astype(np.float32)
        p = np.repeat(p[:, None], 3, axis=1) + 1e-3 * rng.random((n, 3, 3)).astype(np.float32)
        t = np.arange(3 * n, dtype=np.int32).reshape(-1, 3)
        tree = gpu_ctx.build(p.reshape(-1, 3), t, 256, flags=svo_amd.BUILD_NO_VERTEX_EDGE)
        for field in ("neighbors", "childs", "origin"):
            a = tree.field(field)
            seen.add(a.nbytes >> 18)
            rows = a.shape[0]
            k = max(1, (1 << 20) // (a.nbytes // rows))
            parts = [tree.field_rows(field, s, min(k, rows - s)) for s in range(0, rows, k)]
            assert np.array_equal(a, np.concatenate(parts))
        tree.free()
    print(sorted(seen))


def test_source_alignment(gpu_ctx):
    """A batch's second tree, whose arrays begin off 16 and off 4 bytes."""
    p, t = meshgen.noisy_icosphere(5, seed=1)
    trees, st = gpu_ctx.build_batch([(p, t, 9), (p, t, 512)])
    assert not any(st)
    alone = gpu_ctx.build(p, t, 512)
    assert trees[1].info.n_nodes > 1 << 20
    for field in ("is_leaf", "width", "origin", "childs", "code", "edges"):
        assert np.array_equal(trees[1].field(field).view(np.uint8),
                              alone.field(field).view(np.uint8)), field
    for x in (*trees, alone):
        x.free()


def test_threads(gpu_ctx, tree):
    want = {f: tree.field(f).copy() for f in FIELDS[:4]}
    bad = []

    def read(f):
        for _ in range(8):
            if not np.array_equal(tree.field(f), want[f]):
                bad.append(f)

    th = [threading.Thread(target=read, args=(f,)) for f in FIELDS[:4] for _ in range(2)]
    for x in th:
        x.start()
    for x in th:
        x.join()
    assert not bad


@pytest.mark.parametrize("at", [0, 4])
def test_pinned_destination(tree, at):
    """To pinned memory, which the runtime copies to directly."""
    hip = svo_amd.lib()  # (finds the symbols of the runtime that it has loaded)
    for field in ("neighbors", "nodes_aos"):
        fid = svo_amd.FIELDS[field]
        n = int(svo_amd.lib().svo_tree_field_bytes(tree._h, fid))
        ptr = ctypes.c_void_p()
        assert hip.hipHostMalloc(ctypes.byref(ptr), ctypes.c_size_t(n + 64), 0) == 0
        buf = np.ctypeslib.as_array((ctypes.c_uint8 * (n + 64)).from_address(ptr.value))
        buf[:] = 0xAB
        svo_amd._check(svo_amd.lib().svo_tree_copy_field(tree._h, fid, ptr.value + at, n), field)
        ok = np.array_equal(buf[at: at + n], _whole(tree, field))
        ok = ok and (buf[:at] == 0xAB).all() and (buf[at + n:] == 0xAB).all()
        assert hip.hipHostFree(ptr) == 0
        assert ok, field
