"""Lookups and read-outs from a thread whose last HIP call failed: the error of
that call is not theirs."""
import ctypes

import numpy as np
import pytest

import svo_amd
from svo_amd import meshgen

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tree(gpu_ctx):
    p, t = meshgen.noisy_icosphere(4, seed=2)
    tree = gpu_ctx.build(p, t, 128)
    yield tree
    tree.free()


@pytest.fixture
def stale():
    """Leaves an error behind as a program's own call would."""
    hip = svo_amd.lib()  # (finds the symbols of the runtime that it has loaded)

    def fail():
        assert hip.hipSetDevice(ctypes.c_int(9999)) != 0
        assert hip.hipPeekAtLastError() != 0
    yield fail
    hip.hipGetLastError()


@pytest.mark.parametrize("n", [1, 1000, 1 << 17])
def test_lookups(tree, stale, n):
    nb = tree.field("neighbors").reshape(-1, 27)
    rng = np.random.default_rng(n)
    node = rng.integers(0, nb.shape[0], n).astype(np.uint32)
    slot = rng.integers(0, 27, n).astype(np.uint8)
    stale()
    assert np.array_equal(tree.query_neighbors(node, slot), nb[node, slot])


@pytest.mark.parametrize("field", ["neighbors", "nodes_aos", "level_nodes"])
def test_read_out(tree, stale, field):
    want = tree.field(field).copy()
    stale()
    assert np.array_equal(tree.field(field).view(np.uint8), want.view(np.uint8))
