"""Neighbor lookups through the pinned ring: counts around a wavefront, a
workgroup, all 32 of them and their four at a time, the largest count that
takes the ring and one more, nodes and slots out of range, from threads at once
and between read-outs that use the same ring."""
import threading

import numpy as np
import pytest

import svo_amd
from svo_amd import meshgen

pytestmark = pytest.mark.gpu

FITS = 1 << 17


@pytest.fixture(scope="module")
def table(gpu_ctx):
    p, t = meshgen.noisy_icosphere(4, seed=2)
    trees, st = gpu_ctx.build_batch([(p, t, 7), (p, t, 96)], semantics=svo_amd.SEM_INTENDED)
    assert not any(st)
    yield trees[1], trees[1].field("neighbors").reshape(-1, 27)
    for t in trees:
        t.free()


def _ask(table, n, seed):
    tree, nb = table
    rng = np.random.default_rng(seed)
    node = rng.integers(0, nb.shape[0], n).astype(np.uint32)
    slot = rng.integers(0, 27, n).astype(np.uint8)
    want = nb[node, slot].copy()
    for k, bad in enumerate((nb.shape[0], 0xFFFFFFFF)):  # out of range: none
        node[k::97], want[k::97] = bad, 0xFFFFFFFF
    slot[5::89], want[5::89] = 27, 0xFFFFFFFF
    slot[6::89], want[6::89] = 255, 0xFFFFFFFF
    assert np.array_equal(tree.query_neighbors(node, slot), want), n


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1023, 1025, 32767, 32768, 32769, 100000,
                               FITS - 1, FITS, FITS + 1])
def test_counts(table, n):
    _ask(table, n, n)


def test_threads(table):
    bad = []

    def run(k):
        try:
            for i in range(20):
                _ask(table, 1000 * k + i + 1, i)
                if k % 2:
                    assert np.array_equal(table[0].field("neighbors").reshape(-1, 27), table[1])
        except AssertionError as e:
            bad.append(e)

    th = [threading.Thread(target=run, args=(k,)) for k in range(6)]
    for x in th:
        x.start()
    for x in th:
        x.join()
    assert not bad
