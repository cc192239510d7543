"""The radix sort where its tile size changes (1024, 2048 and 4096 keys: below
2^18, below 2^21 and from there on) and at the tiles' ends, with passes of odd
and even number and a last digit of every width, in scratch memory and in
place in the caller's, whose keys stand at any alignment of their type."""
import ctypes as C

import numpy as np
import pytest

import svo_amd

pytestmark = pytest.mark.gpu

SIZES = [2, 1023, 1024, 1025, 2047, 2049, (1 << 18) - 1, 1 << 18, (1 << 18) + 1, (1 << 21) - 1,
         1 << 21, (1 << 21) + 1]


def _want(keys, bits):
    if bits == 8 * keys.dtype.itemsize:
        return np.sort(keys)
    return keys[np.argsort(keys & keys.dtype.type((1 << bits) - 1), kind="stable")]


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("dtype,bits", [(np.uint32, 9), (np.uint32, 17), (np.uint32, 32),
                                        (np.uint64, 36), (np.uint64, 63)])
@pytest.mark.parametrize("offset", [0, 1, 3])
def test_sizes(gpu_ctx, n, dtype, bits, offset):
    rng = np.random.default_rng(n + bits)
    keys = rng.integers(0, np.iinfo(dtype).max, n, dtype=dtype, endpoint=True)
    keys[n // 3: n // 2] = keys[n // 3]  # a run of equal keys
    want = _want(keys, bits)
    print(f"n {n} {np.dtype(dtype).name} bits {bits} offset {offset}", flush=True)
    if offset == 0:
        assert np.array_equal(svo_amd.k_radix_sort(keys, bits), want)
    lib, size = svo_amd.lib(), keys.dtype.itemsize
    p, total = C.c_void_p(), size * (n + offset + 4)
    svo_amd._check(lib.svo_device_alloc(gpu_ctx.handle, total, C.byref(p)), "device alloc")
    try:
        guard = np.full(n + offset + 4, 7, dtype)
        guard[offset: offset + n] = keys
        svo_amd._check(lib.svo_device_copy(gpu_ctx.handle, p, guard.ctypes.data, total, 0), "up")
        svo_amd._check(lib.svo_k_radix_sort_noalloc(0, C.c_void_p(p.value + size * offset), n, size,
                                                    bits, None), "sort")
        svo_amd._check(lib.svo_device_copy(gpu_ctx.handle, guard.ctypes.data, p, total, 1), "down")
    finally:
        lib.svo_device_free(gpu_ctx.handle, p, total)
    assert np.array_equal(guard[offset: offset + n], want)
    assert (guard[:offset] == 7).all() and (guard[offset + n:] == 7).all()
