"""The stable sort of rows by key that lays like frames side by side
(filter_kernels.hip), against numpy's.

The order decides only which rows share a tile, so no query's outputs show a
mistake in it; the library's C++ launcher is called by its symbol."""
import ctypes

import numpy as np
import pytest

from devmem import DevBuf
from mdsctk_amd import knn

SORT = "_ZN6mdsctk17launch_sort_orderEPKiPiiPjS3_S1_S2_lPvmP12ihipStream_t"
SCRATCH = "_ZN6mdsctk18sort_order_scratchEl"


def _sorted_rows(keys):
    lib = knn.load()
    scratch = lib[SCRATCH]
    scratch.restype, scratch.argtypes = ctypes.c_size_t, [ctypes.c_int64]
    sort = lib[SORT]
    vp, i64 = ctypes.c_void_p, ctypes.c_int64
    sort.restype = ctypes.c_int
    sort.argtypes = [vp, vp, ctypes.c_int, vp, vp, vp, vp, i64, vp, ctypes.c_size_t, vp]
    n = len(keys)
    need = scratch(n)
    d_keys, d_rows = DevBuf.upload(keys), DevBuf.upload(np.arange(n, dtype=np.int32))
    d_out, d_order, d_temp = DevBuf(4 * n), DevBuf(4 * n), DevBuf(need)
    assert sort(None, None, 0, d_keys.ptr, d_out.ptr, d_rows.ptr, d_order.ptr, n, d_temp.ptr, need,
                None) == 0
    return d_order.download((n,), np.int32), d_keys.download((n,), np.uint32)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 65, 1024, 1025, 40007, 262144, 262145, 600001])
@pytest.mark.parametrize("kind", ["any", "few", "one"])
def test_sort_order_is_numpys_stable_sort(n, kind):
    """Less than a wave's round, either side of a workgroup and of the size from
    which a workgroup takes more rounds; 32-bit keys, few different ones, one."""
    rng = np.random.default_rng(n)
    keys = rng.integers(0, {"any": 2**32, "few": 300, "one": 1}[kind], n, dtype=np.uint32)
    order, after = _sorted_rows(keys)
    np.testing.assert_array_equal(order, np.argsort(keys, kind="stable").astype(np.int32))
    np.testing.assert_array_equal(after, keys)
