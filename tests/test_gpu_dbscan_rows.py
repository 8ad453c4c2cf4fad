"""chaos_dbscan_rows on device memory: row-major points of the caller are split
into columns on the device, labels stay there."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# sizes around a block of the splitting kernel and the slabs of 2^20 points
@pytest.mark.parametrize("n", [1, 85, 86, 5000, 1048576, 1048577])
@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("masked", [False, True])
def test_rows_in_device_memory_equal_rows_on_the_host(chaos, n, dim, masked):
    rng = np.random.default_rng(n + dim)
    pts = np.ascontiguousarray(rng.integers(0, max(2, int(n ** 0.5)), size=(n, dim)) * 0.4)
    inc = (rng.random(n) < 0.8).astype(np.int32) if masked else None
    print(f"rows on the device n={n} dim={dim} masked={masked}", flush=True)
    want, k = chaos.dbscan(pts, 0.5, 3, include=inc)
    lib, bufs = chaos.lib, []

    def device(a):
        p = C.c_void_p()
        chaos._check(lib.chaos_device_malloc(C.byref(p), C.c_size_t(a.nbytes), 0))
        chaos._check(lib.chaos_memcpy_h2d(p, a.ctypes.data_as(C.c_void_p), C.c_size_t(a.nbytes)))
        bufs.append(p)
        return p

    labels = np.full(n, -7, dtype=np.int32)
    o = chaos.make_options(device_buffers=True)
    clusters = C.c_int(-1)
    d_pts, d_lab = device(pts), device(labels)
    d_inc = device(inc) if masked else None
    as_d, as_i = C.POINTER(C.c_double), C.POINTER(C.c_int)
    chaos._check(lib.chaos_dbscan_rows(C.byref(o), C.cast(d_pts, as_d), n, dim, 0.5, 3, 0,
                                       C.cast(d_inc, as_i) if masked else None, C.cast(d_lab, as_i),
                                       C.byref(clusters)))
    chaos._check(lib.chaos_memcpy_d2h(labels.ctypes.data_as(C.c_void_p), d_lab, C.c_size_t(labels.nbytes)))
    back = np.empty_like(pts)
    chaos._check(lib.chaos_memcpy_d2h(back.ctypes.data_as(C.c_void_p), d_pts, C.c_size_t(back.nbytes)))
    for p in bufs:
        chaos._check(lib.chaos_device_free(p))
    assert clusters.value == k
    assert np.array_equal(labels, want)
    assert np.array_equal(back, pts)
