"""Embedding rows of a chunk in one launch: equal to the rows read one at a time, in the list's order."""
import ctypes as C

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wtype,n", [(0, 300), (oracle.TYPE_Q4K, 256), (oracle.TYPE_Q6K, 768)])
@pytest.mark.parametrize("n_rows", [1, 2, 63, 64])
def test_rows(wtype, n, n_rows):
    from kore_amd import hip, qmv
    rng = np.random.default_rng(n_rows)
    row_bytes = 4 * n if wtype == 0 else n // 256 * oracle.BLOCK_BYTES[wtype]
    table = rng.integers(0, 120, 70 * row_bytes, dtype=np.uint8)      # finite floats and f16 scales
    rows = rng.integers(0, 70, n_rows).astype(np.int64)
    dt = hip.DeviceBuffer((table.size + 3) // 4)
    hip.check(hip.lib().hipMemcpy(dt.ptr, table.ctypes.data, table.size, hip.H2D), "H2D")
    out, one = hip.DeviceBuffer(n_rows * n), hip.DeviceBuffer(n)
    L = qmv.lib()
    get = L.kore_qmv_get_rows_dev
    get.argtypes = [C.c_int, C.c_void_p, C.c_void_p, C.c_int, C.c_int64, C.c_void_p, C.c_void_p]
    assert get(wtype, dt.ptr, rows.ctypes.data, n_rows, n, out.ptr, None) == 0
    hip.synchronize()
    got = out.download().reshape(n_rows, n).view(np.uint32)
    for z in sorted({0, n_rows // 2, n_rows - 1}):
        assert L.kore_qmv_get_row_dev(wtype, dt.ptr, int(rows[z]), n, one.ptr, None) == 0
        hip.synchronize()
        assert np.array_equal(got[z], one.download().view(np.uint32)), z
    bad = np.array([0, -1], np.int64)
    assert get(wtype, dt.ptr, bad.ctypes.data, 2, n, out.ptr, None) != 0
    assert get(wtype, dt.ptr, rows.ctypes.data, 65, n, out.ptr, None) != 0
    for b in (dt, out, one):
        b.free()
