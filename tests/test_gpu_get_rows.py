"""Embedding rows of a chunk in one launch: every row the host's own conversion of it, in the list's order."""
import ctypes as C

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

F32, F16, BF16 = 0, 1, 30


def host_row(wtype, raw, n):
    if wtype == F32:
        return raw.view(np.float32)
    if wtype == F16:
        return raw.view(np.float16).astype(np.float32)
    if wtype == BF16:
        return (raw.view(np.uint16).astype(np.uint32) << 16).view(np.float32)
    return oracle.dequant_row(wtype, raw, n)


@pytest.mark.parametrize("wtype,n", [(F32, 300), (F16, 300), (BF16, 258), (oracle.TYPE_Q4K, 256), (oracle.TYPE_Q6K, 768)])
@pytest.mark.parametrize("n_rows", [1, 2, 63, 64])
def test_rows(wtype, n, n_rows):
    from kore_amd import hip, qmv
    rng = np.random.default_rng(n_rows)
    row_bytes = {F32: 4 * n, F16: 2 * n, BF16: 2 * n}.get(wtype) or n // 256 * oracle.BLOCK_BYTES[wtype]
    table = rng.integers(0, 120, 70 * row_bytes, dtype=np.uint8)      # finite floats and f16 scales
    rows = rng.integers(0, 70, n_rows).astype(np.int64)
    dt = hip.DeviceBuffer((table.size + 3) // 4)
    hip.check(hip.lib().hipMemcpy(dt.ptr, table.ctypes.data, table.size, hip.H2D), "H2D")
    out = hip.DeviceBuffer(n_rows * n)
    get = qmv.lib().kore_qmv_get_rows_dev
    get.argtypes = [C.c_int, C.c_void_p, C.c_void_p, C.c_int, C.c_int64, C.c_void_p, C.c_void_p]
    assert get(wtype, dt.ptr, rows.ctypes.data, n_rows, n, out.ptr, None) == 0
    hip.synchronize()
    got = out.download().reshape(n_rows, n).view(np.uint32)
    for z, r in enumerate(rows):
        ref = host_row(wtype, table[r * row_bytes:(r + 1) * row_bytes].copy(), n)
        assert np.array_equal(got[z], ref.view(np.uint32)), z
    bad = np.array([0, -1], np.int64)
    assert get(wtype, dt.ptr, bad.ctypes.data, 2, n, out.ptr, None) != 0
    assert get(wtype, dt.ptr, rows.ctypes.data, 65, n, out.ptr, None) != 0
    for b in (dt, out):
        b.free()
