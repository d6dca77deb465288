"""Batched attention where magnitudes differ widely, against attention in float64, every (row, head) by its own
norm: what a row does not attend, or attends with next to no weight, must not cost it precision, and zeros are
ordinary values.

Bound: ordinary rows of these sizes measure 1e-7 to 4e-7 of their 2-norm (fp32 sums); where a score may be off by
2^-21 its weight is off by 3.3e-7 more.  1e-6 holds both.
"""
import numpy as np
import pytest

from tests.test_gpu_prefill_split import inputs, reference, run

pytestmark = pytest.mark.gpu

GEOMETRIES = [(4, 2, 64), (6, 2, 96), (7, 1, 128), (2, 1, 200)]


def check(q, k, v, pos0, nh, nkv, hd, rows=slice(None), tol=1e-6):
    out, ref = run(q, k, v, pos0, nh, nkv, hd)[rows], reference(q, k, v, pos0, nh, nkv, hd)[rows]
    err = np.linalg.norm(out - ref, axis=-1) / np.maximum(np.linalg.norm(ref, axis=-1), 1e-300)
    assert np.all(np.isfinite(out)), "rows %s" % np.argwhere(~np.isfinite(out).all(-1))[:4].tolist()
    assert err.max() <= tol, "%.2e at %s" % (err.max(), np.unravel_index(err.argmax(), err.shape))


@pytest.mark.parametrize("nh,nkv,hd", GEOMETRIES)
@pytest.mark.parametrize("n,pos0", [(20, 0), (43, 32)])
@pytest.mark.parametrize("qs,ks", [(0.0, 0.0), (0.0, 1.0), (0.0, 1e-3), (1.0, 0.0), (3e-3, 0.0), (1e-25, 1e-25)])
def test_zero_and_tiny_operands(nh, nkv, hd, n, pos0, qs, ks):
    """Scores of zero: every row is a mean of V, masked keys (the diagonal's among them) stay masked."""
    q, k, v = inputs(n, pos0, nh, nkv, hd, 11)
    check(q * np.float32(qs), k * np.float32(ks), v, pos0, nh, nkv, hd)


@pytest.mark.parametrize("nh,nkv,hd", GEOMETRIES[:3])
def test_some_zero_rows(nh, nkv, hd):
    q, k, v = inputs(50, 30, nh, nkv, hd, 12)
    q[::3] = 0.0
    k[40:56] = 0.0
    v[8:12] = 0.0
    check(q, k, v, 30, nh, nkv, hd)
