"""Batched attention where magnitudes differ widely, against attention in float64, every (row, head) by its own
norm: what a row does not attend, or attends with next to no weight, must not cost it precision, and zeros are
ordinary values.

Bound: ordinary rows of these sizes measure 1e-7 to 5e-7 of their 2-norm (fp32 sums); where a score may be off by
2^-21 its weight is off by 3.3e-7 more.  1e-6 holds both.
"""
import numpy as np
import pytest

from tests.test_gpu_prefill_split import BASE, inputs, reference, run

pytestmark = pytest.mark.gpu

GEOMETRIES = [(4, 2, 64), (6, 2, 96), (7, 1, 128), (2, 1, 200)]


def unrotate(x, pos, hd):
    """x [n][heads * hd] as the library is to hold it after its rotation -> the rows to pass in (fp32)."""
    h = x.reshape(x.shape[0], -1, hd).astype(np.float64)
    inv = np.array([np.float32(np.power(BASE, -2.0 * i / hd)) for i in range(hd // 2)], np.float32).astype(np.float64)
    a = pos[:, None, None] * inv
    lo, hi = h[..., :hd // 2], h[..., hd // 2:]
    y = np.concatenate([lo * np.cos(a) + hi * np.sin(a), hi * np.cos(a) - lo * np.sin(a)], -1)
    return y.reshape(x.shape).astype(np.float32)


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


@pytest.mark.parametrize("nh,nkv,hd", GEOMETRIES)
@pytest.mark.parametrize("f", [1e2, 1e4, 1e6, 1e8, 1e16, 1e30])
def test_large_v_of_a_later_key(nh, nkv, hd, f):
    """V of position 56 is f times the others': the rows before it do not attend it."""
    q, k, v = inputs(64, 0, nh, nkv, hd, 13)
    v[56] *= np.float32(f)
    check(q, k, v, 0, nh, nkv, hd)


@pytest.mark.parametrize("nh,nkv,hd", GEOMETRIES)
@pytest.mark.parametrize("f", [1e2, 1e4, 1e6, 1e8])
def test_large_v_of_a_negligible_key(nh, nkv, hd, f):
    """An early key that no row gives any weight, V f times the others'; the tiles after it pay nothing."""
    q, k, v = inputs(70, 60, nh, nkv, hd, 14)
    q[:, ::hd] = 8.0                                  # position 3's score is some 160 below the others'
    k[:, ::hd] = 0.0
    k[3] = 0.0
    k[3, ::hd] = -20.0 * np.float32(np.sqrt(hd))
    q, k = unrotate(q, np.arange(60, 130), hd), unrotate(k, np.arange(130), hd)
    v[3] *= np.float32(f)
    check(q, k, v, 60, nh, nkv, hd)


@pytest.mark.parametrize("nh,nkv,hd", GEOMETRIES)
def test_v_whose_scale_changes(nh, nkv, hd):
    """V falls by 2^20 after the first tiles, which the later rows give next to no weight (and then rises again)."""
    q, k, v = inputs(96, 96, nh, nkv, hd, 15)
    v[:32] *= np.float32(2.0 ** 20)
    v[96:128] *= np.float32(2.0 ** 10)
    q[:, ::hd] = 8.0
    k[:, ::hd] = 0.0
    k[:32, ::hd] = -20.0 * np.float32(np.sqrt(hd))
    k[96:128, ::hd] = -10.0 * np.float32(np.sqrt(hd))
    q, k = unrotate(q, np.arange(96, 192), hd), unrotate(k, np.arange(192), hd)
    check(q, k, v, 96, nh, nkv, hd)


@pytest.mark.parametrize("nh,nkv,hd", GEOMETRIES)
@pytest.mark.parametrize("f", [1e3, 1e7])
def test_large_channel_of_v(nh, nkv, hd, f):
    """One channel of V is f times the others, which keep their own precision."""
    q, k, v = inputs(48, 40, nh, nkv, hd, 16)
    v = v.reshape(88, nkv, hd)
    v[..., 5] *= np.float32(f)
    v = v.reshape(88, -1)
    out, ref = run(q, k, v, 40, nh, nkv, hd), reference(q, k, v, 40, nh, nkv, hd)
    for d in (slice(0, 5), slice(5, 6), slice(6, hd)):
        err = np.linalg.norm(out[..., d] - ref[..., d], axis=(0, 2)) / np.linalg.norm(ref[..., d], axis=(0, 2))
        assert err.max() <= 1e-6, (d, err.max())


@pytest.mark.parametrize("nh,nkv,hd", GEOMETRIES)
@pytest.mark.parametrize("drop", [6.0, 14.0, 22.0, 40.0])
def test_sink(nh, nkv, hd, drop):
    """Position 0 takes nearly all the weight and its V is zero: the output is what the other keys' small weights,
    exp(-drop) of the largest, make of it."""
    q, k, v = inputs(40, 100, nh, nkv, hd, 20)
    q *= np.float32(0.2)
    q[:, ::hd] = 8.0
    k[:, ::hd] = 0.0
    k[0] = 0.0
    k[0, ::hd] = np.float32(drop * np.sqrt(hd) / 8.0)
    q, k = unrotate(q, np.arange(100, 140), hd), unrotate(k, np.arange(140), hd)
    v[0] = 0.0
    # the weights' arguments are differences of scores of up to drop, in fp32 (base 2, a rounding each way)
    check(q, k, v, 100, nh, nkv, hd, tol=1e-6 + drop * 1.45 * 2.0 ** -23)


@pytest.mark.parametrize("nh,nkv,hd", GEOMETRIES)
def test_zero_v_of_some_keys(nh, nkv, hd):
    """Keys of a group, and whole groups, whose V is zero and that get nearly all the weight."""
    q, k, v = inputs(40, 70, nh, nkv, hd, 21)
    q[:, ::hd] = 8.0
    k[:, ::hd] = 0.0
    zero = [2, 40, 41, 42, 43, 44, 45, 46, 47]
    k[zero, ::hd] = 2.0 * np.float32(np.sqrt(hd))
    q, k = unrotate(q, np.arange(70, 110), hd), unrotate(k, np.arange(110), hd)
    v[zero] = 0.0
    # scores of 16 and their differences, in base 2, each rounded in fp32
    check(q, k, v, 70, nh, nkv, hd, tol=1e-6 + 16 * 1.45 * 2.0 ** -22 * 0.69)


@pytest.mark.parametrize("nh,nkv,hd,n,pos0", [(7, 1, 128, 300, 500),      # key segments
                                              (56, 8, 128, 700, 0),       # long items halved
                                              (4, 2, 64, 900, 0), (33, 3, 96, 500, 100)])
@pytest.mark.parametrize("key", [3, 333])
def test_large_v_where_the_work_is_split(nh, nkv, hd, n, pos0, key):
    """Only some of the workgroups that share a row meet the large V."""
    q, k, v = inputs(n, pos0, nh, nkv, hd, 22)
    v[key] *= np.float32(1e8)
    out = run(q, k, v, pos0, nh, nkv, hd)
    for z in sorted({0, 1, n // 3, key - pos0 - 1, key - pos0, key - pos0 + 1, n - 1}):
        if 0 <= z < n:
            p = pos0 + z
            ref = reference(q[z:z + 1], k[:p + 1], v[:p + 1], p, nh, nkv, hd)[0]
            err = np.linalg.norm(out[z] - ref, axis=-1) / np.linalg.norm(ref, axis=-1)
            assert err.max() <= 1e-6, (z, err.max())


@pytest.mark.parametrize("nh,nkv,hd", GEOMETRIES)
@pytest.mark.parametrize("f", [1e2, 1e3, 1e4, 1e6, 1e8, 1e16, 1e30])
def test_large_k_of_a_later_key(nh, nkv, hd, f):
    """K of position 60 is f times its neighbours' in its group: rows before it do not attend it."""
    q, k, v = inputs(64, 0, nh, nkv, hd, 17)
    k[60] *= np.float32(f)
    check(q, k, v, 0, nh, nkv, hd, rows=slice(0, 60))


@pytest.mark.parametrize("nh,nkv,hd", GEOMETRIES)
@pytest.mark.parametrize("f", [1e4, 1e8])
def test_large_k_of_a_negligible_key(nh, nkv, hd, f):
    """Position 61's K is f times the others' and its score far below theirs."""
    q, k, v = inputs(60, 70, nh, nkv, hd, 18)
    q[:, ::hd] = 3.0
    k[:, ::hd] = 0.5
    k[61, ::hd] = -np.float32(f) * 30
    k[61].reshape(nkv, hd)[:, 1:] = 0.0
    q, k = unrotate(q, np.arange(70, 130), hd), unrotate(k, np.arange(130), hd)
    check(q, k, v, 70, nh, nkv, hd)


@pytest.mark.parametrize("nh,nkv,hd", GEOMETRIES)
def test_large_channel_of_q_that_k_lacks(nh, nkv, hd):
    """q's largest channel is 1e7 times the others, and every K is zero there."""
    q, k, v = inputs(40, 40, nh, nkv, hd, 19)
    q[:, ::hd] = 1e7
    q[:, hd // 2::hd] = 0.0
    k[:, ::hd] = 0.0
    k[:, hd // 2::hd] = 0.0
    check(q, k, v, 40, nh, nkv, hd)


@pytest.mark.parametrize("nh,nkv,hd", GEOMETRIES)
@pytest.mark.parametrize("spread", [3, 8])
def test_v_of_many_sizes(nh, nkv, hd, spread):
    """Every key's V its own size, and rows that attend a few keys, the smallest ones among them."""
    q, k, v = inputs(96, 100, nh, nkv, hd, 23)
    v *= np.exp2(np.random.default_rng(24).uniform(-spread, spread, (196, 1))).astype(np.float32)
    q *= np.float32(4.0)
    # scores of up to 4 * 4 sigma / ln 2, each and their differences rounded in fp32
    check(q, k, v, 100, nh, nkv, hd, tol=1e-6 + 24 * 2.0 ** -22 * 0.69)


@pytest.mark.parametrize("nh,nkv,hd", GEOMETRIES)
@pytest.mark.parametrize("key", [0, 45])
@pytest.mark.parametrize("drop", [8.0, 16.0, 24.0])
def test_sink_with_a_small_v(nh, nkv, hd, key, drop):
    """A key takes nearly all the weight and its V is 2^-9 of the others'."""
    q, k, v = inputs(40, 100, nh, nkv, hd, 25)
    q *= np.float32(0.2)
    q[:, ::hd] = 8.0
    k[:, ::hd] = 0.0
    k[key] = 0.0
    k[key, ::hd] = np.float32(drop * np.sqrt(hd) / 8.0)
    q, k = unrotate(q, np.arange(100, 140), hd), unrotate(k, np.arange(140), hd)
    v[key] *= np.float32(2.0 ** -9)
    check(q, k, v, 100, nh, nkv, hd, tol=1e-6 + drop * 1.45 * 2.0 ** -23)
