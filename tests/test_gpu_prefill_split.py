"""prefill_kernel's split-fp16 products, and the fp32 ones that it falls back to, against attention in float64:
head dims and rows at the edges of its tiles (padded dims, strips of 32 query rows, 32-key tiles, key segments),
operands far outside fp16's range, and infinities and NaN in the cache.

Bound: a weight 2^(t - m) is off by ln2 times the error of its argument: the split keeps 22 bits of each
operand (three products), one rounding per 16 dims at the size of the score, and t stays below 64 for
these inputs, so 64 * 2^-24 * (hd / 16 + 4) <= 8e-5 at head_dim 256 for every key at once; the sums over
keys average it down.  3e-5 of a row's largest output holds with room, every (row, head) by its own.
"""
import numpy as np
import pytest

from kore_amd import KoreAttn

pytestmark = pytest.mark.gpu
BASE = 1e4


def rope32(x, pos, hd):
    """x [n][heads][hd] fp32, rotated as the library does (double angles, fp32 products)."""
    inv = np.array([np.float32(np.power(BASE, -2.0 * i / hd)) for i in range(hd // 2)], np.float32)
    a = pos[:, None].astype(np.float64) * inv.astype(np.float64)
    c, s = np.cos(a).astype(np.float32)[:, None], np.sin(a).astype(np.float32)[:, None]
    lo, hi = x[..., :hd // 2], x[..., hd // 2:]
    with np.errstate(invalid="ignore", over="ignore"):
        return np.concatenate([lo * c - hi * s, lo * s + hi * c], -1)


def reference(q, k, v, pos0, nh, nkv, hd):
    """Rows pos0.. of q over all rows of k, v (positions 0..), in float64."""
    n, m = q.shape[0], k.shape[0]
    qr = rope32(q.reshape(n, nh, hd), np.arange(pos0, pos0 + n), hd).astype(np.float64)
    kr = rope32(k.reshape(m, nkv, hd), np.arange(m), hd).astype(np.float64)
    v = v.reshape(m, nkv, hd).astype(np.float64)
    out = np.empty((n, nh, hd))
    with np.errstate(invalid="ignore", over="ignore"):
        for z in range(n):
            e = pos0 + z + 1
            for h in range(nh):
                g = h // (nh // nkv)
                s = (kr[:e, g] * qr[z, h]).sum(-1) / np.sqrt(hd)
                w = np.exp(s - s.max())
                out[z, h] = (w[:, None] * v[:e, g]).sum(0) / w.sum()
    return out


def run(q, k, v, pos0, nh, nkv, hd):
    n = q.shape[0]
    with KoreAttn(1, pos0 + n, nh, nkv, hd, BASE) as a:
        if pos0:
            a.prefill(0, 0, np.zeros((pos0, nh * hd), np.float32), k[:pos0], v[:pos0])
        return a.prefill(0, pos0, q, k[pos0:], v[pos0:]).reshape(n, nh, hd)


def inputs(n, pos0, nh, nkv, hd, seed=0):
    r = np.random.default_rng(seed)
    m = pos0 + n
    return (r.standard_normal((n, nh * hd)).astype(np.float32), r.standard_normal((m, nkv * hd)).astype(np.float32),
            r.standard_normal((m, nkv * hd)).astype(np.float32))


def close(out, ref):
    err, top = np.abs(out - ref).max(-1), np.abs(ref).max(-1)
    assert np.all(err <= 3e-5 * top), (err / top).max()


@pytest.mark.parametrize("nh,nkv,hd,n,pos0", [
    (3, 3, 2, 5, 0), (4, 2, 14, 33, 0), (2, 1, 30, 31, 2), (11, 1, 32, 12, 70), (5, 5, 34, 40, 31),
    (6, 2, 62, 43, 1), (14, 2, 64, 19, 300), (3, 1, 66, 65, 0), (22, 2, 96, 12, 95), (7, 1, 98, 37, 5),
    (12, 2, 126, 9, 33), (9, 3, 128, 65, 400), (12, 1, 128, 11, 0), (2, 2, 130, 35, 20), (4, 1, 160, 33, 64),
    (3, 3, 190, 6, 40), (5, 1, 192, 26, 7), (2, 1, 222, 70, 0), (4, 2, 256, 33, 130), (1, 1, 256, 1, 0),
])
def test_edges(nh, nkv, hd, n, pos0):
    q, k, v = inputs(n, pos0, nh, nkv, hd)
    out, ref = run(q, k, v, pos0, nh, nkv, hd), reference(q, k, v, pos0, nh, nkv, hd)
    close(out, ref)


@pytest.mark.parametrize("nh,nkv,hd", [(4, 2, 64), (6, 2, 96), (7, 1, 128), (2, 1, 200)])
@pytest.mark.parametrize("qs,ks,vs", [(1e6, 1e-6, 1e-12), (1e-9, 1e9, 1e12), (1e-3, 1e3, 1e30), (1.0, 1.0, 1e-30)])
def test_scales(nh, nkv, hd, qs, ks, vs):
    q, k, v = inputs(40, 50, nh, nkv, hd, 1)
    q, k, v = q * np.float32(qs), k * np.float32(ks), v * np.float32(vs)
    out, ref = run(q, k, v, 50, nh, nkv, hd), reference(q, k, v, 50, nh, nkv, hd)
    close(out, ref)


@pytest.mark.parametrize("nh,nkv,hd", [(4, 2, 64), (9, 3, 96), (7, 1, 128)])
def test_scales_that_differ_by_row(nh, nkv, hd):
    """Every key has its own scale: rows of V over 2^24, of K over 2^12 (their scores stay small)."""
    q, k, v = inputs(60, 40, nh, nkv, hd, 2)
    r = np.random.default_rng(3)
    v *= np.exp2(r.integers(-12, 13, (100, 1))).astype(np.float32)
    k *= np.exp2(r.integers(-12, 1, (100, 1))).astype(np.float32)
    out, ref = run(q, k, v, 40, nh, nkv, hd), reference(q, k, v, 40, nh, nkv, hd)
    close(out, ref)


@pytest.mark.parametrize("nh,nkv,hd", [(4, 2, 64), (6, 2, 96), (7, 1, 128), (2, 1, 136)])
@pytest.mark.parametrize("where", ["k_inf", "k_nan", "v_inf", "v_ninf", "v_nan", "q_inf", "v_both"])
def test_non_finite(nh, nkv, hd, where):
    """They reach the rows that attend them, and the dims they are in, and nothing else."""
    q, k, v = inputs(45, 60, nh, nkv, hd, 4)
    at, dim = 83, 3                    # a key of the chunk: rows before it do not attend it
    if where == "q_inf":
        q[at - 60, dim] = np.inf
    elif where == "v_both":
        v[at, dim], v[at + 2, dim], v[20, dim + 1] = np.inf, -np.inf, -np.inf
    else:
        x = {"inf": np.inf, "ninf": -np.inf, "nan": np.nan}[where.split("_")[1]]
        (k if where[0] == "k" else v)[at, dim] = x
    out, ref = run(q, k, v, 60, nh, nkv, hd), reference(q, k, v, 60, nh, nkv, hd)
    assert np.array_equal(np.isnan(out), np.isnan(ref))
    assert np.array_equal(np.isposinf(out), np.isposinf(ref)) and np.array_equal(np.isneginf(out), np.isneginf(ref))
    f = np.isfinite(ref)
    assert np.max(np.abs(out[f] - ref[f])) <= 3e-5 * np.max(np.abs(ref[f]))
