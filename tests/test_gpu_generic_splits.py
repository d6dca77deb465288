"""The decode of geometries without MFMA kernels at the edges of its tiles: 32-row tiles and splits, the new
row in every tile position and split, more than eight heads per kv-head (passes), rows of 8- and 16-byte
multiples, and stale non-finite values in the slot the new row takes.

Reference: the oracle's kore loops; bound 1e-5 of the largest output (fp64 scores; the sums over keys are
fp32 on both sides, at most 600 of them: 600 * 2^-24 = 3.6e-5 if every rounding went one way, a tenth of it
as they come)."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def check(nh, nkv, hd, ctx, positions, poison=None):
    from kore_amd import KoreAttn
    rng = np.random.default_rng(nh * 1000 + hd + ctx)
    kv = oracle.KV(1, ctx, nh, nkv, hd, 1e6)
    n0 = positions[0]
    with KoreAttn(1, ctx, nh, nkv, hd, 1e6) as a:
        if n0:
            x = [rng.standard_normal((n0, h * hd)).astype(np.float32) for h in (nh, nkv, nkv)]
            a.prefill(0, 0, *x)
            kv.prefill(0, 0, *x)
        if poison is not None:   # a row the decode overwrites
            x = [np.full((1, h * hd), poison, np.float32) for h in (nh, nkv, nkv)]
            a.prefill(0, n0, *x)
        for pos in positions:
            q, k, v = (rng.standard_normal(h * hd).astype(np.float32) for h in (nh, nkv, nkv))
            out = a.decode(0, pos, q, k, v)
            ref = kv.decode(0, pos, q, k, v)
            assert np.max(np.abs(out - ref)) <= 1e-5 * np.max(np.abs(ref)), pos
        n = positions[-1] + 1
        kg, vg = a.read_kv(0, 0, n)
    assert np.array_equal(kg, kv.kcache()[0][:n]) and np.array_equal(vg, kv.vcache()[0][:n])


@pytest.mark.parametrize("nh,nkv,hd", [(3, 3, 2), (8, 2, 6), (11, 1, 34), (33, 3, 96), (9, 1, 100), (17, 1, 130),
                                       (2, 1, 254), (4, 2, 256), (12, 1, 64)])
@pytest.mark.parametrize("n0", [0, 30, 63, 590])
def test_edges(nh, nkv, hd, n0):
    check(nh, nkv, hd, n0 + 4, [n0, n0 + 1, n0 + 2, n0 + 3])


@pytest.mark.parametrize("poison", [np.nan, np.inf])
def test_stale_slot(poison):
    check(33, 3, 96, 70, [64], poison=poison)


def test_many_splits():
    """More tiles than splits: several tiles each."""
    check(64, 32, 36, 600, [590, 591])


@pytest.mark.parametrize("nh,nkv,hd,n0,bad", [(33, 3, 96, 32, range(32, 33)),     # the new row, alone in its tile and split
                                              (2, 2, 34, 64, range(64, 65)),
                                              (64, 32, 36, 598, range(64, 96)),   # the first of a split's two tiles
                                              (64, 32, 36, 598, range(96, 128)),  # the second
                                              (64, 32, 36, 598, range(64, 128))]) # a whole split
def test_tile_of_minus_infinity(nh, nkv, hd, n0, bad):
    """Rows whose scores are -inf (an infinity in K against a q of the other sign) weigh nothing, also where they
    are all of a tile."""
    from kore_amd import KoreAttn
    rng = np.random.default_rng(5)
    q, k, v = (rng.standard_normal((n0 + 1, h * hd)).astype(np.float32) for h in (nh, nkv, nkv))
    for d in (hd // 2 - 1, hd - 1):                  # the pair with the slowest rotation: both stay below 0
        q[:, d::hd] = -1.0
    k.reshape(-1, nkv, hd)[list(bad), :, hd // 2 - 1] = np.inf
    kv = oracle.KV(1, n0 + 1, nh, nkv, hd, 1e6)
    with KoreAttn(1, n0 + 1, nh, nkv, hd, 1e6) as a, np.errstate(invalid="ignore"):
        a.prefill(0, 0, q[:n0], k[:n0], v[:n0])
        kv.prefill(0, 0, q[:n0], k[:n0], v[:n0])
        out, ref = a.decode(0, n0, q[n0], k[n0], v[n0]), kv.decode(0, n0, q[n0], k[n0], v[n0])
    assert np.all(np.isfinite(ref))
    assert np.max(np.abs(out - ref)) <= 1e-5 * np.max(np.abs(ref))


def test_many_rows_against_float64():
    """63 splits merged.  2-norm of the error, mean of six draws: 1.56e-7, and 1.98e-7 where the sum of the weights
    is added up one split after the other and the factors between splits are rounded."""
    from kore_amd import KoreAttn
    from tests.test_gpu_prefill_split import reference
    nh, nkv, hd, n0, errs = 33, 3, 96, 2000, []
    for seed in range(6):
        rng = np.random.default_rng(seed)
        q, k, v = (rng.standard_normal((n0 + 1, h * hd)).astype(np.float32) for h in (nh, nkv, nkv))
        q[:, ::17] *= 4
        k[:, ::17] *= 4
        with KoreAttn(1, n0 + 1, nh, nkv, hd, 1e4) as a:
            a.prefill(0, 0, np.zeros_like(q[:n0]), k[:n0], v[:n0])
            out = a.decode(0, n0, q[n0], k[n0], v[n0]).reshape(nh, hd)
        ref = reference(q[n0:], k, v, n0, nh, nkv, hd)[0]
        errs.append(np.linalg.norm(out - ref) / np.linalg.norm(ref))
    assert np.mean(errs) <= 1.8e-7, errs
