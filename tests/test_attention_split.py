"""Attention on the bf16 matrix cores (head dim 64, grids large enough that the
library takes it there), against float64: ragged query and key counts, strided
and unaligned operands, scales, non-finite and extreme values.

Bar: scores err by at most 1e-6 of sum |q k| times the scale (the SGEMM bar at
64 products is 1e-5 sqrt(64) = 8e-5 of it; measured 1e-7), which moves a
weight by that factor; 2e-5 relative to sum_j p_j |v_j| covers it at the
magnitudes drawn here (scores within +-6)."""

import numpy as np
import pytest

from conftest import rng
from gpu_util import announce, down, empty, up

pytestmark = pytest.mark.gpu

D = 64


def _ref(Q, K, V, scale):
    S = Q.astype(np.float64) @ K.astype(np.float64).transpose(0, 2, 1) * scale
    with np.errstate(invalid="ignore", over="ignore"):
        P = np.exp(S - S.max(-1, keepdims=True))
        P /= P.sum(-1, keepdims=True)
        return P @ V.astype(np.float64), P @ np.abs(V.astype(np.float64))


def _run(native, Q, K, V, scale):
    b, Sq, _ = Q.shape
    Sk = K.shape[1]
    dQ, dK, dV, dO = up(native, Q), up(native, K), up(native, V), empty(native, b * Sq * D)
    native.attention(Sq, Sk, D, scale, dQ, D, dK, D, dV, D, dO, D, 1, b, (0, Sq * D), (0, Sk * D),
                     (0, Sk * D), (0, Sq * D))
    return down(native, dO, (b, Sq, D))


@pytest.mark.parametrize("b,Sq,Sk", [(200, 127, 513), (200, 128, 576), (100, 129, 1023),
                                     (100, 255, 640), (60, 400, 801), (24, 1000, 1000),
                                     (210, 100, 449)])
def test_ragged_sizes(native, b, Sq, Sk):
    announce(f"attention split {b} x {Sq} x {Sk}")
    g = rng(b + Sq + Sk)
    Q, K, V = (g.normal(0, 1, (b, s, D)).astype(np.float32) for s in (Sq, Sk, Sk))
    O = _run(native, Q, K, V, 0.125)
    want, mag = _ref(Q, K, V, 0.125)
    assert np.all(np.abs(O - want) <= 2e-5 * mag)


@pytest.mark.parametrize("b,Sq,Sk", [(256, 128, 101), (256, 128, 128), (256, 127, 129),
                                     (256, 97, 160), (256, 128, 161), (128, 250, 192),
                                     (128, 256, 225), (256, 100, 257)])
def test_few_key_blocks(native, b, Sq, Sk):
    """Two to five blocks of 64 keys: the start and the end of the pipeline
    over key blocks, with one half of the last block empty or not."""
    announce(f"attention split, few blocks {b} x {Sq} x {Sk}")
    g = rng(b + Sq + Sk)
    Q, K, V = (g.normal(0, 1, (b, s, D)).astype(np.float32) for s in (Sq, Sk, Sk))
    O = _run(native, Q, K, V, 0.125)
    want, mag = _ref(Q, K, V, 0.125)
    assert np.all(np.abs(O - want) <= 2e-5 * mag)


def test_strided_and_unaligned(native):
    """Heads cut out of [batch, seq, 3 * heads * 64 + 1] rows, one float off
    16-byte alignment, merged heads out; rows past the output untouched."""
    announce("attention split strided")
    g = rng(17)
    B, S, H = 16, 500, 12
    W = 3 * H * D + 1
    X = g.normal(0, 1, (B * S * W + 1,)).astype(np.float32)
    Y = X[1:].reshape(B, S, W)
    dX, dO = up(native, X), up(native, np.full(B * S * (H * D + 3), 9.0, np.float32))
    st = (S * W, D)
    native.attention(S, S, D, 0.2, dX, W, dX, W, dX, W, dO, H * D + 3, B, H, st, st, st,
                     (S * (H * D + 3), D), offsets=(1, 1 + H * D, 1 + 2 * H * D, 0))
    O = down(native, dO, (B, S, H * D + 3))
    assert np.all(O[:, :, H * D:] == 9.0)
    for b in (0, 7, 15):
        q, k, v = (np.ascontiguousarray(Y[b, :, i * H * D:(i + 1) * H * D].reshape(S, H, D)
                                        .transpose(1, 0, 2)) for i in range(3))
        want, mag = _ref(q, k, v, 0.2)
        got = O[b, :, :H * D].reshape(S, H, D).transpose(1, 0, 2)
        assert np.all(np.abs(got - want) <= 2e-5 * mag)


def test_non_finite_values(native):
    """A -inf score drops its key; NaN and +inf reach the rows they belong to,
    and no others."""
    announce("attention split: non-finite operands")
    g = rng(23)
    b, Sq, Sk = 200, 128, 576
    Q = np.abs(g.normal(0, 1, (b, Sq, D))).astype(np.float32) + 0.1
    K, V = (g.normal(0, 1, (b, Sk, D)).astype(np.float32) for _ in range(2))
    clean = _run(native, Q, K, V, 0.125)
    K2, V2, Q2 = K.copy(), V.copy(), Q.copy()
    K2[3, 100, 5] = -np.inf       # -inf score for every row: the key drops out
    V2[5, 9, 11] = np.inf         # +inf in column 11 of every row
    V2[6, 570, 3] = np.nan
    Q2[9, 17, 0] = np.inf         # the row's scores are +-inf: NaN
    O = _run(native, Q2, K2, V2, 0.125)
    want, mag = _ref(Q[3:4], np.delete(K[3:4], 100, 1), np.delete(V[3:4], 100, 1), 0.125)
    assert np.all(np.abs(O[3:4] - want) <= 2e-5 * mag)
    assert np.all(np.isposinf(O[5, :, 11])) and np.all(np.isnan(O[6, :, 3]))
    assert np.all(np.isnan(O[9, 17]))
    same = np.ones(O.shape, bool)
    same[3], same[5, :, 11], same[6, :, 3], same[9, 17] = False, False, False, False
    _, mag = _ref(Q, K, V, 0.125)
    assert np.all(np.abs(O - clean)[same] <= 4e-5 * mag[same])


@pytest.mark.parametrize("qs,vs", [(1e-30, 1.0), (1.0, 1e-36), (1.0, 1e30), (40.0, 1.0),
                                   (1e19, 1.0)])
def test_extreme_magnitudes(native, qs, vs):
    """Tiny and huge operands: scores that vanish, values near both ends of the
    range, one key taking all the weight."""
    announce(f"attention split q {qs} v {vs}")
    g = rng(29)
    b, Sq, Sk = 200, 128, 576
    Q = (g.normal(0, 1, (b, Sq, D)) * qs).astype(np.float32)
    K = g.normal(0, 1, (b, Sk, D)).astype(np.float32)
    V = (g.normal(0, 1, (b, Sk, D)) * vs).astype(np.float32)
    O = _run(native, Q, K, V, 0.125)
    want, mag = _ref(Q, K, V, 0.125)
    # scores of magnitude s carry an absolute error of about s 2^-22
    S = np.abs(Q.astype(np.float64) @ K.astype(np.float64).transpose(0, 2, 1)).max(-1) * 0.125
    factor = np.minimum(2.0, 2e-5 + 2.0 ** -20 * S)[..., None]
    top = np.abs(V).max(1, keepdims=True).astype(np.float64)
    assert np.all(np.isfinite(O))
    assert np.all(np.abs(O - want) <= factor * np.maximum(mag, top * (factor > 1e-3)) + 1e-44)


@pytest.mark.parametrize("qs", [1e15, 1e19])
def test_huge_scores_pick_one_key(native, qs):
    """Scores around 1e15 (on the bf16 matrix cores) and 1e19 (operands over 2^60:
    every row redone in fp32).  A score of 64 products errs by at most 64 * 2^-24 of
    sum |q k|, which is under four times the row's largest score: 2^-16 of that.
    Where the second score is further off, the row is the value of its first key."""
    announce(f"attention split: scores about {qs}")
    g = rng(31)
    b, Sq, Sk = 200, 128, 576
    Q = (g.normal(0, 1, (b, Sq, D)) * qs).astype(np.float32)
    K, V = (g.normal(0, 1, (b, Sk, D)).astype(np.float32) for _ in range(2))
    O = _run(native, Q, K, V, 0.125)
    S = Q.astype(np.float64) @ K.astype(np.float64).transpose(0, 2, 1)
    first = S.argmax(-1)
    top = np.partition(S, Sk - 2, axis=-1)[..., -2:]
    largest = np.abs(S).max(-1)
    mag = np.abs(Q.astype(np.float64)) @ np.abs(K.astype(np.float64)).transpose(0, 2, 1)
    assert np.all(mag.max(-1) < 4 * largest)
    clear = top[..., 1] - top[..., 0] > 2.0 ** -16 * largest
    assert clear.mean() > 0.99
    want = np.take_along_axis(V, first[..., None], axis=1)
    assert np.all(np.isfinite(O))
    assert np.array_equal(O[clear], want[clear])


@pytest.mark.parametrize("Sq,Sk", [(128, 576), (97, 530), (130, 31 + 512)])
def test_values_near_the_bottom_of_the_range(native, Sq, Sk):
    """V elements under 2^-134 have no bf16 part; their averages are not zero.
    Beside columns of zeros, and in one head of many.  Each of the Sk products
    of P and V rounds to a subnormal once: Sk * 2^-149 above the bar."""
    announce(f"attention split: subnormal values {Sq} x {Sk}")
    g = rng(Sq + Sk)
    b = 200
    Q, K, V = (g.normal(0, 1, (b, s, D)).astype(np.float32) for s in (Sq, Sk, Sk))
    V[3] = g.uniform(2e-41, 4e-41, V[3].shape)
    V[3, :, 7] = 0.0
    V[7] = (1e-36 * V[7]).astype(np.float32)
    V[9, :, 5], V[9, :, 6] = 0.0, 2000.0 * V[9, :, 6]
    O = _run(native, Q, K, V, 0.125)
    want, mag = _ref(Q, K, V, 0.125)
    assert np.all(np.abs(O - want) <= 2e-5 * mag + Sk * 2.0 ** -149)
    assert np.all(O[3, :, 7] == 0.0) and np.all(O[9, :, 5] == 0.0)


@pytest.mark.parametrize("Sq,Sk", [(128, 576), (97, 530), (130, 31 + 512)])
def test_rows_redone(native, Sq, Sk):
    """An infinite value in some heads: their rows come from the fp32 matrix
    cores, and agree in every other column; a NaN stays in its column."""
    announce(f"attention split: rows redone {Sq} x {Sk}")
    g = rng(Sq + Sk)
    b = 200
    Q, K, V = (g.normal(0, 1, (b, s, D)).astype(np.float32) for s in (Sq, Sk, Sk))
    want, mag = _ref(Q, K, V, 0.125)
    V[::3, Sk - 1, 63], V[1::3, 0, 2] = np.inf, np.nan
    O = _run(native, Q, K, V, 0.125)
    assert np.all(np.isposinf(O[::3, :, 63])) and np.all(np.isnan(O[1::3, :, 2]))
    same = np.ones(O.shape, bool)
    same[::3, :, 63] = same[1::3, :, 2] = False
    assert np.all((np.abs(O - want) <= 2e-5 * mag)[same])


@pytest.mark.parametrize("zeros", [1, 3, 9])
def test_sums_that_cancel_to_zero(native, zeros):
    """A row of equal weights over a column of V whose values cancel, in few and in
    many columns: zero to within the rounding of its terms, and next to it a column
    whose values are too small for bf16 parts, in the same row."""
    announce(f"attention split: {zeros} columns cancel")
    g = rng(41 + zeros)
    b, Sq, Sk = 200, 128, 576
    Q, K, V = (g.normal(0, 1, (b, s, D)).astype(np.float32) for s in (Sq, Sk, Sk))
    Q[3, 5] = Q[9, 77] = 0.0
    V[3, ::2, 7:7 + zeros] = -V[3, 1::2, 7:7 + zeros]
    V[9, :, 7] = 3e-41
    O = _run(native, Q, K, V, 0.125)
    want, mag = _ref(Q, K, V, 0.125)
    assert np.all(np.abs(O - want) <= 2e-5 * mag + Sk * 2.0 ** -149)
    assert np.all(O[9, :, 7] > 2.9e-41)
