"""The products that run on the bf16 matrix cores with every float split in
three (forced tiles 1 and 5), against float64.

Bars: the SGEMM bar of gpu_util (1e-5 sqrt(K) of sum |a b| per element and
normwise); the split itself stays under it by far (2^-26 per product).  Sums
whose products leave the normal range add K * 2^-149 per element, one
rounding of a subnormal per product.
"""

import numpy as np
import pytest

from conftest import rng
from gpu_util import announce, down, empty, gemm_tolerance_ok, up

pytestmark = pytest.mark.gpu

TILE_128x128, TILE_128x64, TILE_256x128 = 1, 4, 5


def _run(native, A, B, ta=0, tb=0, tile=TILE_128x128, splits=1, pad=0, off=0):
    """op(A) op(B) through silgpu_sgemm_tuned; pad floats between rows, off
    floats ahead of each operand, C surrounded by values that must survive."""
    M, K = (A.shape[1], A.shape[0]) if ta else A.shape
    N = B.shape[0] if tb else B.shape[1]

    def put(X):
        Y = np.full((X.shape[0], X.shape[1] + pad), np.nan, np.float32)
        Y[:, :X.shape[1]] = X
        return up(native, np.concatenate([np.full(off, np.nan, np.float32), Y.ravel()])), \
            Y.shape[1]

    dA, lda = put(A)
    dB, ldb = put(B)
    ldc = N + pad
    dC = up(native, np.full(off + M * ldc + 64, 7.0, np.float32))
    native.sgemm_tuned(ta, tb, M, N, K, dA.at(4 * off), lda, 0, dB.at(4 * off), ldb, 0,
                       dC.at(4 * off), ldc, 0, tile=tile, splits=splits)
    out = down(native, dC, (off + M * ldc + 64,))
    C = out[off:off + M * ldc].reshape(M, ldc)
    assert np.all(out[:off] == 7.0) and np.all(out[off + M * ldc:] == 7.0)
    assert np.all(C[:, N:] == 7.0)
    return C[:, :N].copy()


def _check(C, A, B, ta=0, tb=0):
    A64, B64 = (A.T if ta else A).astype(np.float64), (B.T if tb else B).astype(np.float64)
    K = A64.shape[1]
    ok, nw, el = gemm_tolerance_ok(C, A64 @ B64, np.abs(A64) @ np.abs(B64), K)
    assert ok, (nw, el)


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("tile,M,N,K", [
    (1, 1, 1, 1), (1, 2, 3, 2), (1, 127, 129, 15), (1, 128, 128, 32), (1, 129, 127, 33),
    (1, 64, 200, 31), (1, 130, 260, 95), (1, 256, 128, 96), (1, 257, 131, 161),
    (5, 1, 130, 1), (5, 255, 127, 16), (5, 256, 128, 48), (5, 257, 129, 17), (5, 40, 513, 47),
    (5, 300, 300, 64), (5, 511, 255, 65), (5, 512, 256, 129)])
def test_tile_edges(native, tile, M, N, K, ta, tb):
    announce(f"bf16 split tile {tile} {M}x{N}x{K} ta={ta} tb={tb}")
    g = rng(31 * M + 7 * N + K)
    A = g.normal(0, 1, (K, M) if ta else (M, K)).astype(np.float32)
    B = g.normal(0, 1, (N, K) if tb else (K, N)).astype(np.float32)
    _check(_run(native, A, B, ta, tb, tile), A, B, ta, tb)
    _check(_run(native, A, B, ta, tb, tile, pad=3, off=1), A, B, ta, tb)
    if K >= 64:
        _check(_run(native, A, B, ta, tb, tile, splits=2, pad=1), A, B, ta, tb)


def test_k_splits_are_the_sum_of_their_ranges(native):
    announce("bf16 split: K splits add up")
    g = rng(5)
    A = g.normal(0, 1, (300, 640)).astype(np.float32)
    B = g.normal(0, 1, (640, 200)).astype(np.float32)
    for tile in (TILE_128x128, TILE_256x128):
        want = np.zeros((300, 200), np.float32)
        for k0 in (0, 224, 448):  # ranges of whole 32s: 224, 224, 192
            k1 = min(640, k0 + 224)
            want = want + _run(native, A[:, k0:k1].copy(), B[k0:k1].copy(), tile=tile)
        assert np.array_equal(_run(native, A, B, tile=tile, splits=3), want)


@pytest.mark.parametrize("tile", [1, 5])
def test_infinities_and_nans(native, tile):
    """Every output is what IEEE arithmetic gives: inf, -inf, NaN (also inf *
    0) and finite ones in the same tile."""
    announce(f"bf16 split tile {tile}: non-finite operands")
    g = rng(9)
    A = g.normal(0, 1, (300, 70)).astype(np.float32)
    B = g.normal(0, 1, (70, 150)).astype(np.float32)
    A[3, 5], A[40, 6], A[41, 6], A[200, 0] = np.inf, -np.inf, np.nan, np.inf
    A[200, 1] = -np.inf
    B[5, 7], B[9, 100], B[69, 149] = 0.0, np.inf, np.nan
    with np.errstate(invalid="ignore"):
        want = (A[:, :, None].astype(np.float64) * B[None].astype(np.float64)).sum(1)
    C = _run(native, A, B, tile=tile)
    assert np.array_equal(np.isnan(C), np.isnan(want))
    inf = np.isinf(want)
    assert np.array_equal(C[inf], want[inf].astype(np.float32))
    fin = np.isfinite(want)
    bound = 1e-5 * np.sqrt(70) * (np.abs(np.nan_to_num(A, posinf=0, neginf=0)).astype(np.float64)
                                  @ np.abs(np.nan_to_num(B, posinf=0, neginf=0)))
    assert np.all(np.abs(C[fin] - want[fin]) <= bound[fin])


@pytest.mark.parametrize("tile", [1, 5])
@pytest.mark.parametrize("name,a,b", [
    ("lowest", -3.4028234e38, 1e-3),       # rounds to a bf16 infinity
    ("near the top", 1e30, 1e7),
    ("tiny", 1e-36, 1.0),                  # parts under bf16's normal range
    ("tiny both", 1e-17, 1e-18),
    ("tiny by huge", 1e-37, 1e30),
    ("subnormal by huge", 1e-41, 1e25)])
def test_extreme_magnitudes(native, tile, name, a, b):
    announce(f"bf16 split tile {tile}: {name}")
    g = rng(77)
    K = 65
    A = (np.float64(a) * g.uniform(0.5, 1, (200, K))).astype(np.float32)
    B = (np.float64(b) * g.uniform(0.5, 1, (K, 140)) * np.where(g.random((K, 140)) < .5, -1, 1)
         ).astype(np.float32)
    C = _run(native, A, B, tile=tile)
    A64, B64 = A.astype(np.float64), B.astype(np.float64)
    bar = 1e-5 * np.sqrt(K) * (np.abs(A64) @ np.abs(B64)) + K * 2.0 ** -149
    assert np.all(np.abs(C - A64 @ B64) <= bar)


def _near_the_bottom(C, A, B):
    A64, B64 = A.astype(np.float64), B.astype(np.float64)
    K = A.shape[1]
    bar = 1e-5 * np.sqrt(K) * (np.abs(A64) @ np.abs(B64)) + K * 2.0 ** -149
    return np.all(np.abs(C - A64 @ B64) <= bar)


@pytest.mark.parametrize("tile", [1, 5])
@pytest.mark.parametrize("a,b,K", [(4e-41, 1e3, 8192), (1e-41, 1.0, 8192), (4e-41, 1e3, 70),
                                   (1e-44, 900.0, 333), (1e-30, 1e-9, 2048)])
def test_sums_of_elements_that_round_to_zero(native, tile, a, b, K):
    """|x| under 2^-134 has no bf16 part, and a product under 2^-149 no value:
    the sums of many are normal floats."""
    announce(f"bf16 split tile {tile}: {a} by {b}, K={K}")
    g = rng(K)
    A = (np.float64(a) * g.uniform(0.5, 1, (140, K))).astype(np.float32)
    B = (np.float64(b) * g.uniform(0.5, 1, (K, 135))).astype(np.float32)
    B[:, 7] = 0.0
    assert _near_the_bottom(_run(native, A, B, tile=tile), A, B)


@pytest.mark.parametrize("tile", [1, 5])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_one_subnormal_element_anywhere(native, tile, ta, tb):
    """A single element that rounds to zero beside zeros, at the edges of the
    tiles and of the K range, in A or in B: its row (column) is not lost."""
    M, N, K = 259, 133, 277
    for r, k in [(0, 0), (258, 276), (127, 255), (128, 256), (255, 16), (256, 275), (31, 1)]:
        announce(f"bf16 split tile {tile} ta={ta} tb={tb}: subnormal at {r}, {k}")
        for swap in (False, True):
            g = rng(r + k)
            A, B = np.zeros((M, K), np.float32), np.zeros((K, N), np.float32)
            small, big = (B.T, A.T) if swap else (A, B)
            r_ = min(r, small.shape[0] - 1)
            small[r_, k] = 3e-41
            big[:] = g.uniform(1000, 1023, big.shape)
            C = _run(native, np.ascontiguousarray(A.T) if ta else A,
                     np.ascontiguousarray(B.T) if tb else B, ta, tb, tile,
                     splits=2 if swap else 1)
            assert _near_the_bottom(C, A, B), (r, k, swap)


@pytest.mark.parametrize("tile", [1, 5])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("few", [True, False])
def test_sums_that_cancel_beside_sums_that_vanish(native, tile, ta, tb, few):
    """Sums that are exactly zero because their terms cancel, few and many in a wave's
    tile, and among them one of elements that have no bf16 part, which is not zero."""
    announce(f"bf16 split tile {tile} ta={ta} tb={tb}: cancelled sums, few={few}")
    M, N, K = 300, 150, 330
    g = rng(K + few)
    A = g.uniform(0.5, 1, (M, K)).astype(np.float32)
    B = g.uniform(0.5, 1, (K, N)).astype(np.float32)
    for m, n in [(0, 0), (129, 37), (299, 149)] if few else \
            [(m, n) for m in range(0, 300, 9) for n in range(0, 150, 10)]:
        A[m, 1::2] = -A[m, ::2]
        B[1::2, n] = B[::2, n]
    A[70], B[:, 70] = 0.0, 0.0
    A[70, 11], B[11, 70] = 3e-41, 1000.0
    C = _run(native, np.ascontiguousarray(A.T) if ta else A,
             np.ascontiguousarray(B.T) if tb else B, ta, tb, tile)
    assert _near_the_bottom(C, A, B) and C[70, 70] > 0


@pytest.mark.parametrize("tile", [1, 5])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K", [(33, 65, 1), (257, 129, 5), (130, 131, 8), (259, 70, 71),
                                   (128, 257, 130)])
def test_products_redone_whole(native, tile, ta, tb, M, N, K):
    """Every sum small beside elements that lose parts: all of C comes from
    the fp32 matrix cores."""
    announce(f"bf16 split tile {tile} redone {M}x{N}x{K} ta={ta} tb={tb}")
    g = rng(M + N + K)
    A = (1e-34 * g.normal(0, 1, (M, K))).astype(np.float32)
    B = g.normal(0, 1, (K, N)).astype(np.float32)
    for splits in (1, 2) if K >= 64 else (1,):
        C = _run(native, np.ascontiguousarray(A.T) if ta else A,
                 np.ascontiguousarray(B.T) if tb else B, ta, tb, tile, splits, pad=3, off=1)
        assert _near_the_bottom(C, A, B)


@pytest.mark.parametrize("tile", [1, 5])
def test_rows_of_any_scale_keep_their_accuracy(native, tile):
    """Rows of A and columns of B from 1e-12 to 1e12, elements over 1e16 within
    a row: every element within the bar of its own sum |a b|."""
    announce(f"bf16 split tile {tile}: mixed scales")
    g = rng(13)
    A = (g.normal(0, 1, (260, 90)) * 10.0 ** g.uniform(-12, 12, (260, 1))
         * 10.0 ** g.uniform(-8, 8, (260, 90))).astype(np.float32)
    B = (g.normal(0, 1, (90, 140)) * 10.0 ** g.uniform(-6, 6, (1, 140))).astype(np.float32)
    A[:, 0], B[0, :70] = 1e15, 0.0
    C = _run(native, A, B, tile=tile)
    A64, B64 = A.astype(np.float64), B.astype(np.float64)
    assert np.all(np.abs(C - A64 @ B64) <= 1e-5 * np.sqrt(90) * (np.abs(A64) @ np.abs(B64)))


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("tile,M,N,K", [(1, 511, 1027, 333), (5, 700, 1027, 333)])
def test_batches_of_two_levels(native, tile, M, N, K, ta, tb):
    """Batched products as the planner sends them here: 2 x 3 of them, the inner
    three side by side in one row, A's outer stride wider than its product and B the
    same for both.  In one product every sum is redone on the fp32 matrix cores."""
    announce(f"bf16 split tile {tile} batched {M}x{N}x{K} ta={ta} tb={tb}")
    g = rng(M + 2 * ta + tb)
    ar, ac = (K, M) if ta else (M, K)
    br, bc = (N, K) if tb else (K, N)
    A = g.normal(0, 1, (2, ar + 2, 3, ac + 1)).astype(np.float32)
    B = g.normal(0, 1, (br, 3, bc)).astype(np.float32)
    A[1, :, 1] *= 1e-34
    dA, dB = up(native, A), up(native, B)
    dC = up(native, np.full((2, M, 3, N + 1), 7.0, np.float32))
    native.gemm(ta, tb, M, N, K, dA, 3 * (ac + 1), dB, 3 * bc, dC, 3 * (N + 1), 2, 3,
                ((ar + 2) * 3 * (ac + 1), ac + 1), (0, bc), (M * 3 * (N + 1), N + 1))
    assert native.last_plan() == [(tile, 1, M)], native.last_plan()
    C = down(native, dC, (2, M, 3, N + 1))
    assert np.all(C[..., N] == 7.0)
    for o in range(2):
        for i in range(3):
            a, b = A[o, :ar, i, :ac], B[:, i]
            assert _near_the_bottom(C[o, :, i, :N], a.T if ta else a, b.T if tb else b), (o, i)


@pytest.mark.parametrize("K", [96, 768, 4096])
def test_no_less_accurate_than_the_fp32_instruction(native, K):
    """Against the 64 x 64 tile of the fp32 matrix cores on the same operands."""
    announce(f"bf16 split accuracy K={K}")
    g = rng(K)
    A = g.uniform(-1, 1, (256, K)).astype(np.float32)
    B = g.uniform(-1, 1, (K, 256)).astype(np.float32)
    want = A.astype(np.float64) @ B.astype(np.float64)
    err = {t: np.linalg.norm(_run(native, A, B, tile=t) - want) for t in (1, 2, 5)}
    assert err[1] <= err[2] and err[5] <= err[2], err


def test_each_tile_id_names_one_kernel(native):
    """Tile 4 stays the fp32 128 x 64 tile on a C of 1.5 M elements and beyond, tile
    5 the bf16 kernel, and the plan that silgpu_gemm_last_plan reports gives the
    same bits when forced; a K-contiguous operand with rows 2^21 floats apart
    takes the fp32 tiles."""
    announce("bf16 split: tile ids, long rows")
    g = rng(4)
    A = g.normal(0, 1, (2048, 3072)).astype(np.float32)
    B = g.normal(0, 1, (3072, 768)).astype(np.float32)
    C4 = _run(native, A, B, tile=TILE_128x64)
    assert native.last_plan() == [(TILE_128x64, 1, 2048)]
    C5 = _run(native, A, B, tile=TILE_256x128)
    assert native.last_plan() == [(TILE_256x128, 1, 2048)]
    assert not np.array_equal(C4, C5)  # other instructions, other roundings
    _check(C4, A, B)
    dA, dB, dC = up(native, A), up(native, B), empty(native, 2048 * 768)
    native.sgemm(0, 0, 2048, 768, 3072, dA, 3072, 0, dB, 768, 0, dC, 768, 0)
    (tile, splits, rows), = native.last_plan()
    assert rows == 2048
    want = down(native, dC, (2048, 768))
    assert np.array_equal(_run(native, A, B, tile=tile, splits=splits), want)
    M, N, K, ld = 5, 150, 33, 1 << 21
    buf = empty(native, M * ld)
    for m in range(M):
        native.call("silgpu_memcpy_h2d", native.vp(buf.at(4 * m * ld)),
                    A[m, :K].ctypes.data_as(native.C.c_void_p), native.C.c_size_t(4 * K))
    dB, dC = up(native, np.ascontiguousarray(B[:K, :N])), empty(native, M * N)
    for tile in (TILE_128x128, TILE_256x128):
        native.sgemm_tuned(0, 0, M, N, K, buf, ld, 0, dB, N, 0, dC, N, 0, tile=tile, splits=1)
        assert native.last_plan() == [(TILE_128x64, 1, M)]
        _check(down(native, dC, (M, N)), A[:M, :K].copy(), B[:K, :N].copy())


@pytest.mark.parametrize("M,N,K,ta,tb,fp32_splits", [
    (1675, 1882, 4787, 0, 0, 4), (3776, 2496, 4096, 0, 1, 8), (1472, 2560, 2048, 0, 0, 4),
    (2496, 1984, 6784, 1, 0, 16), (768, 3072, 2048, 1, 0, 4), (301, 2510, 2363, 0, 0, 6),
    (2368, 1344, 2560, 0, 0, 4)])
def test_planned_products_are_no_less_accurate(native, M, N, K, ta, tb, fp32_splits):
    """The library's own plan against the fp32 matrix cores with the K splits
    that a plan on fp32 tiles alone has: error over 256 rows of C.  The two
    errors are sums of 256 N independent roundings, so their ratio is known to
    about 2 / sqrt(256 N) < 0.4%."""
    announce(f"planned accuracy {M}x{N}x{K} ta={ta} tb={tb}")
    g = rng(M + K)
    A = g.uniform(-1, 1, (K, M) if ta else (M, K)).astype(np.float32)
    B = g.uniform(-1, 1, (N, K) if tb else (K, N)).astype(np.float32)
    rows = np.sort(g.choice(M, 256, replace=False))
    want = (A[:, rows].T if ta else A[rows]).astype(np.float64) @ (B.T if tb else B).astype(
        np.float64)
    dA, dB, dC = up(native, A), up(native, B), empty(native, M * N)
    lda, ldb = (M if ta else K), (K if tb else N)
    native.sgemm(ta, tb, M, N, K, dA, lda, 0, dB, ldb, 0, dC, N, 0)
    err = np.linalg.norm(down(native, dC, (M, N))[rows] - want)
    native.sgemm_tuned(ta, tb, M, N, K, dA, lda, 0, dB, ldb, 0, dC, N, 0, tile=2,
                       splits=fp32_splits)
    fp32 = np.linalg.norm(down(native, dC, (M, N))[rows] - want)
    assert err <= 1.004 * fp32, (err / fp32, native.last_plan())
