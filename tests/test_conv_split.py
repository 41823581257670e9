"""conv2d on the bf16 matrix cores (C_in a multiple of 16, sizes the library
gives to it), against float64: tile edges, even and odd kernels, non-square
images, images smaller than the kernel, K splits, and padding next to
non-finite pixels.  Bar: the SGEMM bar over the K*K*C_in products."""

import numpy as np
import pytest

from conftest import rng
from gpu_util import announce, down, empty, gemm_tolerance_ok, up

pytestmark = pytest.mark.gpu


def _im2col(x, K):
    N, H, W, C = x.shape
    p = K // 2
    xp = np.zeros((N, H + K, W + K, C), x.dtype)
    xp[:, p:p + H, p:p + W] = x
    return np.concatenate([xp[:, i:i + H, j:j + W].reshape(N * H * W, C)
                           for i in range(K) for j in range(K)], axis=1)


TILE_256x128 = 5


def _run(native, x, w):
    N, H, W, Ci = x.shape
    Co, K = w.shape[:2]
    dx, dw, dy = up(native, x), up(native, w), empty(native, N * H * W * Co)
    native.conv2d(dx, dw, dy, N, H, W, Ci, K, Co)
    assert [p[0] for p in native.last_plan()] == [TILE_256x128], native.last_plan()
    return down(native, dy, (N * H * W, Co))


@pytest.mark.parametrize("N,H,W,Ci,K,Co", [
    (2, 9, 13, 64, 3, 70), (1, 16, 16, 128, 3, 128), (1, 17, 15, 128, 3, 129),
    (3, 5, 7, 64, 5, 1), (2, 8, 33, 80, 2, 100), (1, 2, 3, 160, 5, 40), (1, 40, 40, 48, 4, 130),
    (4, 28, 28, 512, 1, 130), (1, 1, 300, 112, 3, 127), (2, 31, 17, 176, 3, 260)])
def test_conv_edges(native, N, H, W, Ci, K, Co):
    announce(f"conv split {N}x{H}x{W}x{Ci} k{K} -> {Co}")
    g = rng(N + H + W + Ci + K + Co)
    x = g.normal(0, 1, (N, H, W, Ci)).astype(np.float32)
    w = g.normal(0, 1, (Co, K, K, Ci)).astype(np.float32)
    A, B = _im2col(x, K).astype(np.float64), w.reshape(Co, -1).T.astype(np.float64)
    ok, nw, el = gemm_tolerance_ok(_run(native, x, w), A @ B, np.abs(A) @ np.abs(B), K * K * Ci)
    assert ok, (nw, el)


def test_padding_is_zero_beside_non_finite_pixels(native):
    announce("conv split: NaN and inf pixels")
    g = rng(8)
    x = g.normal(0, 1, (1, 20, 20, 64)).astype(np.float32)
    w = g.normal(0, 1, (96, 3, 3, 64)).astype(np.float32)
    x[0, 0, 0, :4] = np.nan          # where the loads of padding point
    x[0, 19, 19, 0] = np.inf
    x[0, 10, 10, 5] = -3.4e38
    y = _run(native, x, w).reshape(20, 20, 96)
    A = _im2col(x, 3).astype(np.float64)
    with np.errstate(invalid="ignore"):
        want = (A @ w.reshape(96, -1).T.astype(np.float64)).reshape(20, 20, 96)
    nan = np.zeros((20, 20), bool)
    nan[:2, :2] = True
    assert np.isnan(y[nan]).all()
    inf = np.zeros((20, 20), bool)
    inf[18:, 18:] = True
    assert np.isinf(y[inf]).all() and np.array_equal(np.sign(y[inf]), np.sign(want[inf]))
    fin = ~(nan | inf)
    fin[9:12, 9:12] = False          # 3.4e38 times a weight over 1 overflows
    bar = 1e-5 * 24 * (np.abs(np.nan_to_num(A, posinf=0)) @ np.abs(w.reshape(96, -1).T))
    assert np.all(np.abs(y - want)[fin] <= bar.reshape(20, 20, 96)[fin])
    big = np.abs(want[9:12, 9:12]) < 3.4e38
    assert np.allclose(y[9:12, 9:12][big], want[9:12, 9:12][big], rtol=1e-5)


@pytest.mark.parametrize("H,W,K", [(20, 20, 3), (9, 33, 5)])
def test_sums_of_elements_that_round_to_zero(native, H, W, K):
    """Pixels under 2^-134 have no bf16 part: alone in the image (a corner
    pixel, one that only padded taps reach) and all over it."""
    announce(f"conv split: subnormal pixels {H}x{W} k{K}")
    g = rng(H + W)
    w = g.uniform(500, 1000, (96, K, K, 64)).astype(np.float32)
    for where in [(0, 0, 0), (0, H - 1, W - 1), (1, 0, W - 1), (1, H - 1, 0), None]:
        x = np.zeros((2, H, W, 64), np.float32)
        if where is None:
            x[:] = g.uniform(2e-41, 4e-41, x.shape)
        else:
            x[where] = 3e-41
        A, B = _im2col(x, K).astype(np.float64), w.reshape(96, -1).T.astype(np.float64)
        n = K * K * 64
        err = np.abs(_run(native, x, w) - A @ B)
        assert np.all(err <= 1e-5 * np.sqrt(n) * (np.abs(A) @ np.abs(B)) + n * 2.0 ** -149), where
