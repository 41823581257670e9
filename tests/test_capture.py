"""Products and convolutions recorded into a HIP graph on the library's stream:
a K split whose planes do not fit the workspace yet runs unsplit there, and a
workspace that a graph uses outlives its growth.  Every replay is compared
with the eager result, with eager work and synchronisations in between."""

import ctypes as C
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

from conftest import rng
from gpu_util import announce, down, empty, up

pytestmark = pytest.mark.gpu


class Graph:
    def __init__(self, native, record):
        self.hip = C.CDLL("libamdhip64.so")
        s = C.c_void_p()
        native.call("silgpu_get_stream", C.byref(s))
        self.stream, g, self.exe = s, C.c_void_p(), C.c_void_p()
        self._ok(self.hip.hipStreamBeginCapture(s, 2))  # relaxed
        record()
        self._ok(self.hip.hipStreamEndCapture(s, C.byref(g)))
        self._ok(self.hip.hipGraphInstantiate(C.byref(self.exe), g, None, None, C.c_size_t(0)))

    def replay(self):
        self._ok(self.hip.hipGraphLaunch(self.exe, self.stream))

    @staticmethod
    def _ok(rc):
        assert rc == 0, rc


def test_replays_match_the_eager_result(native):
    announce("captured products and convolution")
    g = rng(3)
    M, N, K = 700, 600, 2051
    A, B = g.normal(0, 1, (M, K)).astype(np.float32), g.normal(0, 1, (K, N)).astype(np.float32)
    dA, dB, dC = up(native, A), up(native, B), empty(native, M * N)
    x = g.normal(0, 1, (4, 28, 28, 64)).astype(np.float32)
    w = g.normal(0, 0.1, (128, 3, 3, 64)).astype(np.float32)
    dx, dw, dy = up(native, x), up(native, w), empty(native, 4 * 28 * 28 * 128)

    def gemm():
        native.gemm(0, 0, M, N, K, dA, K, dB, N, dC, N)

    def conv():
        native.conv2d(dx, dw, dy, 4, 28, 28, 64, 3, 128)

    conv()
    assert native.last_plan()[0][1] > 1  # a K split, in the workspace by now
    gemm()
    want_c, want_y = down(native, dC, (M, N)), down(native, dy, (4 * 28 * 28, 128))
    assert native.last_plan()[0][1] > 1  # a K split, in the workspace by now
    graph = Graph(native, lambda: (gemm(), conv()))
    big = [empty(native, 2048 * 8192) for _ in range(2)] + [empty(native, 2048 * 2048)]
    for rep in range(3):
        native.call("silgpu_fill_u32", native.vp(dC), 0x7fc00000, M * N)
        native.call("silgpu_fill_u32", native.vp(dy), 0x7fc00000, 4 * 28 * 28 * 128)
        graph.replay()
        assert np.array_equal(down(native, dC, (M, N)), want_c)
        assert np.array_equal(down(native, dy, (4 * 28 * 28, 128)), want_y)
        # eager work that grows the workspace between the replays
        native.sgemm_tuned(0, 0, 2048, 2048, 8192, big[0], 8192, 0, big[1], 2048, 0, big[2],
                           2048, 0, tile=5, splits=8 * (rep + 1))
        native.sync()


def _in_a_new_process(name):
    """Runs this file's function `name` where no workspace has been allocated yet."""
    here = Path(__file__).resolve().parent
    code = (f"import sys; sys.path[:0] = [{str(here)!r}, {str(here.parent)!r}]\n"
            f"import test_capture as t\nfrom silarray_amd import _native as native\n"
            f"native.init()\nt.{name}(native)\nprint('done')")
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=110)
    assert r.returncode == 0 and r.stdout.endswith("done\n"), r.stdout + r.stderr


def _float64(native, dA, dB, M, N, K):
    A, B = down(native, dA, (M, K)).astype(np.float64), down(native, dB, (K, N)).astype(np.float64)
    return A @ B, 1e-5 * np.sqrt(K) * (np.abs(A) @ np.abs(B))


def splits_without_room(native):
    """Products and a convolution whose plans split K, recorded with no workspace:
    the plans that need none are recorded, and their replays are right."""
    g = rng(4)
    M, N, K = 700, 600, 2051
    dA = up(native, g.normal(0, 1, (M, K)).astype(np.float32))
    dB = up(native, g.normal(0, 1, (K, N)).astype(np.float32))
    x = g.normal(0, 1, (4, 28, 28, 64)).astype(np.float32)
    w = g.normal(0, 0.1, (128, 1, 1, 64)).astype(np.float32)
    w3 = np.zeros((128, 3, 3, 64), np.float32)
    w3[:, 1, 1] = w[:, 0, 0]  # a 1 x 1 kernel in the middle of a 3 x 3 one
    dx, dw = up(native, x), up(native, w3)
    dC, dF, dy = empty(native, M * N), empty(native, M * N), empty(native, 4 * 28 * 28 * 128)
    plans = {}

    def forced(tile, dst):
        native.sgemm_tuned(0, 0, M, N, K, dA, K, 0, dB, N, 0, dst, N, 0, tile=tile, splits=8)

    def record():
        native.gemm(0, 0, M, N, K, dA, K, dB, N, dC, N)
        plans["gemm"] = native.last_plan()
        forced(5, dF)
        plans["forced"] = native.last_plan()
        native.conv2d(dx, dw, dy, 4, 28, 28, 64, 3, 128)
        plans["conv"] = native.last_plan()

    graph = Graph(native, record)
    assert all(p[1] == 1 for plan in plans.values() for p in plan), plans
    assert plans["forced"] == [(5, 1, M)], plans
    # without K splits the fp32 tiles are ahead of the bf16 kernel's 13 workgroups
    assert plans["conv"] == [(4, 1, 4 * 28 * 28)], plans
    want, bar = _float64(native, dA, dB, M, N, K)
    X, W = x.reshape(-1, 64).astype(np.float64), w.reshape(128, 64).T.astype(np.float64)
    for rep in range(3):
        for buf, n in ((dC, M * N), (dF, M * N), (dy, 4 * 28 * 28 * 128)):
            native.call("silgpu_fill_u32", native.vp(buf), 0x7fc00000, n)
        graph.replay()
        for buf in (dC, dF):
            assert np.all(np.abs(down(native, buf, (M, N)) - want) <= bar)
        y = down(native, dy, (4 * 28 * 28, 128))
        assert np.all(np.abs(y - X @ W) <= 1e-5 * 8 * (np.abs(X) @ np.abs(W)))
        if rep == 0:  # the same calls outside a capture: K splits, and a workspace
            record()
            assert plans["gemm"][0][1] > 1 and plans["forced"] == [(5, 8, M)], plans
            assert plans["conv"][0][1] > 1, plans
            native.sync()


def test_splits_that_do_not_fit_yet_run_without(native):
    announce("capture without a workspace")
    _in_a_new_process("splits_without_room")


def growth_between_captures(native):
    """Ten captures, each with the workspace as it is, which then has to grow by
    64 MiB: every graph keeps its block and replays into it, and all blocks together
    take no more than four times the largest request (2 GiB of 2.5; one more block of
    each size would be 3.4 GiB)."""
    hip = C.CDLL("libamdhip64.so")

    def free():
        a, b = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(a), C.byref(b)) == 0
        return a.value

    g = rng(6)
    M, N, K = 2048, 2048, 1280
    dA = up(native, g.normal(0, 1, (M, K)).astype(np.float32))
    dB = up(native, g.normal(0, 1, (K, N)).astype(np.float32))
    dC = [empty(native, M * N) for _ in range(11)]

    def product(i, splits):
        native.sgemm_tuned(0, 0, M, N, K, dA, K, 0, dB, N, 0, dC[i], N, 0, tile=5, splits=splits)
        if splits == 4:
            assert native.last_plan() == [(5, 4, M)]

    product(10, 1)  # code objects loaded
    native.sync()
    before, graphs = free(), []
    for i in range(10):
        product(10, 4 * i + 4)  # 4 (i + 1) planes of 16 MiB
        graphs.append(Graph(native, lambda: product(i, 4)))
    native.sync()
    assert before - free() <= 4 * 640 << 20, (before - free()) >> 20
    product(10, 4)
    want = down(native, dC[10], (M, N))
    for rep in range(3):
        for i, graph in enumerate(graphs):
            native.call("silgpu_fill_u32", native.vp(dC[i]), 0x7fc00000, M * N)
            graph.replay()
        product(10, 40)
        for i in range(10):
            assert np.array_equal(down(native, dC[i], (M, N)), want), (rep, i)


def test_workspace_growth_between_captures_is_bounded(native):
    announce("workspace growth between captures")
    _in_a_new_process("growth_between_captures")
