"""The choice of tile and K splits (silarray_amd/csrc/gemm_plan.h), walked on the
CPU: a small program built from that header prints the plan of each product it
is given, beside the plan of the fp32 tiles that accuracy is measured against.
"""

from __future__ import annotations

import math
import random
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "silarray_amd" / "csrc"
TILE_128x128, TILE_64x64, TILE_128x64, TILE_256x128, TILE_K2, TILE_K4 = 1, 2, 4, 5, 9, 10

DRIVER = r"""
#include <cstdio>
#include "gemm_plan.h"
using namespace silgpu;
int main() {
  long long M, N, K, batch;
  int dtl, vec;
  double room;
  while (std::scanf("%lld %lld %lld %lld %d %d %lf", &M, &N, &K, &batch, &dtl, &vec, &room) == 7) {
    if (batch < 0) {  // a convolution of K taps of -batch channels
      const long long Kd = K * -batch;
      const plan p = conv_plan(M, -batch, N, Kd, 256, vec, vec && batch % 16 == 0, room);
      const plan f = conv_fp32_plan(M, -batch, N, Kd, 256, vec, room);
      std::printf("%d %d %d %d  %d %d %d %d\n", p.tile, p.splits, p.tail_rows, p.tail_splits,
                  f.tile, f.splits, f.tail_rows, f.tail_splits);
      continue;
    }
    const plan p = choose_plan(M, N, K, batch, dtl, vec, room);
    const plan f = fp32_plan(M, N, K, batch, dtl, 0.0).p;
    std::printf("%d %d %d %d  %d %d %d %d\n", p.tile, p.splits, p.tail_rows, p.tail_splits,
                f.tile, f.splits, f.tail_rows, f.tail_splits);
  }
}
"""


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "driver.cpp").write_text(DRIVER)
    cxx = shutil.which("g++") or "/opt/rocm/llvm/bin/clang++"
    subprocess.run([cxx, "-std=c++17", "-O1", f"-I{CSRC}", str(d / "driver.cpp"), "-o",
                    str(d / "driver")], check=True)

    def run(shapes, room=math.inf):
        """[(M, N, K, batch, aligned)] -> [(plan, fp32 plan)]; a batch of -c: a
        convolution, M pixels, K taps of c channels each, N channels out"""
        text = "".join(f"{M} {N} {K} {b} {int(v and K % 16 == 0)} {int(v)} {room}\n"
                       for M, N, K, b, v in shapes)
        out = subprocess.run([str(d / "driver")], input=text, check=True, capture_output=True,
                             text=True).stdout.split("\n")
        rows = [tuple(map(int, line.split())) for line in out if line]
        return [(r[:4], r[4:]) for r in rows]

    return run


def _bf16(p):
    return p[0] in (TILE_128x128, TILE_256x128)


def _squared_error(tile, splits, tail_rows, tail_splits, M, K):
    """Mean square of a sum's rounding error in units of one fp32 product's: its K range."""
    groups = {TILE_K2: 2, TILE_K4: 4}.get(tile, 1)
    main = K / (max(splits, 1) * groups)
    return (main * (M - tail_rows) + K / max(tail_splits, 1) * tail_rows) / M


# Square of the bf16 kernel's error over the fp32 kernels' for the same K range,
# measured (uniform[-1, 1]) at the upper end of each span.
MEASURED = [(256, 0.69), (768, 0.728), (2048, 0.748), (8192, 0.801), (16384, 0.833),
            (32768, 0.885), (65536, 0.967)]


def _worse(p, f, M, K):
    """How much larger the squared error is than the fp32 plan's."""
    e = _squared_error(*p, M, K)
    if _bf16(p):
        k = e
        assert k <= 65536
        hi = next(i for i, (n, _) in enumerate(MEASURED) if k <= n)
        if hi == 0:
            e *= MEASURED[0][1]
        else:  # between two spans, by the logarithm
            (k0, r0), (k1, r1) = MEASURED[hi - 1], MEASURED[hi]
            e *= r0 + (r1 - r0) * math.log(k / k0) / math.log(k1 / k0)
    return e / _squared_error(*f, M, K)


# Products whose fp32 plan is a K split on tiles that are no longer run.
@pytest.mark.parametrize("M,N,K,aligned,fp32_splits", [
    (1675, 1882, 4787, False, 4), (3776, 2496, 4096, True, 8), (1472, 2560, 2048, True, 4),
    (2496, 1984, 6784, True, 16), (768, 3072, 2048, True, 4), (2048, 768, 3072, True, 4)])
def test_k_ranges_of_products_that_were_split(plans, M, N, K, aligned, fp32_splits):
    (p, f), = plans([(M, N, K, 1, aligned)])
    assert f[1:3] == (fp32_splits, 0)
    assert _worse(p, f, M, K) <= 1.0, (p, f)


def _draw(rng, hi=8192):
    def log_int(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))
    M, N, K = (log_int(33, hi) for _ in range(3))
    if rng.random() < 0.5:
        M, N, K = (max(64, v // 64 * 64) for v in (M, N, K))
    return M, N, K


def test_no_plan_adds_up_more_in_a_row_than_the_fp32_tiles_would(plans):
    rng = random.Random(1)
    shapes = []
    for i in range(20000):
        M, N, K = _draw(rng)
        batch = rng.randint(2, 48) if i % 4 == 3 and K > 128 else 1  # short ones: 64x64 always
        shapes.append((M, N, K, batch, K % 4 == 0 and N % 4 == 0))
    got = plans(shapes)
    assert sum(_bf16(p) for p, _ in got) > 3000
    for (M, N, K, b, _), (p, f) in zip(shapes, got):
        assert _worse(p, f, M, K) <= 1.005, ((M, N, K, b), p, f)


def test_large_products_need_no_workspace_that_they_never_needed(plans):
    """Partial planes stay within 1 GiB where the fp32 tiles' plan has none."""
    rng = random.Random(2)
    shapes = [(n, n, n, 1, True) for n in (8192, 16384, 32768, 65536, 70000, 100000)]
    shapes += [(*_draw(rng, 120000), 1, True) for _ in range(5000)]
    got = plans(shapes)
    assert all(p[1] == 1 for p, _ in got[:6])
    for (M, N, K, _, _), (p, f) in zip(shapes, got):
        planes = 4.0 * M * N * p[1] if p[1] > 1 else 0.0
        assert planes <= max(2.0 ** 30, 4.0 * M * N * f[1] if f[1] > 1 else 0.0), (M, N, K, p, f)


@pytest.mark.parametrize("room", [0, 5 << 20, 32 << 20])
def test_plans_within_little_scratch(plans, room):
    """Where partial planes have to fit (a fixed scratch area, a workspace that may
    not grow), they do, and no K range is longer, for its error, than those of the
    fp32 tiles' plan with as many K splits as fit."""
    rng = random.Random(3)
    shapes = [(2048, 2048, 32764, 1, False)] + [(*_draw(rng), 1, True) for _ in range(10000)]
    free, narrow = plans(shapes), plans(shapes, room)

    def planes(p, M, N):
        return [4 * sp * rows * N for sp, rows in ((p[1], M - p[2]), (p[3], p[2])) if sp > 1]

    changed = 0
    for (M, N, K, _, _), (p, f), (p0, _) in zip(shapes, narrow, free):
        assert all(b <= room for b in planes(p, M, N)), (M, N, K, p)
        if all(b <= room for b in planes(p0, M, N)):
            assert p == p0 or planes(f, M, N), (M, N, K, p, p0)
        changed += p != p0
        fit = [max(1, min(f[1], room // (4 * (M - f[2]) * N))), f[2],
               max(1, min(f[3], room // (4 * f[2] * N))) if f[2] else 1]
        assert _worse(p, (f[0], *fit), M, K) <= 1.005, (M, N, K, p, f)
    assert changed > 100


def test_convolutions_add_up_no_longer_ranges(plans):
    rng = random.Random(4)
    shapes = [(16 * 56 * 56, 128, 9, -64, True), (4 * 28 * 28, 128, 9, -64, True)]
    for _ in range(4000):
        n, hw, k = rng.choice([1, 2, 4, 8, 16]), rng.randint(3, 80), rng.choice([1, 2, 3, 5, 7])
        shapes.append((n * hw * hw, rng.choice([16, 40, 64, 96, 128, 200, 256, 512]), k * k,
                       -16 * rng.randint(1, 32), True))
    for room in (math.inf, 0, 4 << 20):
        got = plans(shapes, room)
        assert sum(p[0] == TILE_256x128 for p, _ in got) > 500
        for (M, N, K, b, _), (p, f) in zip(shapes, got):
            assert _worse(p, f, M, K * -b) <= 1.005, ((M, N, K, b), p, f)
            if p[1] > 1:
                assert 4 * p[1] * (M - p[2]) * N <= room
            if p[3] > 1:
                assert 4 * p[3] * p[2] * N <= room
