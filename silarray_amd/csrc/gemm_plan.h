// The choice of a matrix product's tile and K splits, from its sizes alone: host
// code without a GPU header, so that a test can walk it on the CPU.
#pragma once

#include <cmath>
#include <cstdint>
#include <initializer_list>

#include "intmath.h"

namespace silgpu {
namespace {

// Tile configurations.  128x128 and 256x256 run on the bf16 kernel
// (gemm_split.h), as 128 x 128 and 256 x 128 workgroups; each id names one kernel.
enum tile_cfg {
  TILE_AUTO = 0,
  TILE_128x128 = 1,
  TILE_64x64 = 2,
  TILE_32x128 = 3,
  TILE_128x64 = 4,
  TILE_256x256 = 5,
  // M <= 32 (batch 1, A not transposed): sgemm_skinny_k with 32Q columns per
  // workgroup; the automatic choice is TILE_SKINNY (Q = 1) or, for wide and
  // deep products, TILE_SKINNY_Q2.
  TILE_SKINNY = 6,
  TILE_SKINNY_Q2 = 7,
  TILE_SKINNY_Q4 = 8,
  // 64 x 64 tiles with the K range halved between two wave groups of each
  // workgroup (launch_k2), or quartered between four (launch_k4).
  TILE_64x64_K2 = 9,
  TILE_64x64_K4 = 10
};

struct plan {
  int tile;
  int splits;
  // Batch 1: the last tail_rows rows of C run as a second product with
  // tail_splits K splits (the main product then fills whole rounds of CUs).
  int tail_rows = 0;
  int tail_splits = 1;
};

// The 32x128 tile for M <= 32, K split for about 256 workgroups.
inline plan small_m_tiles(int64_t M, int64_t N, int64_t K, int64_t batch) {
  plan p{TILE_32x128, 1};
  if (batch == 1) {
    int64_t sp = cdiv(256, cdiv(M, 32) * cdiv(N, 128));
    if (sp > K / 256) sp = K / 256;
    if (sp > 64) sp = 64;
    if (sp > 1) p.splits = static_cast<int>(sp);
  }
  return p;
}

// K splits for the small-M kernel: about one workgroup per CU (measured best
// on MI355X for M <= 32 at N, K in 768..4096), each K range at least 128
// deep.
inline int skinny_splits(int64_t M, int64_t N, int64_t K, int Q) {
  (void)M;
  int64_t sp = 256 / cdiv(N, 32 * Q);
  if (sp > K / 128) sp = K / 128;
  if (sp > 65535) sp = 65535;
  return sp < 1 ? 1 : static_cast<int>(sp);
}

// Mean length of the K ranges that a plan adds up in one accumulator.
inline double k_range(const plan &p, int64_t M, int64_t K) {
  const int groups = p.tile == TILE_64x64_K2 ? 2 : p.tile == TILE_64x64_K4 ? 4 : 1;
  const double main = double(K) / double((p.splits > 1 ? p.splits : 1) * groups);
  if (p.tail_rows == 0) return main;
  return (main * double(M - p.tail_rows) +
          double(K) / double(p.tail_splits > 1 ? p.tail_splits : 1) * double(p.tail_rows)) /
         double(M);
}

// A sum's rounding error grows with the square root of its K range.  The bf16
// kernel's is r(range) times the fp32 kernels' over the same range, so where they
// add up `fp32_range` it may add up a range with r^2 range under that.  r^2 on
// MI355X, 512 x 512, uniform[-1, 1] (within 0.02 on normal values, lower on
// positive ones), and between the measured ranges by the logarithm:
inline bool split_range_ok(double range, double fp32_range) {
  constexpr struct {
    double range, r2;
  } t[] = {{256, 0.690},   {768, 0.728},   {2048, 0.748}, {8192, 0.801},
           {16384, 0.833}, {32768, 0.885}, {65536, 0.967}};
  if (range > 65536) return false;
  if (range <= t[0].range) return range * t[0].r2 <= fp32_range;
  int i = 1;
  while (range > t[i].range) ++i;
  const double f = std::log(range / t[i - 1].range) / std::log(t[i].range / t[i - 1].range);
  return range * (t[i - 1].r2 + f * (t[i].r2 - t[i - 1].r2)) <= fp32_range;
}

// K splits that the fp32 plan would not have needed take at most this much for
// their partial planes.
constexpr double kMaxPlaneBytes = 0x1p30;
inline double plane_bytes(int sp, int64_t M, int64_t N) {
  return sp > 1 ? double(sp) * double(M) * double(N) * 4.0 : 0.0;
}

// The K splits that fit `room` bytes of scratch, at most sp.
inline int splits_within(int sp, int64_t M, int64_t N, double room) {
  if (plane_bytes(sp, M, N) <= room) return sp;
  const double fit = room / plane_bytes(2, M, N) * 2.0;
  return fit >= 2.0 ? static_cast<int>(fit) : 1;
}
inline bool plan_fits(const plan &p, int64_t M, int64_t N, double room) {
  return plane_bytes(p.splits, M, N) <= room && plane_bytes(p.tail_splits, p.tail_rows, N) <= room;
}

inline double plane_sum_time(int sp, int64_t rows, int64_t cols) {
  return 0.8e-6 + double(sp + 1) * double(rows) * double(cols) * 4.0 / 5.0e12 + 0.05e-6 * sp;
}

// Shape heuristic: a cost model of each candidate tile and K
// split -- workgroup rounds per CU, the tile's sustained MFMA efficiency,
// occupancy, a K-loop ramp, a per-K-step latency floor and the split-K
// partial pass -- calibrated on MI355X tile x split sweeps (squares up to
// 4096^3, linear_sigmoid 256x4096x4096, transformer projections, small and
// ragged products).  M <= 32 with batch 1 goes to the small-M kernel.
//
// fp32_plan: the plan on the fp32 tiles and its predicted time (0 where a rule
// and not the model chose it).  With max_range = 0 the 256x256 and 128x128 fp32
// tiles are candidates too.  Nothing runs them (the bf16 kernel is faster), but
// a product's accuracy is measured against the plan they would have had: an
// entry point owes no longer K ranges than that.  max_range > 0: the tiles that
// run, K ranges up to max_range, partial planes within `room`; a time of kNoPlan
// if there is none.
constexpr double kNoPlan = 1e30;
struct fp32_pick {
  plan p;
  double time;
};

inline fp32_pick fp32_plan(int64_t M, int64_t N, int64_t K, int64_t batch, bool dtl_ok,
                           double max_range, double room = INFINITY) {
  auto tiles = [&](int bm, int bn) { return cdiv(M, bm) * cdiv(N, bn) * batch; };
  auto allowed = [&](const plan &p) {
    return max_range <= 0.0 ||
           (k_range(p, M, K) <= max_range * 1.001 && plan_fits(p, M, N, room));
  };
  // Predicted time of each (tile, K split): every CU runs ceil(WG / 256)
  // workgroups, min(that, occupancy) of them at once; a SIMD holding a
  // single wavefront reaches kSingleWave of the rate it reaches with two or
  // more.  eff is the fraction of fp32 MFMA peak each tile reaches at large
  // K -- for the LDS-direct kernel where the operands allow it, else for the
  // register-staged one -- and the K loop reaches half its rate at klen =
  // kK0.  A workgroup also takes at least lat per 16-deep K step (one global
  // -> LDS round trip that nothing else hides when a CU holds few
  // workgroups: the floor of small products).  Split-K adds the partial-sum
  // pass: a launch, (splits + 1) M x N fp32 passes and a per-plane latency.
  // A 128x64 launch of at most one workgroup per CU runs 8 waves (two per
  // SIMD, launch_tb), at kEff8 of the 4-wave tile's rate.  Fitted on MI355X
  // to full tile x split sweeps (splits 1, 2, 3, 4, 6, 8, 16) of 46 shapes
  // from 64 x 768 x 2048 to 2048 x 2304 x 768, aligned and ragged, with the
  // picks of the large squares (2048^3 .. 8192^3) held: the plan costs 1.5%
  // more than the best fixed plan (geometric mean; before the 3- and 6-way
  // splits and the 8-wave tile were modelled, 2.1%).  Against the previous
  // plans, 51 shapes: 0.57% faster in the geometric mean, 2048x768x768
  // 30.0 -> 28.3 us, 768^3 20.0 -> 17.6, 512x1024x4096 41.2 -> 39.6, and
  // one shape slower, 100x5000x5000 70.3 -> 74.7.
  struct cand {
    int tile, bm, bn, bk, waves, occupancy;
    double eff, lat;
  };
  // The 128x64 tile runs the LDS-direct kernel when the operands allow it
  // (fitted 0.82 of peak at three workgroups per CU on the 2048-row
  // transformer and square shapes), the register-staged one otherwise.
  const bool dtl128 = dtl_ok && M % 128 == 0 && N % 128 == 0;
  const bool dtl64 = dtl_ok && M % 128 == 0 && N % 64 == 0;
  const cand cands[] = {{TILE_256x256, 256, 256, 16, 8, 1, 0.87, 1.15e-6},
                        {TILE_128x128, 128, 128, 16, 4, 3, dtl128 ? 0.81 : 0.70, 1.25e-6},
                        {TILE_128x64, 128, 64, 16, 4, dtl64 ? 3 : 5, dtl64 ? 0.86 : 0.71, 0.57e-6},
                        {TILE_64x64, 64, 64, 16, 4, 8, 0.64, 0.442e-6}};
  constexpr double kK0 = 48.0, kSingleWave = 0.8755, kLaunch = 4.0e-6, kEff8 = 0.909;
  const double rate_cu = 157.3e12 / 256.0;
  auto round_time = [&](const cand &cd, int64_t nwg, double klen) {
    const int64_t per_cu = cdiv(nwg, 256);
    const int64_t conc = per_cu < cd.occupancy ? per_cu : cd.occupancy;
    const bool w8 = cd.tile == TILE_128x64 && dtl64 && K % 32 == 0 && nwg <= 256;
    const double per_simd = double(conc) * (w8 ? 8 : cd.waves) / 4.0;
    const double f = per_simd >= 2.0 ? 1.0 : per_simd >= 1.0 ? kSingleWave
                                                              : kSingleWave * per_simd;
    const double t = double(per_cu) * 2.0 * cd.bm * cd.bn * klen /
                     (rate_cu * cd.eff * (w8 ? kEff8 : 1.0) * f * (klen / (klen + kK0)));
    const double floor_t = double(cdiv(per_cu, conc)) * (klen / 16.0) * cd.lat;
    return t > floor_t ? t : floor_t;
  };
  plan best{TILE_128x64, 1};
  double best_t = kNoPlan;
  for (const cand &cd : cands) {
    const bool wide = cd.tile == TILE_256x256 || cd.tile == TILE_128x128;
    if (wide && max_range > 0.0) continue;
    for (int sp : {1, 2, 3, 4, 6, 8, 16}) {
      if (sp > 1 && (batch != 1 || K / sp < 64)) continue;
      // (3- and 6-way splits of the larger tiles won nowhere in the sweeps.)
      if ((sp == 3 || sp == 6) && wide) continue;
      if (!allowed(plan{cd.tile, sp})) continue;
      if (max_range > 0.0 && double(sp) * max_range > double(K) * 1.001 &&
          plane_bytes(sp, M, N) > kMaxPlaneBytes)
        continue;  // more K splits than accuracy asks for
      const int64_t wg = tiles(cd.bm, cd.bn) * sp;
      const double klen = double(cdiv(cdiv(K, sp), cd.bk) * cd.bk);
      double t = round_time(cd, wg, klen);
      if (sp > 1) t += plane_sum_time(sp, M, N);
      if (t < best_t * 0.999) {
        best_t = t;
        best = plan{cd.tile, sp};
      }
    }
  }
  // Peeling a thin last round: when the tiles of an unsplit product fill
  // whole rounds of the 256 CUs plus part of another, the tile rows past
  // the last whole round can run as a second product split along K, so
  // the first launch has no partly filled round.  Same per-round model,
  // plus one launch for the second product.
  if (batch == 1) {
    for (const cand &cd : cands) {
      if (max_range > 0.0 && (cd.tile == TILE_256x256 || cd.tile == TILE_128x128)) continue;
      const int64_t tm = cdiv(M, cd.bm), tn = cdiv(N, cd.bn), wg = tm * tn;
      if (wg <= 256 || wg % 256 == 0) continue;
      const int64_t rows_main = (wg / 256) * 256 / tn;
      if (rows_main < 1 || rows_main >= tm) continue;
      const double t_main = round_time(cd, rows_main * tn, double(cdiv(K, cd.bk) * cd.bk));
      const int64_t mt = M - rows_main * cd.bm;
      for (int sp : {1, 2, 3, 4, 6, 8}) {
        if (sp > 1 && K / sp < 128) continue;
        const double klen = double(cdiv(cdiv(K, sp), cd.bk) * cd.bk);
        double t = t_main + round_time(cd, cdiv(mt, cd.bm) * tn * sp, klen) + kLaunch;
        if (sp > 1) t += plane_sum_time(sp, mt, N);
        const plan pl{cd.tile, 1, static_cast<int>(mt), sp};
        if (t < best_t * 0.97 && allowed(pl)) {
          best_t = t;
          best = pl;
        }
      }
    }
  }
  // Where the pick adds K splits in a second launch and 64 x 64 tiles times
  // at most 8 K splits fill 7/8 or more of the CUs in one round, the 64 x 64
  // tile with the K range halved inside each workgroup (TILE_64x64_K2)
  // needs fewer splits, or none, for the same fill.  A rule rather than a
  // candidate of the model: the model's times of the split plans miss by
  // -5..+5 us on these shapes, while this tile's time is a steady ~4 us
  // launch and ramp plus its MFMA time.  MI355X, us, previous pick ->
  // TILE_64x64_K2: 1024^3 24.1 -> 20.7 (2 splits -> none), 256x4096x4096
  // 70.1 -> 67.2, 512x1024x1024 18.3 -> 16.0, 256x2048x512 14.3 -> 12.2,
  // 256x1024x4096 23.9 -> 22.7, 128x2048x768 12.6 -> 11.0, 512^3 10.8 ->
  // 10.0; with 192 tiles (1024x768x2048) it lost, 34.2 -> 36.0.
  if (batch == 1 && dtl_ok && best.splits > 1 && best.tail_rows == 0 && M % 64 == 0 &&
      N % 64 == 0 && K % 64 == 0) {
    const int64_t t64 = (M / 64) * (N / 64);
    int64_t sp = t64 > 0 ? 256 / t64 : 0;
    if (sp > 8) sp = 8;
    while (sp > 1 && K / sp < 128) --sp;
    // Unsplit with K >= 3072: four wave groups (four waves per SIMD) of at
    // least 768 each beat two (256x4096x4096 67.4 -> 65.2 us, 1024x1024x3072
    // 51.7 -> 50.8); with shorter groups the two-group tile wins (1024^3
    // 20.9 against 21.5).
    if (sp == 1 && t64 >= 224 && K >= 3072 && K % 128 == 0 &&
        allowed(plan{TILE_64x64_K4, 1}))
      return fp32_pick{plan{TILE_64x64_K4, 1}, 0.0};
    const plan k2{TILE_64x64_K2, static_cast<int>(sp)};
    if (sp >= 1 && t64 * sp >= 224 && allowed(k2)) return fp32_pick{k2, 0.0};
  }
  // Batched products never split K across workgroups; where their 64 x 64
  // tiles fill at most one round of the CUs, the K groups are the only K
  // parallelism there is.  MI355X, us, previous pick -> K groups: 8 x
  // 256x256x4096 120.8 -> 65.7 (four groups), 4 x 512x512x2048 63.3 -> 36.5,
  // 16 x 128x128x1024 33.0 -> 20.4, 48 x 64x64x512 18.5 -> 12.4, 64 x
  // 64x64x256 11.2 -> 8.9; with 512 tiles (8 x 512x512x512) two groups lost,
  // 21.4 -> 23.0.
  if (batch > 1 && dtl_ok && M % 64 == 0 && N % 64 == 0 && K % 64 == 0 &&
      (M / 64) * (N / 64) * batch <= 256)
    return fp32_pick{plan{K >= 3072 && K % 128 == 0 ? TILE_64x64_K4 : TILE_64x64_K2, 1}, 0.0};
  // A batched pick of unsplit 128 x 64 tiles that leaves its last round at
  // most half full (batched products cannot peel it into a split second
  // launch) runs faster as twice as many 64 x 64 tiles on two K groups:
  // MI355X, us, 288 to 640 tiles of 128 x 64: 3 x 1024^3 66.8 -> 55.6,
  // 12 x 512x512x1024 67.3 -> 56.9, 5 x 512x1024x2048 126.6 -> 101.1,
  // 9 x 512x512x2048 126.5 -> 101.2, 10 x 512x1024x1024 96.0 -> 90.1 (11 of
  // 11 shapes); with a fuller last round (448 tiles) 67.1 against 72.2, and
  // with whole rounds or one partial one it lost 2-8%.
  if (batch > 1 && dtl_ok && best.tile == TILE_128x64 && best.splits == 1 && M % 128 == 0 &&
      N % 64 == 0 && K % 64 == 0) {
    const int64_t t = (M / 128) * (N / 64) * batch;
    if (t > 256 && t < 768 && t % 256 != 0 && t % 256 <= 128)
      return fp32_pick{plan{TILE_64x64_K2, 1}, 0.0};
  }
  return fp32_pick{best, best_t};
}

// room: bytes of scratch for partial planes (the small-M plans leave theirs to the
// launch).
inline plan choose_plan(int64_t M, int64_t N, int64_t K, int64_t batch, bool dtl_ok, bool vec,
                        double room = INFINITY) {
  auto tiles = [&](int bm, int bn) { return cdiv(M, bm) * cdiv(N, bn) * batch; };
  // M <= 32: the small-M kernel (splits chosen at launch), or where it does
  // not apply (batched, A transposed) the 32x128 tile.  Where 32-column
  // groups would each walk 2048 or more rows of B in 128-byte pieces (wide N
  // and deep K), 64-column groups with twice the K splits read 256-byte
  // pieces: 19.8 -> 17.9 us at 8 x 4096 x 4096 on MI355X; at N 768..3072
  // the 32-column groups measured ahead, so the wider groups need N > 3072.
  if (M <= 32 && batch == 1)
    return plan{N > 3072 && K / skinny_splits(M, N, K, 1) >= 2048 ? TILE_SKINNY_Q2 : TILE_SKINNY,
                0};
  if (M <= 32) return small_m_tiles(M, N, K, batch);
  // Batched products with a short K loop (attention's Q K^T at head dim 64)
  // are bound by storing C, which the many small tiles overlap with other
  // tiles' K loops: 64x64 measured 25% faster than 128x128 at
  // 48 x 512x512x64 on MI355X.
  if (batch > 1 && K <= 128 && M >= 64 && N >= 64) return plan{TILE_64x64, 1};
  // The best fp32 plan, with the K splits of it that fit, and where it does not run
  // so, the best one that adds up no longer K ranges on the tiles that do.
  fp32_pick ref = fp32_plan(M, N, K, batch, dtl_ok, 0.0);
  const bool wide_ref = ref.p.tile == TILE_256x256 || ref.p.tile == TILE_128x128;
  const bool fits = plan_fits(ref.p, M, N, room);
  ref.p.splits = splits_within(ref.p.splits, M, N, room);
  ref.p.tail_splits = splits_within(ref.p.tail_splits, ref.p.tail_rows, N, room);
  const double range = k_range(ref.p, M, K);
  fp32_pick pick = ref;
  int min_splits = (2 * ref.p.splits + 2) / 3;
  if (wide_ref || !fits) {
    pick = fp32_plan(M, N, K, batch, dtl_ok, range, room);
    // (5 and 7 splits, say, which no candidate has.)
    if (pick.time == kNoPlan) pick.p = plan{wide_ref ? TILE_128x64 : ref.p.tile, ref.p.splits};
  }
  // On the bf16 tiles also no fewer than two thirds of the K splits that suit
  // the tiles that run best.
  if (wide_ref)
    min_splits =
        (2 * splits_within(fp32_plan(M, N, K, batch, dtl_ok, INFINITY).p.splits, M, N, room) + 2) / 3;
  if (pick.time == 0.0) return pick.p;  // by rule
  // The bf16 kernel's tiles (gemm_split.h), one workgroup per CU: `launch`
  // once, per round of workgroups `fixed` for the first loads and the stores
  // and per K tile c0 with an idle chip around it, c1 more with every CU busy;
  // a K range that ends inside a K tile runs its last three masked.  Fitted on
  // MI355X to K sweeps (32 .. 2048) of 32 to 512 workgroups.
  struct wide_cand {
    int tile, bm, bn, bk;
    double c0, c1, fixed, launch;
  };
  const wide_cand wides[] = {{TILE_256x256, 256, 128, 16, 0.92e-6, 0.28e-6, 5.5e-6, 5.0e-6},
                             {TILE_128x128, 128, 128, 32, 1.13e-6, 0.27e-6, 3.5e-6, 4.0e-6}};
  // The pick by time; where it sums too long a range, the pick among those that
  // do not, with 5 and 16 splits as well.
  for (const bool exact : {false, true}) {
    // Rows that are not 16-byte aligned cost the register-staged tiles scalar
    // loads, which the model leaves out, and the bf16 kernel nothing.
    double to_beat = pick.time * (vec ? 0.90 : 1.15);
    plan best = pick.p;
    bool wide = false;
    for (const wide_cand &w : wides) {
      for (int sp : {1, 2, 3, 4, 5, 6, 8, 12, 16}) {
        if (batch != 1 ? sp > 1 || K < 320 : sp > 1 && K / sp < 128) continue;
        if (!exact && (sp == 5 || sp == 16)) continue;
        if (sp < min_splits || (exact && !split_range_ok(double(K) / sp, range))) continue;
        if (plane_bytes(sp, M, N) > (sp > ref.p.splits ? std::fmin(room, kMaxPlaneBytes) : room))
          continue;
        const int64_t wg = tiles(w.bm, w.bn) * sp;
        const double stages = double(cdiv(cdiv(K, sp), w.bk)) + (K % w.bk ? 1.5 : 0.0);
        const double fill = wg < 256 ? double(wg) / 256.0 : 1.0;
        double t = w.launch +
                   double(cdiv(wg, 256)) * (w.fixed + stages * (w.c0 + w.c1 * fill));
        if (sp > 1) t += plane_sum_time(sp, M, N);
        if (t < to_beat) {
          to_beat = t;
          wide = true;
          best = plan{w.tile, sp};
        }
      }
    }
    if (!wide || exact || split_range_ok(double(K) / best.splits, range)) return best;
  }
  return pick.p;
}

// A convolution's plan: M output pixels by C_out channels, K = Kd products of which
// C_in belong to one tap, as a plan of that M x C_out product.  vec: C_in a
// multiple of 4, operands 16-byte aligned; bf16_ok: sizes that the bf16 kernel's
// gather takes; room: bytes of scratch for partial planes.
//
// The fp32 plan: where nothing is left over, 128 x 64 tiles of the LDS-direct
// kernel, three workgroups to a CU.  Between one and two tiles per CU (two on some
// CUs, one on others) the K range is split in two, so the pieces fill three rounds.
// When the pieces fill whole rounds of all CUs plus a thin last round, the tile rows
// of that last round run as a second launch split further along K (one piece per CU
// at most) with its own split sum, instead of a round of a few workgroups at full
// depth.
// (Measured: 88.5 -> 85.2 us at 16x28x28x128 -> 256, K = 1152; with K = 576 the
// halves are too short and the split sum costs more than the balance gains, 48.7 ->
// 56.6 us at 8x56x56x64 -> 128.)
inline plan conv_fp32_plan(int64_t M, int64_t C_in, int64_t C_out, int64_t Kd, int64_t cus,
                           bool vec, double room) {
  if (!vec || C_in % 16 != 0 || M % 128 != 0 || C_out % 64 != 0)
    return plan{C_out <= 32 ? TILE_64x64 : TILE_128x64, 1};
  const int BK = C_in % 32 == 0 ? 32 : 16;
  const int64_t tiles_n = C_out / 64, tiles_m = M / 128, tiles = tiles_m * tiles_n;
  const int64_t slots = cus * 3, kt = Kd / BK;
  const int gs = tiles > cus && 2 * tiles > slots && 4 * (2 * tiles) <= 5 * slots &&
                         kt % 2 == 0 && Kd >= 1024
                     ? 2 : 1;
  const int64_t pieces = tiles * gs, rem = pieces % slots;
  int64_t tail = 0;
  int splits = 1;
  if (pieces > slots && rem > 0 && rem * 4 <= slots) {
    const int64_t rem_rows = cdiv(rem, tiles_n * gs);
    tail = rem_rows * 128;
    for (int64_t sp = 2; sp <= kt; ++sp)
      if (kt % sp == 0 && rem_rows * tiles_n * sp <= cus) splits = int(sp);
  }
  // (The kernel wants whole K tiles in every split: all of them or none.)
  plan p{TILE_128x64, gs, static_cast<int>(tail), splits};
  if (plane_bytes(gs, M - tail, C_out) > room) p.splits = 1;
  if (plane_bytes(splits, tail, C_out) > room) p.tail_splits = 1;
  return p;
}

// The bf16 kernel against the fp32 ones, as choose_plan weighs them: its 256 x 128
// tiles, and K splits, in rounds of the CUs (a K tile costs a sixth more than a
// product's for the gather) against 92 TFLOP/s on full 128 x 64 tiles and 55 on the
// register-staged ones, on 3 and 4 workgroups per CU, after 6 us of launch and first
// loads; of those that sum no longer K ranges, for their error, than the fp32 plan.
inline plan conv_plan(int64_t M, int64_t C_in, int64_t C_out, int64_t Kd, int64_t cu_count,
                      bool vec, bool bf16_ok, double room) {
  plan best = conv_fp32_plan(M, C_in, C_out, Kd, cu_count, vec, room);
  if (!bf16_ok) return best;
  const double range = (double(Kd) / best.splits * double(M - best.tail_rows) +
                        double(Kd) / best.tail_splits * double(best.tail_rows)) / double(M);
  const bool full_tiles = M % 128 == 0 && C_out % 64 == 0;
  const double cus = double(cu_count);
  const double tiles = double(cdiv(M, 128) * cdiv(C_out, 64));
  const double busy = tiles < cus ? cus / tiles : 1.0;  // idle CUs at full depth
  double best_t = 0.9 * (6.0e-6 + busy * 2.0 * double(cdiv(M, 128) * 128) *
                                      double(cdiv(C_out, 64) * 64) * double(Kd) /
                                      (full_tiles ? 92e12 : 55e12));
  for (int sp : {1, 2, 3, 4, 6, 8, 12, 16}) {
    if (sp > 1 && Kd / sp < 128) continue;
    if (plane_bytes(sp, M, C_out) > room || !split_range_ok(double(Kd) / sp, range)) continue;
    const double wgs = double(cdiv(M, 256) * cdiv(C_out, 128) * sp);
    const double fill = wgs < cus ? wgs / cus : 1.0;
    double t = 5.0e-6 + std::ceil(wgs / cus) * (5.5e-6 + double(cdiv(Kd, 16 * sp)) *
                                                             (0.92e-6 + 0.28e-6 * fill) * 1.17);
    if (sp > 1) t += 2.5e-6 + double(sp + 1) * double(M) * double(C_out) * 4.0 / 5.0e12;
    if (t < best_t) {
      best_t = t;
      best = plan{TILE_256x256, sp};
    }
  }
  return best;
}

}  // namespace
}  // namespace silgpu
