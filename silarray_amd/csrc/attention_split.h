// Fused attention on the bf16 matrix cores, every float split in three
// (gemm_split.h), for head dim 64 where 128-row workgroups fill a good part of
// the chip (attention_rule).
//
// Workgroup: 8 waves over 128 query rows of one (batch, head): wave w takes
// row group w % 4 (32 rows) and key half w / 4 of every 64-key block.  Both
// products are computed transposed on the 32x32x16 MFMA, as in attention_k:
//   S^T (32 keys x 32 rows) = K Q^T, Q split once into registers, K staged in
//     LDS as fragments of 32 keys x 16 d in lane order (one ds_read_b128 each);
//   O^T (32 d x 32 rows) += V^T P^T: lane (c, s) holds the scores of row c at
//     keys 8 (r / 4) + 4 s + r % 4 in register r, and V's fragments put the
//     same 8 keys of each 16 into k slot s, so P is split where it stands and
//     never leaves registers.
// K and V blocks are split by the whole workgroup on their way into LDS, two
// slots each, one barrier per block.  Each wave runs one block ahead of itself:
// the products of the next block's scores stand between the instructions of
// this block's softmax and the split of P, those of O between the splits of the
// K two blocks and the V one block on, in an order fixed by scheduling
// barriers; the loads of the blocks after those are in flight meanwhile.
//
// What bounds it: the MFMAs of a block take 1.3 us of a SIMD, the vector work
// of its two waves about as much, and a block takes 2.4 us (3.2 us with every
// CU busy, where the chip's power lowers the clock).  With each wave's products,
// softmax, split and products one after the other a block took 3.2 and 4.1 us.
// On the fp32 matrix cores the MFMAs alone took 3.4 us, but there twelve waves
// fit a CU, so small grids stay there.  MI355X, us, fp32 -> this: heads x
// queries x keys 24x1000x1000 70.5 -> 46-47, 48x512x512 39.1 -> 27-30,
// 16x2048x2048 184 -> 111, 48x2048x2048 510 -> 310, 16x1000x1000 (128
// workgroups) 54.7 -> 48.7; 24x512x512 27.6 -> 27.6 and 48x300x300 20.2 ->
// 21.0 stay.  (One after the other, in a run of its own: 76.8 -> 64.9, 40.8 ->
// 37.3, 199 -> 132, 515 -> 366, 56.4 -> 60.9.)  Error against float64 5.1e-7 ->
// 4.1e-7 at 1000 keys.
// Non-finite scores and results so small that parts below bf16's subnormals
// could show are redone by the two waves of the row group on the fp32 matrix
// cores (below).  24x1000x1000, us: 46; a NaN in V, or a zero column beside large
// ones, 48; every row redone 145 (543 with one wave and 4-byte loads; 70 on
// attention_k).
#pragma once

#include "bf16_split.h"

namespace silgpu {
namespace {

constexpr int kSaWaves = 8, kSaThreads = kSaWaves * kWave;
constexpr int kSaRows = 128, kSaKeys = 64;

template <int D>
struct sa_cfg {
  static constexpr int kG = D / 16;                   // 16-deep d groups
  static constexpr int kKs = 2 * kG * 192;            // 16-byte slots: 2 key groups x kG x 3
  static constexpr int kVs = (D / 32) * 4 * 192;      // d blocks x 16-key groups x 3
  static constexpr int kBuf = kKs + kVs;
  static constexpr int UK = kSaKeys * D / 4 / kSaThreads;  // float4 units of K per thread
  static constexpr int WV = 8;                             // keys per unit of V
  static constexpr int UV = kSaKeys * D / WV / kSaThreads;
  static constexpr int kSwz = 128 / D;
  static_assert(D == 64 && UK == 2 && UV == 1 && 2 * kBuf * 16 <= 160 * 1024, "block");
};

// Online softmax step of one row group over a 32-key block: st holds the
// scores of this lane's row at keys key0 + 8 (r / 4) + 4 s + r % 4, and
// leaves as the exponentials; keys at Sk and beyond count as -inf.  A NaN
// score makes the row NaN so that it is redone; there (REDO) a row without a
// finite score so far takes nothing from the block, as in attention_k.
struct sa_row {
  float m = -INFINITY, l = 0.0f;

  // x = score * scale rounded on its own (not folded into the exponent's
  // subtraction: the row maximum must give exactly 2^0, however large).
  __device__ __forceinline__ void scale(floatx16 &st, float scale2, int key0, int s, int Sk) {
#pragma unroll
    for (int r = 0; r < 16; ++r) st[r] *= scale2;
    if (key0 + 32 > Sk) {
      asm volatile("");  // a branch, not 16 selects on every block
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (key0 + 8 * (r / 4) + 4 * s + r % 4 >= Sk) st[r] = -INFINITY;
    }
  }
  // Takes the block's maximum rm in: returns the factor that brings earlier
  // sums to the new maximum, base what exponents are taken against.
  __device__ __forceinline__ float raise(float rm, float &base) {
    const float mn = fmaxf(m, rm);
    const bool none = mn == -INFINITY;  // no finite score in this row yet
    const float alpha = none ? 1.0f : __builtin_amdgcn_exp2f(m - mn);
    base = none ? 0.0f : mn;  // exp2(-inf) = 0
    m = mn;
    return alpha;
  }
  // The whole step, for the redo: a row without a finite score so far takes
  // nothing from the block, as in attention_k.
  __device__ __forceinline__ float step(floatx16 &st, float scale2, int key0, int s, int Sk) {
    scale(st, scale2, key0, s, Sk);
    float rm = -INFINITY, base;
#pragma unroll
    for (int r = 0; r < 16; ++r) rm = fmaxf(rm, st[r]);
    rm = pair_reduce<32>(rm, [](float a, float b) { return fmaxf(a, b); });
    const float alpha = raise(rm, base);
    float rs = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      st[r] = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(st[r] - base);
      rs += st[r];
    }
    l = l * alpha + pair_reduce<32>(rs, [](float a, float b) { return a + b; });
    return alpha;
  }
};

__device__ __forceinline__ floatx16 zero16() {
  floatx16 z;
#pragma unroll
  for (int r = 0; r < 16; ++r) z[r] = 0.0f;
  return z;
}

// Whether a launch takes this kernel: its time (256 workgroups of 128 rows a
// round; a round 9 us and 0.0394 us a key, keys in whole blocks) against
// attention_k's (768 of 32 rows, 0.0125 us a key and 0.0207 more for each
// workgroup that shares a CU), both fitted to 4 .. 96 heads of 33 .. 2048
// queries and keys.  The line is where the measured times cross: attention_k's
// is overestimated by 15% on average.  Rows whose lane offsets exceed 32 bits
// stay with attention_k.
inline bool attention_rule(const attn_args &a, int64_t batch, int64_t D) {
  if (D != 64 || a.Sk < 1 || a.ldk >= (int64_t(1) << 23)) return false;
  const double wgs = double(batch) * double(cdiv(a.Sq, kSaRows)), keys = double(a.Sk);
  const double t_split =
      std::ceil(wgs / 256) * (double(cdiv(a.Sk, kSaKeys) * kSaKeys) * 0.0394 + 9.0) - 2.0;
  const int64_t old = batch * cdiv(a.Sq, 32), rest = old % 768;
  const double t_fp32 = 4.0 + keys * (double(old / 768) * 0.0745 +
                                      (rest ? 0.0125 + 0.0207 * double(cdiv(rest, 256)) : 0.0));
  return t_split < 0.84 * t_fp32;
}

template <int D>
__global__ __launch_bounds__(kSaThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
void attention_split_k(attn_args a) {
  using C = sa_cfg<D>;
  constexpr int NB = D / 32;  // 32-wide blocks of O
  __shared__ uint4 lds[2 * C::kBuf];
  __shared__ float smx[2][kSaWaves], smv[kSaWaves][kWave];
  __shared__ int sbad[4];
  const int t = threadIdx.x, lane = t % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(t / kWave);
  const int c = lane % 32, s = lane / 32;
  const int rg = wave % 4, kh = wave / 4;
  const int64_t zo = blockIdx.y / a.binner, zi = blockIdx.y % a.binner;
  const float *__restrict__ Q = a.Q + zo * a.sq_o + zi * a.sq_i;
  const float *__restrict__ K = a.K + zo * a.sk_o + zi * a.sk_i;
  const float *__restrict__ V = a.V + zo * a.sv_o + zi * a.sv_i;
  float *__restrict__ O = a.O + zo * a.so_o + zi * a.so_i;
  const int Sq = a.Sq, Sk = a.Sk;
  const int row = blockIdx.x * kSaRows + 32 * rg + c;
  const float scale2 = a.scale * 1.4426950408889634f;  // scale * log2(e)
  const float *qrow = Q + int64_t(min(row, Sq - 1)) * a.ldq;
  float mqk = 0.0f, mv = 0.0f;  // largest magnitudes of Q and K, and of V

  // Q^T fragments: d 16 g + 8 s + j of row c.
  bf16x8 qf[C::kG][3];
#pragma unroll
  for (int g = 0; g < C::kG; ++g) {
    const f4u x = *reinterpret_cast<const f4u *>(qrow + 16 * g + 8 * s);
    const f4u y = *reinterpret_cast<const f4u *>(qrow + 16 * g + 8 * s + 4);
    max_abs(mqk, x[0], x[1]);
    max_abs(mqk, x[2], x[3]);
    max_abs(mqk, y[0], y[1]);
    max_abs(mqk, y[2], y[3]);
    uint4 h, m, l;
    split_pair(x[0], x[1], h.x, m.x, l.x);
    split_pair(x[2], x[3], h.y, m.y, l.y);
    split_pair(y[0], y[1], h.z, m.z, l.z);
    split_pair(y[2], y[3], h.w, m.w, l.w);
    qf[g][0] = __builtin_bit_cast(bf16x8, h);
    qf[g][1] = __builtin_bit_cast(bf16x8, m);
    qf[g][2] = __builtin_bit_cast(bf16x8, l);
  }

  // Staging.  K unit: 4 d of one key.  V unit: WV keys of one d, the keys of k
  // slot vs of 16-key group vg in the order P holds them.
  float kr[C::UK][4], vr[C::WV];
  auto vkey = [&](int j) {  // key within the block
    return 16 * (wave / 2) + 4 * (wave % 2) + (j < 4 ? j : j + 4);
  };
  const int nblocks = (Sk + kSaKeys - 1) / kSaKeys;
  // Lane byte offsets within a block (the host keeps 64 rows under 2^32 bytes).
  uint32_t koff[C::UK];
#pragma unroll
  for (int u = 0; u < C::UK; ++u) {
    const int f = t + u * kSaThreads;
    koff[u] = (uint32_t(f / (D / 4)) * uint32_t(a.ldk) + 4u * uint32_t(f % (D / 4))) * 4u;
  }
  auto load_k = [&](int key0) {
    const bool full = key0 + kSaKeys <= Sk;
    const char *kb = reinterpret_cast<const char *>(K + int64_t(key0) * a.ldk);
#pragma unroll
    for (int u = 0; u < C::UK; ++u) {
      const char *p = kb + koff[u];
      if (!full) {  // rows past the last key read the last one
        const int f = t + u * kSaThreads;
        p = reinterpret_cast<const char *>(K + int64_t(min(key0 + f / (D / 4), Sk - 1)) * a.ldk +
                                           4 * (f % (D / 4)));
      }
      const f4u x = *reinterpret_cast<const f4u *>(p);
#pragma unroll
      for (int j = 0; j < 4; ++j) kr[u][j] = x[j];
    }
  };
  auto load_v = [&](int key0) {
    if (key0 + kSaKeys <= Sk) {
      const float *vb = V + int64_t(key0 + vkey(0)) * a.ldv;
#pragma unroll
      for (int j = 0; j < C::WV; ++j) {
        if (j == 4) vb += 4 * a.ldv;  // the second four keys of the slot
        vr[j] = vb[uint32_t(t) % D];
        vb += a.ldv;
      }
    } else {  // past the last key P is 0, and V has to be finite
#pragma unroll
      for (int j = 0; j < C::WV; ++j)
        vr[j] = V[int64_t(min(key0 + vkey(j), Sk - 1)) * a.ldv + t % D];
    }
  };
  auto mask_v = [&](int key0) {
    if (key0 + kSaKeys > Sk) {
      asm volatile("");
#pragma unroll
      for (int j = 0; j < C::WV; ++j) vr[j] = key0 + vkey(j) < Sk ? vr[j] : 0.0f;
    }
  };
  // Splits pair i of the staged registers (0 .. 3 of K, 4 .. 7 of V), and
  // stores a K unit or the V unit when its last pair is done.
  uint32_t ph[C::WV / 2], pm[C::WV / 2], pl[C::WV / 2];
  auto stage_pair = [&](auto ic, uint4 *B) {
    constexpr int i = decltype(ic)::value;
    if constexpr (i < 4) {
      constexpr int u = i / 2, o = i % 2;
      max_abs(mqk, kr[u][2 * o], kr[u][2 * o + 1]);
      split_pair(kr[u][2 * o], kr[u][2 * o + 1], ph[o], pm[o], pl[o]);
      if constexpr (o == 1) {
        const int f = t + u * kSaThreads, key = f / (D / 4), q = f % (D / 4);
        const int g = q / 4, oc = q / 2 % 2;
        uint2 *d = reinterpret_cast<uint2 *>(B + ((key / 32) * C::kG + g) * 192 + oc * 32 +
                                             ((key % 32) ^ (8 * oc) ^ (C::kSwz * g))) + q % 2;
        d[0] = make_uint2(ph[0], ph[1]);
        d[128] = make_uint2(pm[0], pm[1]);
        d[256] = make_uint2(pl[0], pl[1]);
      }
    } else {
      constexpr int o = i - 4;
      max_abs(mv, vr[2 * o], vr[2 * o + 1]);
      split_pair(vr[2 * o], vr[2 * o + 1], ph[o], pm[o], pl[o]);
      if constexpr (o == 3) {
        uint4 *p = B + ((t % D / 32) * 4 + wave / 2) * 192 + (wave % 2) * 32 + t % 32;
        p[0] = make_uint4(ph[0], ph[1], ph[2], ph[3]);
        p[64] = make_uint4(pm[0], pm[1], pm[2], pm[3]);
        p[128] = make_uint4(pl[0], pl[1], pl[2], pl[3]);
      }
    }
  };
  auto sync = [] {
    __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (3 << 14));  // lgkmcnt(0) alone
    asm volatile("s_barrier" ::: "memory");
  };

  constexpr int pa[6] = {2, 1, 0, 1, 0, 0}, pb[6] = {0, 1, 2, 0, 1, 0};  // small products first
  floatx16 acc[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) acc[j] = zero16();
  sa_row sm;
  auto k_frag = [&](const uint4 *B, int g, bf16x8 (&kf)[3]) {
#pragma unroll
    for (int q = 0; q < 3; ++q)
      kf[q] = __builtin_bit_cast(
          bf16x8, B[(kh * C::kG + g) * 192 + q * 64 + s * 32 + (c ^ (8 * s) ^ (C::kSwz * g))]);
  };

  // Block kb: the scores of block kb + 1 (products with MORE) beside the
  // softmax of block kb, then O += V P beside the staging of K of block kb + 2
  // and V of block kb + 1.  st comes in as the raw scores of block kb and
  // leaves as those of the next.
  floatx16 st = zero16();
  auto block = [&](auto more, int kb) {
    constexpr bool MORE = decltype(more)::value;
    uint4 *Kb = lds + ((kb + 1) & 1) * C::kKs, *Kn = lds + (kb & 1) * C::kKs;
    uint4 *Vb = lds + 2 * C::kKs + (kb & 1) * C::kVs;
    uint4 *Vn = lds + 2 * C::kKs + ((kb + 1) & 1) * C::kVs;
    const int key0 = kb * kSaKeys + 32 * kh;
    bf16x8 kf[2][3];
    if constexpr (MORE) {
      k_frag(Kb, 0, kf[0]);
      k_frag(Kb, 1, kf[1]);
    }
    sm.scale(st, scale2, key0, s, Sk);
    floatx16 sn = zero16();
    float rm = -INFINITY, alpha = 1.0f, base = 0.0f, rs = 0.0f;
    uint32_t h[8], m[8], l[8];
    bf16x8 vf[2][NB][3];
    auto v_frag = [&](auto gc, auto ic) {
      constexpr int g = decltype(gc)::value, i = decltype(ic)::value;
      vf[g][i / 3][i % 3] = __builtin_bit_cast(
          bf16x8, Vb[((i / 3) * 4 + 2 * kh + g) * 192 + (i % 3) * 64 + lane]);
    };
    __builtin_amdgcn_sched_barrier(0);
    static_for<0, 24>([&](auto kc) {
      constexpr int k = decltype(kc)::value;
      if constexpr (MORE) {
        constexpr int g = k / 6, q = k % 6;
        sn = mma(kf[g % 2][pa[q]], qf[g][pb[q]], sn);
        if constexpr (q == 5 && g + 2 < C::kG) k_frag(Kb, g + 2, kf[g % 2]);
      }
      if constexpr (k < 2) {
#pragma unroll
        for (int r = 8 * k; r < 8 * k + 8; ++r) rm = fmaxf(rm, st[r]);
      } else if constexpr (k == 2) {
        rm = pair_reduce<32>(rm, [](float x, float y) { return fmaxf(x, y); });
      } else if constexpr (k == 3) {
        alpha = sm.raise(rm, base);
      } else if constexpr (k < 20) {
        constexpr int p = (k - 4) / 2;
        if constexpr (k % 2 == 0) {
          st[2 * p] = __builtin_amdgcn_exp2f(st[2 * p] - base);
          st[2 * p + 1] = __builtin_amdgcn_exp2f(st[2 * p + 1] - base);
          rs += st[2 * p];
          rs += st[2 * p + 1];
        } else {
          split_pair(st[2 * p], st[2 * p + 1], h[p], m[p], l[p]);
        }
      } else {
        if constexpr (k == 20) sm.l = sm.l * alpha + pair_reduce<32>(rs, [](float x, float y) {
                                 return x + y;
                               });
#pragma unroll
        for (int r = 8 * (k % 2); r < 8 * (k % 2) + 8; ++r) acc[(k - 20) / 2][r] *= alpha;
      }
      if constexpr (k >= 18)
        v_frag(std::integral_constant<int, 0>{}, std::integral_constant<int, k - 18>{});
      __builtin_amdgcn_sched_barrier(0);
    });
    if constexpr (MORE) mask_v((kb + 1) * kSaKeys);
    __builtin_amdgcn_sched_barrier(0);
    bf16x8 pf[2][3];
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      pf[g][0] = __builtin_bit_cast(bf16x8, make_uint4(h[4 * g], h[4 * g + 1], h[4 * g + 2], h[4 * g + 3]));
      pf[g][1] = __builtin_bit_cast(bf16x8, make_uint4(m[4 * g], m[4 * g + 1], m[4 * g + 2], m[4 * g + 3]));
      pf[g][2] = __builtin_bit_cast(bf16x8, make_uint4(l[4 * g], l[4 * g + 1], l[4 * g + 2], l[4 * g + 3]));
    }
    static_for<0, 24>([&](auto kc) {
      constexpr int k = decltype(kc)::value, g = k / 12, q = k % 12 / 2, j = k % 2;
      acc[j] = mma(vf[g][j][pa[q]], pf[g][pb[q]], acc[j]);
      if constexpr (k >= 2 && k < 8)
        v_frag(std::integral_constant<int, 1>{}, std::integral_constant<int, k - 2>{});
      if constexpr (MORE && k % 3 == 0)
        stage_pair(std::integral_constant<int, k / 3>{}, k / 3 < 4 ? Kn : Vn);
      __builtin_amdgcn_sched_barrier(0);
    });
    if constexpr (MORE) {
      if (kb + 3 < nblocks) load_k((kb + 3) * kSaKeys);
      if (kb + 2 < nblocks) load_v((kb + 2) * kSaKeys);
      st = sn;
      sync();
    }
  };

  // Blocks past the last are staged like others but never loaded: their slots
  // hold old values that no product with a live result reads.
  uint4 *V0 = lds + 2 * C::kKs;
  load_k(0);
  load_v(0);
  mask_v(0);
  static_for<0, 4>([&](auto i) { stage_pair(i, lds); });
  static_for<4, 8>([&](auto i) { stage_pair(i, V0); });
  if (nblocks > 1) {
    load_k(kSaKeys);
    load_v(kSaKeys);
    static_for<0, 4>([&](auto i) { stage_pair(i, lds + C::kKs); });
  }
  if (nblocks > 2) load_k(2 * kSaKeys);
  sync();
#pragma unroll
  for (int g = 0; g < C::kG; ++g) {
    bf16x8 kf[3];
    k_frag(lds, g, kf);
#pragma unroll
    for (int q = 0; q < 6; ++q) st = mma(kf[pa[q]], qf[g][pb[q]], st);
  }
  sync();  // K of block 2 replaces block 0's
  for (int kb = 0; kb + 1 < nblocks; ++kb) block(std::true_type{}, kb);
  block(std::false_type{}, nblocks - 1);

  // Merge the key halves through LDS: half 1 parks (O, m, l), half 0 combines.
  smv[wave][lane] = mv;  // t % D = lane: the largest |V| of column `lane`
  {
    const float q = wave_max(mqk), v = wave_max(mv);
    if (lane == 0) {
      smx[0][wave] = q;
      smx[1][wave] = v;
    }
  }
  float *X = reinterpret_cast<float *>(lds) + rg * (16 * NB + 2) * kWave;
  // K's slots: the last block reads only V's.
  static_assert(4 * (16 * NB + 2) * kWave <= 2 * C::kKs * 4, "merge area");
  auto park = [&] {
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) X[(16 * j + r) * kWave + lane] = acc[j][r];
    X[(16 * NB) * kWave + lane] = sm.m;
    X[(16 * NB + 1) * kWave + lane] = sm.l;
  };
  float lt = 0.0f, mm = 0.0f;
  auto merge = [&] {
    const float m1 = X[(16 * NB) * kWave + lane], l1 = X[(16 * NB + 1) * kWave + lane];
    mm = fmaxf(sm.m, m1);
    const float e0 = mm == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(sm.m - mm);
    const float e1 = mm == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m1 - mm);
    lt = sm.l * e0 + l1 * e1;
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        acc[j][r] = acc[j][r] * e0 + X[(16 * j + r) * kWave + lane] * e1;
  };
  if (kh == 1) park();
  __syncthreads();
  if (kh == 0) {
    merge();
    float bq = 1.0f, bv = 1.0f;
#pragma unroll
    for (int w = 0; w < kSaWaves; ++w) {
      bq = fmaxf(bq, smx[0][w]);
      bv = fmaxf(bv, smx[1][w]);
    }
    // What the split cannot vouch for (s3_check in gemm_split.h has the bounds):
    // scores of operands over 2^60, where what an element under 2^-110 loses
    // could move a score; rows whose maximum or sum is not finite; and in O,
    // before the division,
    //   - small values: P loses at most 2^-134 an element, V too if under 2^-110,
    //     Sk (1 + max |V|) 2^-134 in a column of V, and nothing if that is zero;
    //   - non-finite ones, unless V leaves no way to them but a NaN element.
    bool bad = bq > 0x1p60f || !(lt < INFINITY) || !(mm < INFINITY);
    const float sk = float(Sk), thr = sk * bv * 0x1p-108f;
    uint32_t lo = 0xffffffffu;
    float nf = 0.0f;
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        nf = fmaf(acc[j][r], 0.0f, nf);
        lo = min(lo, __float_as_uint(acc[j][r]) << 1);
      }
    if (__builtin_expect(__any(nf != 0.0f || lo < __float_as_uint(thr) << 1), 0)) {
      bad = bad || (nf != 0.0f && !(bv < 0x1p127f && sk * bv < 0x1p126f));
      uint32_t count = 0, at = 0;  // small ones of this lane, the last one's column
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const bool small = fabsf(acc[j][r]) < thr;
          count += small;
          at = small ? 32 * j + 8 * (r / 4) + 4 * s + r % 4 : at;
        }
      // A few small ones have most likely cancelled (of normal values one sum in 1e7 is
      // exactly zero): the weights of a row add up to 1 or more here, so its terms to
      // the column's smallest |v| or more, and what they lose is nothing beside their
      // rounding where that is over the limit.  (24x1000x1000 with one zero in O: 49.1
      // us; 72 and more with its rows redone, 47.1 without it.)
      uint64_t lanes = __ballot(count > 0);
      if (__popcll(lanes) <= 4 && !__any(count > 1)) {
        for (; lanes; lanes &= lanes - 1) {
          const int d = __builtin_amdgcn_readlane(at, __builtin_ctzll(lanes));
          float hi = 0.0f, mn = INFINITY;
#pragma unroll 8
          for (int k = lane; k < Sk; k += kWave) {
            const float v = fabsf(V[int64_t(k) * a.ldv + d]);
            hi = fmaxf(hi, v);
            mn = fminf(mn, v);
          }
          bad = bad || (wave_max(hi) > 0.0f && !(wave_min(mn) >= thr));
        }
      } else {
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int d = 32 * j + 8 * (r / 4) + 4 * s + r % 4;
            float cv = 0.0f;
#pragma unroll
            for (int w = 0; w < kSaWaves; ++w) cv = fmaxf(cv, smv[w][d]);
            bad = bad || (cv > 0.0f && fabsf(acc[j][r]) < sk * fmaxf(cv, 1.0f) * 0x1p-108f);
          }
      }
    }
    bad = __any(bad);
    if (lane == 0) sbad[rg] = bad;
  }
  __syncthreads();
  if (__builtin_expect(sbad[0] | sbad[1] | sbad[2] | sbad[3], 0)) {  // the whole workgroup
    // The flagged row groups once more on the fp32 matrix cores (32x32x2: lane
    // (c, s) supplies k slot s), straight from memory, each wave its key half.
    // Slot s of step e takes d 8 g + 4 s + e, so Q and K come 16 bytes a lane.
    if (sbad[rg]) {
      sm = sa_row{};
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[j] = zero16();
      f4u q[D / 8];
#pragma unroll
      for (int g = 0; g < D / 8; ++g)
        q[g] = *reinterpret_cast<const f4u *>(qrow + 8 * g + 4 * s);
#pragma unroll 1
      for (int key0 = 32 * kh; key0 < Sk; key0 += kSaKeys) {
        const float *kp = K + int64_t(min(key0 + c, Sk - 1)) * a.ldk + 4 * s;
        f4u k4[D / 8];
#pragma unroll
        for (int g = 0; g < D / 8; ++g) k4[g] = *reinterpret_cast<const f4u *>(kp + 8 * g);
        float v[16][NB];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = key0 + 8 * (r / 4) + 4 * s + r % 4;
          const float *vp = V + int64_t(min(key, Sk - 1)) * a.ldv + c;
#pragma unroll
          for (int j = 0; j < NB; ++j) v[r][j] = key < Sk ? vp[32 * j] : 0.0f;
        }
        floatx16 sc = zero16();
#pragma unroll
        for (int g = 0; g < D / 8; ++g)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            sc = __builtin_amdgcn_mfma_f32_32x32x2f32(k4[g][e], q[g][e], sc, 0, 0, 0);
        const float alpha = sm.step(sc, scale2, key0, s, Sk);
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[j] *= alpha;
#pragma unroll
        for (int r = 0; r < 16; ++r)
#pragma unroll
          for (int j = 0; j < NB; ++j)
            acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(v[r][j], sc[r], acc[j], 0, 0, 0);
      }
      if (kh == 1) park();
    }
    __syncthreads();
    if (kh == 0 && sbad[rg]) merge();
  }
  if (kh == 1) return;
  if (row >= Sq) return;
  const float inv = lt > 0.0f ? 1.0f / lt : 0.0f;
  // Register r of block j is O[row][32 j + 8 (r / 4) + 4 s + r % 4].
  float *orow = O + int64_t(row) * a.ldo + 4 * s;
#pragma unroll
  for (int j = 0; j < NB; ++j)
#pragma unroll
    for (int r = 0; r < 16; r += 4)
      *reinterpret_cast<f4u *>(orow + 32 * j + 2 * r) =
          f4u{acc[j][r] * inv, acc[j][r + 1] * inv, acc[j][r + 2] * inv, acc[j][r + 3] * inv};
}

}  // namespace
}  // namespace silgpu
