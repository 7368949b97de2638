// How a batched decompress + GEMM is cut into launches, workgroups and k ranges.  Host code on numbers alone, included by
// qtip_gemm.hip and, without a device, by tests.
#pragma once
#include <stddef.h>
#include <stdint.h>

#include <initializer_list>

namespace qtip {
namespace {  // (every library that holds this has plans of its own)

constexpr int kFewWaves = 16, kRowsWaves = 8;  // of a workgroup of gemm_few_kernel, of gemm_rows_kernel
// a whole wave-load per stage where two tiles of it fit 32 KiB
constexpr int rows_stage_halves(int NB, int RG) { return NB * (kRowsWaves / RG) <= 8 ? 2 : 1; }

enum GemmForm { kFew, kShared, kRows };  // gemm_few_kernel, gemm_kernel, gemm_rows_kernel
constexpr int form_slices(GemmForm f, int RG) { return (f == kRows ? kRowsWaves : 16) / RG; }  // of k in a workgroup

// How nb batch rows of an m-row matrix run in one launch: the kernel with its NB 16-row batch tiles and RG row-block pairs per
// workgroup, S k ranges of wl_per 64-column wave-loads (S > 1 only when the caller provides room for the partial results).
struct GemmPlan {
  GemmForm form;
  int NB, RG, S, wl_per, nbt, ngroups;
  float us;  // what it is expected to take, with the launch that adds the ranges
};
constexpr int kMaxSplit = 16;

// (step: ranges are multiples of so many wave-loads, 0 for whole stages of the workgroup's slices)
inline GemmPlan gemm_split(int m, int k, int nb, GemmForm form, int NB, int RG, int S, int step = 0) {
  GemmPlan g{};
  g.form = form;
  g.NB = NB;
  g.RG = RG;
  g.nbt = (nb + 16 * NB - 1) / (16 * NB);
  g.ngroups = (((m >> 5) + 1) / 2 + RG - 1) / RG;
  const int nwl = ((k >> 5) + 1) >> 1;
  if (!step) step = form_slices(form, RG);
  g.wl_per = ((nwl + S - 1) / S + step - 1) / step * step;
  g.S = (nwl + g.wl_per - 1) / g.wl_per;  // rounding up may have emptied the last ranges
  return g;
}

// How far fp32 sums of random products are off, in chains of L additions on the matrix cores, KS slices added up in a workgroup
// and S ranges of k after that: measured 1.6e-8 sqrt(5 + 5 L + 1.5 KS + S) in 2-norm, at every plan (L64 KS2 S2 2.9e-7, L56 KS2 S8
// 2.8e-7, L4 KS8 S4 1.03e-7, L128 alone 4.1e-7; a matrix product rounds more than once per 32 columns).  `sum_error`
// is 5 L + 1.5 KS + S.
inline int sum_error(int k, int KS, int wl_per, int S) {
  const int nwl = ((k >> 5) + 1) >> 1, in_range = wl_per < nwl ? wl_per : nwl;
  return 10 * ((in_range + KS - 1) / KS) + (KS < in_range ? KS : in_range) * 3 / 2 + S;
}
inline int sum_error(const GemmPlan& g, int k) { return sum_error(k, form_slices(g.form, g.RG), g.wl_per, g.S); }

// Fine sums: 8, 4 or 2 slices (up to 32, 64, 128 rows) and, while CUs would be idle, ranges of at least 1024 columns, 512 from 33
// rows on.  A plan may be off by no more than such a cut is, the finest among pieces of 128 rows.  The library's product
// of the dense matrix, which projections of many rows would otherwise be, sums in chains of k / 32 and is off by 4 to 7e-7:
// long sums (qtip_decompress_gemm_long_f16) leave the plan to the time alone.
constexpr int kAnyError = 1 << 30;
inline int ranges_by_idle_cus(int k, int ngroups, int least, int cus, bool split) {
  const int nwl = ((k >> 5) + 1) >> 1;
  int S = 1;
  while (split && S < kMaxSplit && ngroups * S * 2 <= cus && nwl / (S * 2) >= least) S *= 2;
  return S;
}
inline int fine_error(int m, int k, int nb, int cus, bool split) {
  if (nb > 128) {
    const int a = fine_error(m, k, 128, cus, split), b = fine_error(m, k, nb - 128, cus, split);
    return a < b ? a : b;
  }
  const int KS = nb <= 32 ? 8 : nb <= 64 ? 4 : 2, RG = nb <= 64 ? 2 : 4, nwl = ((k >> 5) + 1) >> 1;
  const int S = ranges_by_idle_cus(k, (((m >> 5) + 1) / 2 + RG - 1) / RG, nb <= 32 ? 16 : 8, cus, split);
  const int wl_per = ((nwl + S - 1) / S + KS - 1) / KS * KS;
  return sum_error(k, KS, wl_per, (nwl + wl_per - 1) / wl_per);
}

// Up to 16 rows: where the stream of weights is long and a wave's own reads of the activations would stand in its way, they are shared.  us from cold
// memory, gemm_kernel / gemm_few_kernel: 28672x8192 at 4 bits 2 rows 27.5/27.7, 6 27.9/27.9, 9 28.5/29.1, 16 28.0/34.2; at
// 3 bits 2 rows 28.5/27.6, 6 28.3/28.6, 16 27.9/30.0; 22016x4096 at 4 bits 6 rows 15.4/14.7, 9 15.6/15.1, 16 15.9/16.8;
// 10240x8192 at 4 bits 16 rows 18.2/16.9.
inline bool shared_rows(int m, int k, int bits, int nb) {
  const long n = (long)m * k;
  return bits > 2 && ((n >= 1L << 27 && nb > 4) || (n >= 85000000L && nb > 12));
}

// gemm_kernel: 17 to 32 rows, and up to 16 where they are shared.  (us: of 17 rows on)
inline GemmPlan shared_plan(int m, int k, int bits, int nb, int cus, bool split) {
  GemmPlan g = gemm_split(m, k, nb, kShared, nb <= 16 ? 1 : 2, 2, 1);
  g = gemm_split(m, k, nb, kShared, g.NB, 2, ranges_by_idle_cus(k, g.ngroups, 16, cus, split));
  const int per = cus / g.S < g.ngroups ? cus / g.S : g.ngroups;
  g.us = 4.6f + (float)((g.ngroups + per - 1) / per) * (float)(g.wl_per / 8) * (bits == 2 ? 1.87f : 2.08f) + (g.S > 1 ? 3.f : 0.f);
  return g;
}

// The form of gemm_few_kernel with the least expected time, of those off by no more than `most`: fine sums take 7 % longer than
// the fastest form on average, up to 30 % (2048x11008).  Fitted to 540 launches from
// cold memory (2 to 16 rows, all widths, 512x2048 to 57344x8192; 7 % root mean square).
inline GemmPlan few_plan(int m, int k, int bits, int nb, int cus, bool split, int most) {
  const int nwl = ((k >> 5) + 1) >> 1;
  const float step = (bits == 2 ? 0.989f : 1.208f) + (nb > 8 ? (float)(nb - 8) * (bits == 2 ? 0.008f : 0.033f) : 0.f);
  GemmPlan best{};
  for (int RG = 1; RG <= 2; ++RG) {
    const int KS = kFewWaves / RG;
    for (int S = 1; S <= (split ? kMaxSplit : 1) && (S == 1 || nwl / S >= 2); S *= 2) {
      GemmPlan g = gemm_split(m, k, nb, kFew, 1, RG, S, 1);
      if (S > 1 && (g.S == 1 || (long)g.ngroups * S > cus + cus / 8)) break;
      if (sum_error(g, k) > most) g = gemm_split(m, k, nb, kFew, 1, RG, S);  // (no more chain for fewer ranges)
      if (sum_error(g, k) > most) continue;
      const long per = cus / g.S < g.ngroups ? cus / g.S : g.ngroups;
      g.us = 1.12f + (float)((g.ngroups + per - 1) / per) * ((float)((g.wl_per + KS - 1) / KS) * step + 3.f);
      if (g.S > 1) g.us += 1.51f + g.S * (0.21f + 3.23e-6f * nb * m);
      if (!best.RG || g.us < best.us) best = g;
    }
  }
  return best;
}

// Where a lane of gemm_few_kernel reads the activations of wave-load wl, the first of the nst of its wave in a unit, with
// `units` units to go: scalar and lane offset of 16 bytes (16 more at + 32; the next wave-load is KS * 128 bytes on).
// Without anything to read the lane offset is out of range by itself and the scalar one 0: the range check of a buffer load
// need not cover the scalar offset, and one past the end leaves it nothing to check against.  That is so for rows past the
// batch, behind the last unit, and in a wave whose slice has no wave-load in this range of k (nst 0).  last_half: the last
// of the nst ends after 32 columns.
struct FewPlace {
  uint32_t so, vo;
};
constexpr uint32_t kOutOfRange = 0x7FFFFF00u;
constexpr FewPlace few_activations(int lane, int batch, int k, int wl, int units, int nst, bool last_half) {
  const int row = lane & 15, ch = (lane >> 4) & 1, g0 = lane >> 5;
  if (units < 1 || nst < 1) return {0, kOutOfRange};
  const bool in = row < batch && !(last_half && nst == 1 && g0);
  return {(uint32_t)wl * 128, in ? ((uint32_t)row * (uint32_t)k + (uint32_t)(32 * g0 + 8 * ch)) * 2 : kOutOfRange};
}

// What a launch of gemm_rows_kernel (and the one that adds its k ranges) takes, in us.  The terms are fitted to 4000
// measured launches (2 and 4 bits, 17 to 2000 rows, matrices of 512x2048 to 28672x8192): 5 % root mean square, and the
// form with the least of it takes 0.4 % longer than the best one on average.  A fixed part, per unit its
// stores, per wave-load the step, faster where part of the chip idles (the clock), slower where a stage is half
// a wave-load or its pieces of activations do not come out even; for k ranges the partial results and their launch.
inline float rows_time(const GemmPlan& g, int m, int nb, int cus) {
  const int KS = kRowsWaves / g.RG, NB = g.NB;
  const long units = (long)g.ngroups * g.nbt, per = cus / g.S < units ? cus / g.S : units;
  const float form = NB == 6 ? 1.06f : rows_stage_halves(NB, g.RG) == 2 ? 1.f : NB == 4 ? 1.24f : 1.057f;
  const float steps = (float)(g.wl_per / KS) * (0.64f + 0.099f * NB) * form, store = 0.19f + 0.724f * NB;
  auto round = [&](long n) { return steps * (0.8f + 0.2f * (float)(n * g.S) / cus) + store; };
  float us = 5.2f + (float)(units / per) * round(per);
  if (units % per) us += round(units % per);
  if (g.S > 1) us += 1.07f + 0.265f * g.S + (float)nb * m * (1.26e-6f * g.S + 0.77e-6f);
  return us;
}

// gemm_rows_kernel: the form with the least expected time, of those off by no more than `most`.  (Ranges beyond what fills the
// chip are not worth their launch, but may be what keeps the sums fine.)
inline GemmPlan rows_plan(int m, int k, int nb, int cus, bool split, int most) {
  static const int kForms[][2] = {{8, 8}, {8, 4}, {6, 8}, {4, 8}, {4, 4}, {4, 2}, {2, 4}, {2, 2}};
  const int nwl = ((k >> 5) + 1) >> 1;
  GemmPlan best{};
  for (const auto& f : kForms) {
    for (int S = 1; S <= (split ? kMaxSplit : 1) && (S == 1 || nwl / S >= 4); S *= 2) {
      GemmPlan g = gemm_split(m, k, nb, kRows, f[0], f[1], S);
      if (S > 1 && (g.S == 1 || (long)g.ngroups * g.nbt * S > (most == kAnyError ? cus + cus / 8 : 2 * cus))) break;
      if (sum_error(g, k) > most) continue;
      g.us = rows_time(g, m, nb, cus);
      if (!best.RG || g.us < best.us) best = g;
    }
  }
  return best;
}

// A product in up to two launches over the matrix rows: [0, m0) and [m0, m).
struct GemmParts {
  int m0;
  GemmPlan first, rest;
};

// Fine sums, any number of rows.  Without scratch for ranges the bound is that of a cut product all the same where a plan keeps
// it (a caller whose plan has one range need not bring any), else that of the uncut one.
inline GemmPlan fine_plan(int m, int k, int bits, int nb, int cus, bool split) {
  if (nb <= 16 ? shared_rows(m, k, bits, nb) : nb <= 32) return shared_plan(m, k, bits, nb, cus, split);
  GemmPlan g{};
  for (int most : {fine_error(m, k, nb, cus, true), fine_error(m, k, nb, cus, split), kAnyError}) {
    g = nb <= 16 ? few_plan(m, k, bits, nb, cus, split, most) : rows_plan(m, k, nb, cus, split, most);
    if (g.RG) break;
  }
  return g;
}

// Long sums: the least expected time whatever the chains.
inline GemmParts long_plan(int m, int k, int nb, int cus, bool split) {
  GemmParts p{m, rows_plan(m, k, nb, cus, split, kAnyError), {}};
  // Units beyond whole rounds of the chip as a launch of their own, in the form that suits what is left: 22016x4096,
  // 700 rows (258 units of 512 matrix by 128 batch rows on 256 CUs) 144 -> 129 us, 12288x4096, 1400 rows 172 -> 136.
  // Where it should give a twelfth at least: at 0.97 22016x4096 lost 4 % at 1000 to 2000 rows (the clock makes up for
  // part of an idle chip).  Tried where the gain covers the host's search.
  if (p.first.us < 40.f) return p;
  float least = 0.92f * p.first.us;
  for (int NB = 8; NB >= 4; NB -= 2) {
    const int per = cus / ((nb + 16 * NB - 1) / (16 * NB));  // groups a round
    for (int rounds = 1; per && rounds <= 3; ++rounds) {
      const long m0 = (long)per * rounds * kRowsWaves * 64;
      if (m0 >= m) break;
      GemmPlan a = gemm_split((int)m0, k, nb, kRows, NB, kRowsWaves, 1);
      a.us = rows_time(a, (int)m0, nb, cus);
      if (a.us >= least) break;
      const GemmPlan b = rows_plan(m - (int)m0, k, nb, cus, split, kAnyError);
      if (a.us + b.us < least) {
        least = a.us + b.us;
        p = {(int)m0, a, b};
      }
    }
  }
  return p;
}

// The plan of a call is asked for by its size queries and by its launches; a search takes up to 3 us (of 1000 rows; 0.1 to 1
// of few), so each thread keeps those of the last sizes.  The slot: sizes that share one at some row count and bit width (as
// 11008x4096 and 4096x11008 at all of them, if every size had a factor of its own) must not do so at the next.
inline unsigned plan_slot(int m, int k, int bits, int nb, bool split, bool fine) {
  uint32_t h = 0;
  for (uint32_t v : {(uint32_t)m, (uint32_t)k, (uint32_t)(16 * nb + 4 * bits + 2 * split + fine)}) {
    h = (h + v) * 0x9E3779B1u;
    h ^= h >> 15;
  }
  return (h * 0x85EBCA77u) >> 26;
}
inline GemmParts gemm_plan(int m, int k, int bits, int nb, int cus, bool split, bool fine) {
  struct Held {
    int m, k, bits, nb, cus;
    bool split, fine;
    GemmParts plan;
  };
  static thread_local Held held[64];
  Held& h = held[plan_slot(m, k, bits, nb, split, fine)];
  if (h.m != m || h.k != k || h.bits != bits || h.nb != nb || h.cus != cus || h.split != split || h.fine != fine)
    h = {m, k, bits, nb, cus, split, fine,
         fine ? GemmParts{m, fine_plan(m, k, bits, nb, cus, split), {}} : long_plan(m, k, nb, cus, split)};
  return h.plan;
}

// Rows of one pass: as many as 32-bit buffer offsets reach (2 GiB less the offset that stands for padding)
inline int pass_rows(int k) {
  const long fit = 0x7FFFFF00L / (2L * k);
  return fit >= 65536 ? 65536 : fit >= 128 ? (int)(fit & ~127L) : (int)fit;
}

// The next pass of a product with `left` rows to go.  Fine sums: up to 256 rows where a launch of them takes less than one of 128 and
// one of the rest, else 128.
inline int next_pass(int m, int k, int bits, int left, int cus, bool split, bool fine) {
  const int reach = pass_rows(k);
  if (!fine) return left < reach ? left : reach;
  int nb = left < 256 ? left : 256;
  if (nb > 128 && nb <= reach) {
    const GemmPlan whole = gemm_plan(m, k, bits, nb, cus, split, true).first;
    if (sum_error(whole, k) <= fine_error(m, k, nb, cus, split) &&
        whole.us < gemm_plan(m, k, bits, 128, cus, split, true).first.us +
                       gemm_plan(m, k, bits, nb - 128, cus, split, true).first.us)
      return nb;
  }
  if (nb > 128) nb = 128;
  return nb < reach ? nb : reach;
}

inline size_t parts_bytes(const GemmPlan& g, int m, int nb) { return g.S > 1 ? (size_t)g.S * nb * m * sizeof(float) : 0; }

}  // namespace
}  // namespace qtip
