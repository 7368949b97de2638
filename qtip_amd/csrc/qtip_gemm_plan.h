// How a batched decompress + GEMM is cut into launches, workgroups and k ranges.  Host code on numbers alone, included by
// qtip_gemm.hip and, without a device, by tests.
#pragma once
#include <stddef.h>
#include <stdint.h>

namespace qtip {
namespace {  // (every library that holds this has plans of its own)

constexpr int kFewWaves = 16, kRowsWaves = 8;  // of a workgroup of gemm_few_kernel, of gemm_rows_kernel
// a whole wave-load per stage where two tiles of it fit 32 KiB
constexpr int rows_stage_halves(int NB, int RG) { return NB * (kRowsWaves / RG) <= 8 ? 2 : 1; }

// How nb batch rows of an m-row matrix run in one launch: NB 16-row batch tiles of gemm_rows_kernel (0: gemm_few_kernel, 1:
// gemm_kernel), RG row-block pairs per workgroup, S k ranges of wl_per 64-column wave-loads (S > 1 only when the
// caller provides room for the partial results).
struct GemmPlan {
  int NB, RG, S, wl_per, nbt, ngroups;
  float us;  // what it is expected to take, with the launch that adds the ranges
};
constexpr int kMaxSplit = 16;

inline GemmPlan gemm_split(int m, int k, int nb, int NB, int RG, int KS, int S) {
  GemmPlan g{};
  g.NB = NB;
  g.RG = RG;
  g.nbt = NB ? (nb + 16 * NB - 1) / (16 * NB) : 1;
  g.ngroups = (((m >> 5) + 1) / 2 + RG - 1) / RG;
  const int nwl = ((k >> 5) + 1) >> 1;
  g.wl_per = ((nwl + S - 1) / S + KS - 1) / KS * KS;  // stages are groups of KS wave-loads
  g.S = (nwl + g.wl_per - 1) / g.wl_per;              // rounding up may have emptied the last ranges
  return g;
}

// Up to 16 rows: where the weight stream is the bound and the activations would be in its way, they are shared.  us from cold
// memory, gemm_kernel / gemm_few_kernel: 28672x8192 at 4 bits 2 rows 27.5/27.7, 6 27.9/27.9, 9 28.5/29.1, 16 28.0/34.2; at
// 3 bits 2 rows 28.5/27.6, 6 28.3/28.6, 16 27.9/30.0; 22016x4096 at 4 bits 6 rows 15.4/14.7, 9 15.6/15.1, 16 15.9/16.8;
// 10240x8192 at 4 bits 16 rows 18.2/16.9.
inline bool shared_rows(int m, int k, int bits, int nb) {
  const long n = (long)m * k;
  return bits > 2 && ((n >= 1L << 27 && nb > 4) || (n >= 85000000L && nb > 12));
}

// The form of gemm_few_kernel with the least expected time.  Fitted to 540 launches from cold memory (2 to 16 rows, all widths,
// 512x2048 to 57344x8192; 7 % root mean square, 0.1 % longer than the best form on average).
inline GemmPlan few_plan(int m, int k, int bits, int nb, int cus, bool split) {
  if (shared_rows(m, k, bits, nb)) {
    const int nwl = ((k >> 5) + 1) >> 1, ngroups = (((m >> 5) + 1) / 2 + 1) / 2;
    int S = 1;
    while (split && S < kMaxSplit && ngroups * S * 2 <= cus && nwl / (S * 2) >= 16) S *= 2;
    return gemm_split(m, k, nb, 1, 2, 8, S);
  }
  const int nwl = ((k >> 5) + 1) >> 1;
  const float step = (bits == 2 ? 0.989f : 1.208f) + (nb > 8 ? (float)(nb - 8) * (bits == 2 ? 0.008f : 0.033f) : 0.f);
  GemmPlan best{};
  for (int RG = 1; RG <= 2; ++RG) {
    const int KS = kFewWaves / RG;
    for (int S = 1; S <= (split ? kMaxSplit : 1) && (S == 1 || nwl / S >= 2); S *= 2) {
      GemmPlan g = gemm_split(m, k, nb, 0, RG, 1, S);
      if (S > 1 && (g.S == 1 || (long)g.ngroups * S > cus + cus / 8)) break;
      const long per = cus / g.S < g.ngroups ? cus / g.S : g.ngroups;
      g.us = 1.12f + (float)((g.ngroups + per - 1) / per) * ((float)((g.wl_per + KS - 1) / KS) * step + 3.f);
      if (g.S > 1) g.us += 1.51f + g.S * (0.21f + 3.23e-6f * nb * m);
      if (best.RG == 0 || g.us < best.us) best = g;
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

// From 17 rows on: the form with the least expected time.
inline GemmPlan rows_plan(int m, int k, int nb, int cus, bool split) {
  static const int kForms[][2] = {{8, 8}, {8, 4}, {6, 8}, {4, 8}, {4, 4}, {4, 2}, {2, 4}, {2, 2}};
  const int nwl = ((k >> 5) + 1) >> 1;
  GemmPlan best{};
  for (const auto& f : kForms) {
    for (int S = 1; S <= (split ? kMaxSplit : 1) && (S == 1 || nwl / S >= 4); S *= 2) {
      GemmPlan g = gemm_split(m, k, nb, f[0], f[1], kRowsWaves / f[1], S);
      if (S > 1 && (g.S == 1 || (long)g.ngroups * g.nbt * S > cus + cus / 8)) break;
      g.us = rows_time(g, m, nb, cus);
      if (best.NB == 0 || g.us < best.us) best = g;
    }
  }
  return best;
}

// A product in up to two launches over the matrix rows: [0, m0) and [m0, m).
struct GemmParts {
  int m0;
  GemmPlan first, rest;
};

inline GemmParts make_plan(int m, int k, int bits, int nb, int cus, bool split) {
  GemmParts p{m, {}, {}};
  if (nb <= 16) {
    p.first = few_plan(m, k, bits, nb, cus, split);
    return p;
  }
  p.first = rows_plan(m, k, nb, cus, split);
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
      GemmPlan a = gemm_split((int)m0, k, nb, NB, kRowsWaves, 1, 1);
      a.us = rows_time(a, (int)m0, nb, cus);
      if (a.us >= least) break;
      const GemmPlan b = rows_plan(m - (int)m0, k, nb, cus, split);
      if (a.us + b.us < least) {
        least = a.us + b.us;
        p = {(int)m0, a, b};
      }
    }
  }
  return p;
}

// The plan of a call is asked for by its size queries and by its launches; a search takes 1 to 15 us, so each thread
// keeps those of the last sizes.
inline GemmParts gemm_plan(int m, int k, int bits, int nb, int cus, bool split) {
  struct Held {
    int m, k, bits, nb, cus;  // (of split plans; the others come from callers without scratch)
    GemmParts plan;
  };
  static thread_local Held held[64];
  if (!split) return make_plan(m, k, bits, nb, cus, false);
  Held& h = held[((uint32_t)m * 0x9E3779B1u ^ (uint32_t)k * 0x85EBCA77u ^ (uint32_t)(4 * nb + bits) * 0xC2B2AE3Du) >> 26];
  if (h.m != m || h.k != k || h.bits != bits || h.nb != nb || h.cus != cus)
    h = {m, k, bits, nb, cus, make_plan(m, k, bits, nb, cus, true)};
  return h.plan;
}

// Rows of one pass: as many as 32-bit buffer offsets reach (2 GiB less the offset that stands for padding)
inline int pass_rows(int k) {
  const long fit = 0x7FFFFF00L / (2L * k);
  return fit >= 65536 ? 65536 : fit >= 128 ? (int)(fit & ~127L) : (int)fit;
}

inline size_t parts_bytes(const GemmPlan& g, int m, int nb) { return g.S > 1 ? (size_t)g.S * nb * m * sizeof(float) : 0; }

}  // namespace
}  // namespace qtip
