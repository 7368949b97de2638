// Batched decompress + fp16 MFMA GEMM (qtip_decompress_gemm).  Declarations: include/qtip_hip.h.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/qtip_hip.h"
#include "qtip_device.h"
#include "qtip_setup.h"
#include "qtip_gemm_plan.h"

using namespace qtip;

namespace {

// Batched decompress + fp16 MFMA GEMM: out[b][row] = sum_col x[b][col] * W[row][col].
//
// A wave works on a pair of 32-row blocks (64 rows) and 64 columns at a time, a wave-load: two 2x2 tile blocks of
// either row block, 512*K bytes.  Lane bits: 0..2 row r8, 3 row block of the pair, 4 column half c,
// 5 column block; the lane loads the 8*K bytes of reference lanes 4 r8 + 2c and 4 r8 + 2c + 1 of its
// tile block.  For a given (tile row half mh, row half rh, column half of the block kh) the lane's four
// table words are eight weights of ONE matrix row, and the sixteen lanes of a DPP row hold the same
// columns of sixteen different rows, with the four DPP rows holding the four column groups: an operand of
// v_mfma_f32_16x16x32_f16 (row = lane % 16, K group = lane / 16) in which every product is
// wanted, straight from the table lookups, at every bit width.  (Lanes that split a row's columns
// inside a DPP row - the matvec's map - leave half of every product meaningless: twice the products
// and twice the accumulators.)  The successor chunk a lane's last reference lane needs sits 16 lanes
// away or one row on: ds_bpermute.
//
// Three kernels: gemm_few_kernel up to 16 batch rows, gemm_kernel up to 32 (and up to 16 of the largest matrices),
// gemm_rows_kernel beyond.  S > 1: k is cut into S ranges, fp32 partial results go to parts[s][batch][m] and are summed afterwards.
constexpr size_t kGemmTileBytes = 32 * 1024;  // beside the table: tiles of activations, sums of slices
constexpr size_t kGemmLds = kLut128Bytes + kGemmTileBytes;

// 17 to 32 batch rows (NB = 2), and up to 16 of the largest matrices at 3 and 4 bits (NB = 1, see shared_rows).  A workgroup of 16
// waves: two row-block pairs x KS = 8 column slices of 64.  The activations of a stage (16 NB
// batch rows x 512 columns) are shared through LDS, each 16-byte chunk holding the eight values one lane's A operand
// needs, chunk index xor-ed with the row (conflict-free both ways).  The next tile waits in registers; with room for two
// tiles in LDS there is one barrier per stage, else two.  Work unit = (two pairs, k range s); a workgroup keeps one s, so the
// pipeline runs across unit boundaries.  The k slices of a unit meet in the tile buffer at its end.
// NB = 1 waits at its barriers and for LDS (28672x8192, 4 bits, 16 rows: 4.0 TB/s of weights, waits 48 % of the waves' cycles, LDS busy
// 54 %, a fifth of that conflicts; the kernel of one row streams 5.5), NB = 2 for its stages' phases.  The forms of gemm_rows_kernel at 17 to 32 rows have
// half the slices: within what eight of them are off by (fine_error) they take 0.9 to 1.6 times as long, with chains twice as
// long 0.87 to 1.08.  us from cold memory, launches and sums of ranges included, 32 rows at 2 bits: 4096x4096 13.1,
// 22016x4096 19.7, 28672x8192 34, 4096x11008 17.1, 8192x28672 36.
constexpr int kWaves = 16, kThreads = 64 * kWaves;

// CUT: k / 32 is odd.  (A kernel of its own: looking for the last wave-load costs 2 % at 17 to 32 rows.)
template <int K, int NB, bool CUT, typename TOut>
__global__ __launch_bounds__(kThreads, 1) void gemm_kernel(
    TOut* __restrict__ dst, const uint8_t* __restrict__ packed, const uint16_t* __restrict__ x,
    const uint32_t* __restrict__ tlut, int m, int k, int batch, long ldo, int round_f16, int wl_per, int upw_q, int upw_r) {
  constexpr int WAVES = kWaves, RG = 2, THREADS = kThreads, DEPTH = 2;
  constexpr int KS = WAVES / RG;
  constexpr int ROWB = KS * 128;               // bytes per tile row
  constexpr int CPR = ROWB / 16;               // 16-byte chunks per tile row
  constexpr uint32_t TILE = 16 * NB * ROWB;
  constexpr bool DB = 2 * TILE <= kGemmTileBytes;  // two tiles fit
  constexpr int CHUNKS = 16 * NB * CPR;
  constexpr int NX = (CHUNKS + THREADS - 1) / THREADS;  // chunks per thread
  static_assert(TILE <= kGemmTileBytes && TILE >= WAVES * 1024, "the tile, or the exchange in it, does not fit");
  extern __shared__ __align__(16) uint8_t smem[];
  uint32_t* lut = reinterpret_cast<uint32_t*>(smem);
  uint8_t* tile = smem + kLut128Bytes;  // [1 or 2][16*NB rows][ROWB bytes]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rg = wave % RG, ks = wave / RG;
  const int r8 = lane & 7, pb = (lane >> 3) & 1, ch = (lane >> 4) & 1, g0 = lane >> 5;
  const uint32_t slot4 = lds_address(lut) + ((uint32_t)(lane & 31) << 2);
  const int nkb = k >> 5;
  const int nwl = (nkb + 1) >> 1;  // 64-column wave-loads per row
  const int nrb = m >> 5;
  const int npair = (nrb + 1) >> 1;
  const uint32_t rb_bytes = (uint32_t)nkb * 128 * K;
  constexpr uint32_t WL_BYTES = 256 * K;
  const uint32_t loff = (uint32_t)pb * rb_bytes + (uint32_t)g0 * (128 * K) + (uint32_t)(2 * r8 + ch) * (8 * K);
  // lane of the successor piece: the other column half of the row, or the first half of the next row
  const int nxt4 = (ch ? ((lane & ~23) | ((r8 + 1) & 7)) : (lane | 16)) << 2;
  const __amdgpu_buffer_rsrc_t rs_w = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(packed), 0, (int)((size_t)nrb * rb_bytes), 0x00020000);

  // grid = (S, workgroups per k range); unit counts as quotient and remainder from the host
  const int s = blockIdx.x;
  const int u0 = blockIdx.y, ustep = gridDim.y;
  const int wl0 = s * wl_per;  // wl_per is a multiple of KS
  const int wl1 = wl0 + wl_per < nwl ? wl0 + wl_per : nwl;
  const int nst = wl1 > wl0 ? (wl1 - wl0 + KS - 1) / KS : 0;  // stages per unit
  const int upw = upw_q + (u0 < upw_r ? 1 : 0);
  const int T = upw * nst;
  TOut* out_s = dst + (size_t)s * batch * ldo;

  // ---- weight stream of this wave, DEPTH stages in flight
  int l_t = 0, l_q = 0, l_u = u0;
  LaneData<K> buf[DEPTH];
  auto issue = [&](int d) {
    const int pair = l_u * RG + rg;
    const int wl = wl0 + KS * l_t + ks;
    const bool valid = l_q < T && pair < npair && wl < wl1;
    // padding items, the missing second row block of an odd count and the missing second column block of
    // a partial last wave-load: a lane offset that is out of range by itself, zeros without a memory access
    const bool lane_ok = valid && 2 * wl + g0 < nkb && 2 * pair + pb < nrb;
    buf[d] = load_lane_buf<K>(rs_w, lane_ok ? loff : 0x7FFFFF00u,
                              valid ? (uint32_t)(2 * pair) * rb_bytes + (uint32_t)wl * WL_BYTES : 0u);
    ++l_q;
    if (++l_t == nst) {
      l_t = 0;
      l_u += ustep;
    }
  };
  // table words through the scalar cache first, one stage of the stream before the table is built
  constexpr int NTW = kLutEntries * 4 / THREADS;  // distinct table words per thread
  uint32_t tw[NTW];
#pragma unroll
  for (int j = 0; j < NTW; ++j) {
    const uint32_t* tp = tlut + j * (THREADS / 8) + wave * 8;
    typedef uint32_t u32x8_dw __attribute__((ext_vector_type(8), aligned(4)));
    const u32x8_dw sw = *reinterpret_cast<const u32x8_dw*>(tp);
    uint32_t v = sw[0];
#pragma unroll
    for (int e = 1; e < 8; ++e) v = ((lane >> 3) == e) ? sw[e] : v;
    tw[j] = v;
  }
  issue(0);

  // ---- activation tiles: chunk q of a row = slice * 8 + column block * 4 + kh * 2 + column half
  u32x4 xg[NX];
  // (unconditional loads: padding rows and columns have an out-of-range lane offset, which returns zeros.
  // Behind a branch the compiler loses count of the loads in flight and waits for all of them, the weight
  // stream included, at every stage.)
  const __amdgpu_buffer_rsrc_t rs_x =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(x), 0, (int)((size_t)batch * k * 2), 0x00020000);
  auto load_tile = [&](int t) {  // stage t of a unit -> registers (eight consecutive columns)
    const int col0 = 64 * (wl0 + KS * t);
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const int idx = i * THREADS + tid;
      const int b = idx / CPR, c = idx % CPR;
      const bool ok = b < batch && col0 + 8 * c < k && (CHUNKS % THREADS == 0 || idx < CHUNKS);
      xg[i] = __builtin_amdgcn_raw_buffer_load_b128(rs_x, ok ? (uint32_t)(b * k + 8 * c) * 2 : 0x7FFFFF00u,
                                                          (uint32_t)col0 * 2, 0);
    }
  };
  auto store_tile = [&](uint32_t base) {  // columns 0..3 and 4..7 of the eight belong to different chunks
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const int idx = i * THREADS + tid;
      if (CHUNKS % THREADS == 0 || idx < CHUNKS) {
        const int b = idx / CPR, c = idx % CPR;
        const int q = (c & ~1), jh = c & 1;  // chunks q (first half) and q + 1 (second half), word pair jh
        uint8_t* row = tile + base + b * ROWB + 8 * jh;
        *reinterpret_cast<u32x2*>(row + ((q ^ (b & 7)) << 4)) = u32x2{xg[i][0], xg[i][1]};
        *reinterpret_cast<u32x2*>(row + (((q + 1) ^ (b & 7)) << 4)) = u32x2{xg[i][2], xg[i][3]};
      }
    }
  };
  load_tile(0);
#pragma unroll
  for (int it = 0; it < 2 * NTW; ++it) {
    const uint32_t w = tw[it % NTW] ^ ((uint32_t)(it / NTW) << 15);
    const u32x4 v = {w, w, w, w};
    reinterpret_cast<u32x4*>(lut)[it * THREADS + tid] = v;
  }
  store_tile(0);
  load_tile(nst > 1 ? 1 : 0);
  __syncthreads();
#pragma unroll
  for (int d = 1; d < DEPTH; ++d) issue(d);

  float4_t acc[2][2][NB];  // [mh][rh][batch tile]
#pragma unroll
  for (int i = 0; i < 4 * NB; ++i) (&acc[0][0][0])[i] = float4_t{0.f, 0.f, 0.f, 0.f};
  const uint32_t tile_addr = lds_address(tile) + (uint32_t)(lane & 15) * ROWB;
  const uint32_t a7 = (uint32_t)(lane & 7);
  typedef __attribute__((address_space(3))) const u32x4 lds_u32x4_t;

  int c_t = 0, c_u = u0;
  for (int q = 0; q < T; q += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      // (an odd last stage: nothing to multiply, but its loads and barriers stay unconditional - see load_tile)
      const bool live = q + d < T;  // uniform over the workgroup
      const uint32_t cb = DB ? (uint32_t)(d & 1) * TILE : 0u;  // this stage's tile
      if (live) {
        const int pair = c_u * RG + rg;
        const int wl = wl0 + KS * c_t + ks;
        if (pair < npair && wl < wl1) {
          uint32_t P[16];
          packed_states<K>(buf[d], P, [&](uint32_t v) { return (uint32_t)__builtin_amdgcn_ds_bpermute(nxt4, (int)v); });
#pragma unroll
          for (int kh = 0; kh < 2; ++kh) {
            uint32_t Q[16];  // hashes of this kh's registers
#pragma unroll
            for (int i = 0; i < 16; ++i)
              if (((i >> 2) & 1) == kh) Q[i] = pk_hash(P[i]) & 0xFFC0FFC0u;
            uint32_t W[2][2][4];  // [mh][rh]: the B operand's words
#pragma unroll
            for (int mh = 0; mh < 2; ++mh)
#pragma unroll
              for (int rh = 0; rh < 2; ++rh)
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                  const int R = w & 1, j = 2 * (w >> 1) + rh;
                  const int wi = w_index<K>(R, 2 * kh + mh, j);  // register wi / 2, half wi % 2
                  W[mh][rh][w] = lds_word_abs((wi & 1) ? lut128_addr_hi(Q[wi >> 1], slot4) : lut128_addr_lo(Q[wi >> 1], slot4));
                }
            if constexpr (CUT) {
              // no second column block: its zeros decode to table entry 0, which zero activations do not cancel if
              // it is infinite
              if (wl == nwl - 1) {
#pragma unroll
                for (int i = 0; i < 16; ++i) (&W[0][0][0])[i] = g0 ? 0u : (&W[0][0][0])[i];
              }
            }
            __builtin_amdgcn_sched_barrier(0);
            const uint32_t ca = tile_addr + cb + ((((uint32_t)(8 * ks + 4 * g0 + 2 * kh + ch)) ^ a7) << 4);
            u32x4 xa[NB];
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) xa[nb] = *(lds_u32x4_t*)(uintptr_t)(ca + (uint32_t)nb * 16 * ROWB);
#pragma unroll
            for (int mh = 0; mh < 2; ++mh)
#pragma unroll
              for (int rh = 0; rh < 2; ++rh) {
                const u32x4 wv = {W[mh][rh][0], W[mh][rh][1], W[mh][rh][2], W[mh][rh][3]};
#pragma unroll
                for (int nb = 0; nb < NB; ++nb)
                  acc[mh][rh][nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                      __builtin_bit_cast(half8_t, xa[nb]), __builtin_bit_cast(half8_t, wv), acc[mh][rh][nb], 0, 0, 0);
              }
          }
        }
      }
      {
        int t2 = c_t + 2;  // the tile that replaces the next one in its registers
        if (t2 >= nst) t2 -= nst;
        if (t2 >= nst) t2 -= nst;  // nst == 1
        if constexpr (DB) {
          // the next tile (in registers since the previous stage) into the other buffer, the one after it on its way
          store_tile((uint32_t)((d + 1) & 1) * TILE);
          load_tile(t2);
          issue(d);
        }
        __syncthreads();  // every wave has read this stage's tile (and, with two buffers, written the next)
        const bool unit_end = live && c_t + 1 == nst;
        if (unit_end) {
          // ---- end of a unit: the k slices meet in this stage's tile buffer, TI accumulator vectors of every
          // wave at a time, summed in slice order
          constexpr int TI = TILE / (WAVES * 1024);  // vectors that fit
          float* xch = reinterpret_cast<float*>(tile + cb);
          const float4_t* av = &acc[0][0][0];
#pragma unroll
          for (int f0 = 0; f0 < 4 * NB; f0 += TI) {  // (TI divides 4 * NB)
            static_assert((4 * NB) % TI == 0, "whole steps");
#pragma unroll
            for (int t = 0; t < TI; ++t)
              *reinterpret_cast<float4_t*>(xch + ((wave * TI + t) * 64 + lane) * 4) = av[f0 + t];
            __syncthreads();
            // RG * TI * 256 sums: thread -> (pair, vector, element, lane)
            constexpr int SUMS = RG * TI * 256;
#pragma unroll
            for (int i = 0; i < (SUMS + THREADS - 1) / THREADS; ++i) {
              const int idx = i * THREADS + tid;
              if (SUMS % THREADS == 0 || idx < SUMS) {
                const int ln = idx & 63, e = (idx >> 6) & 3, t = (idx >> 8) % TI, g = (idx >> 8) / TI;
                float sum = 0.f;
#pragma unroll
                for (int z = 0; z < KS; ++z) sum += xch[(((z * RG + g) * TI + t) * 64 + ln) * 4 + e];
                const int f = f0 + t, nb = f % NB, mr = f / NB;  // mr = 2 mh + rh
                const int bb = 16 * nb + 4 * (ln >> 4) + e;
                const int row = 64 * (c_u * RG + g) + 32 * ((ln >> 3) & 1) + 8 * mr + (ln & 7);
                if constexpr (sizeof(TOut) == 4) {
                  if (round_f16) sum = (float)(_Float16)sum;
                }
                if (bb < batch && row < m) out_s[(size_t)bb * ldo + row] = (TOut)sum;
              }
            }
            __syncthreads();
          }
#pragma unroll
          for (int i = 0; i < 4 * NB; ++i) (&acc[0][0][0])[i] = float4_t{0.f, 0.f, 0.f, 0.f};
          c_u += ustep;
        }
        c_t = unit_end ? 0 : c_t + (live ? 1 : 0);
        if constexpr (!DB) {
          store_tile(0);
          load_tile(t2);
          issue(d);
          __syncthreads();  // the next tile is complete
        }
      }
    }
  }
}

#include "qtip_gemm_rows.h"
#include "qtip_gemm_few.h"

// out[row][i] = parts[0][row][i] + ... (+ rounding through fp16) for products cut along k, four at a time: mq = m / 4,
// parts[s] dense, rows of out ldo apart
template <typename TOut>
__global__ __launch_bounds__(256) void sum_parts_round_kernel(TOut* __restrict__ out, const float4_t* __restrict__ parts,
                                                              long n, int mq, long ldo, int S, int round_f16) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  float4_t sum = parts[i];
  for (int s = 1; s < S; ++s) sum += parts[(size_t)s * n + i];
  typedef TOut out4_t __attribute__((ext_vector_type(4), aligned(sizeof(TOut))));  // (out may start anywhere)
  out4_t r;
#pragma unroll
  for (int e = 0; e < 4; ++e) r[e] = (TOut)(round_f16 ? (float)(_Float16)sum[e] : sum[e]);
  *reinterpret_cast<out4_t*>(out + (i / mq) * ldo + 4 * (i % mq)) = r;
}

template <int K, typename T>
void launch_gemm(const GemmPlan& g, T* dst, long ldo, const uint8_t* p, const uint16_t* x, const uint32_t* t, int m, int k,
                 int nb, int round_f16, int cus, hipStream_t st) {
  const long units = (long)g.ngroups * g.nbt;
  const int per = (int)(cus / g.S < units ? cus / g.S : units);  // workgroups per k range
  const dim3 grid((unsigned)g.S, (unsigned)per);
  const int uq = (int)(units / per), ur = (int)(units % per);
  if (g.form == kShared) {
    auto* kernel = (k >> 5) & 1 ? gemm_kernel<K, 2, true, T> : gemm_kernel<K, 2, false, T>;
    if constexpr (K > 2)
      if (g.NB == 1) kernel = (k >> 5) & 1 ? gemm_kernel<K, 1, true, T> : gemm_kernel<K, 1, false, T>;
    kernel<<<grid, kThreads, kGemmLds, st>>>(dst, p, x, t, m, k, nb, ldo, round_f16, g.wl_per, uq, ur);
    return;
  }
  if (g.form == kFew) {
    if (g.RG == 2)
      gemm_few_kernel<K, 2, T><<<grid, 64 * kFewWaves, kGemmLds, st>>>(dst, p, x, t, m, k, nb, ldo, round_f16, g.wl_per, uq, ur);
    else
      gemm_few_kernel<K, 1, T><<<grid, 64 * kFewWaves, kGemmLds, st>>>(dst, p, x, t, m, k, nb, ldo, round_f16, g.wl_per, uq, ur);
    return;
  }
  const bool cut = k % (64 * (kRowsWaves / g.RG)) != 0;
#define QTIP_ROWS(NBV, RGV)                                                                                        \
  (cut ? gemm_rows_kernel<K, NBV, RGV, true, T> : gemm_rows_kernel<K, NBV, RGV, false, T>)                        \
      <<<grid, 64 * kRowsWaves, kGemmLds, st>>>(dst, p, x, t, m, k, nb, g.nbt, ldo, round_f16, g.wl_per, uq, ur)
  if (g.NB == 8) {
    if (g.RG == 8) QTIP_ROWS(8, 8);
    else QTIP_ROWS(8, 4);
  } else if (g.NB == 6) {
    QTIP_ROWS(6, 8);
  } else if (g.NB == 4) {
    if (g.RG == 8) QTIP_ROWS(4, 8);
    else if (g.RG == 4) QTIP_ROWS(4, 4);
    else QTIP_ROWS(4, 2);
  } else {
    if (g.RG == 4) QTIP_ROWS(2, 4);
    else QTIP_ROWS(2, 2);
  }
#undef QTIP_ROWS
}

template <typename T>
void launch_gemm(int bits, const GemmPlan& g, T* dst, long ldo, const uint8_t* p, const uint16_t* x, const uint32_t* t,
                 int m, int k, int nb, int round_f16, int cus, hipStream_t st) {
  switch (bits) {
    case 2: return launch_gemm<2, T>(g, dst, ldo, p, x, t, m, k, nb, round_f16, cus, st);
    case 3: return launch_gemm<3, T>(g, dst, ldo, p, x, t, m, k, nb, round_f16, cus, st);
    default: return launch_gemm<4, T>(g, dst, ldo, p, x, t, m, k, nb, round_f16, cus, st);
  }
}

template <typename TOut, bool kFine = true>
int run_gemm(TOut* out, const void* packed, const void* x_f16, const void* tlut, int m, int k, int bits, int batch,
                    int round_f16, void* workspace, size_t workspace_bytes, void* stream) {
  int rc = check_common(out, packed, x_f16, tlut, m, k, bits);
  if (rc) return rc;
  if (batch < 1 || batch > 65535) return QTIP_E_SHAPE;
  if (!aligned16(packed) || !aligned16(x_f16) || (reinterpret_cast<uintptr_t>(tlut) & 3u) ||
      (reinterpret_cast<uintptr_t>(out) & (sizeof(TOut) - 1)))
    return QTIP_E_ALIGN;
  int cus = 0;
  rc = qtip_device_ready(stream, &cus);
  if (rc) return rc;
  const bool split = workspace != nullptr;
  if (workspace) {
    if (workspace_bytes < qtip_gemm_scratch(m, k, bits, batch, kFine)) return QTIP_E_WORKSPACE;
    if (!aligned16(workspace)) return QTIP_E_ALIGN;
  }
  hipStream_t st = (hipStream_t)stream;
  auto* t = (const uint32_t*)tlut;
  for (int b0 = 0, nb; b0 < batch; b0 += nb) {
    nb = next_pass(m, k, bits, batch - b0, cus, split, kFine);
    const GemmParts parts = gemm_plan(m, k, bits, nb, cus, split, kFine);
    const uint16_t* xx = (const uint16_t*)x_f16 + (size_t)b0 * k;
    for (int part = 0; part < 2; ++part) {
      const int first = part ? parts.m0 : 0, rows = part ? m - parts.m0 : parts.m0;
      if (!rows) continue;
      const GemmPlan& g = part ? parts.rest : parts.first;
      const uint8_t* p = (const uint8_t*)packed + (size_t)first * k * bits / 8;
      TOut* o = out + (size_t)b0 * m + first;
      if (g.S > 1) launch_gemm<float>(bits, g, (float*)workspace, rows, p, xx, t, rows, k, nb, 0, cus, st);
      else launch_gemm<TOut>(bits, g, o, m, p, xx, t, rows, k, nb, round_f16, cus, st);
      hipError_t le = hipGetLastError();
      if (le != hipSuccess) return (int)le;
      if (g.S > 1) {
        const long n = (long)nb * rows / 4;
        sum_parts_round_kernel<TOut><<<(int)((n + 255) / 256), 256, 0, st>>>(o, (const float4_t*)workspace, n, rows / 4, m,
                                                                             g.S, round_f16);
        le = hipGetLastError();
        if (le != hipSuccess) return (int)le;
      }
    }
  }
  return QTIP_OK;
}

}  // namespace

hipError_t qtip_gemm_allow_lds() {
  hipError_t e;
#define QTIP_ALLOW(fn, bytes)                                                                                    \
  if ((e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize,   \
                               (int)bytes)) != hipSuccess)                                                       \
    return e;
#define QTIP_ALLOW_GEMM(KB, T)                        \
  QTIP_ALLOW((gemm_kernel<KB, 2, false, T>), kGemmLds)  \
  QTIP_ALLOW((gemm_kernel<KB, 2, true, T>), kGemmLds)   \
  QTIP_ALLOW((gemm_few_kernel<KB, 1, T>), kGemmLds)     \
  QTIP_ALLOW((gemm_few_kernel<KB, 2, T>), kGemmLds)     \
  QTIP_ALLOW((gemm_rows_kernel<KB, 8, 8, false, T>), kGemmLds) \
  QTIP_ALLOW((gemm_rows_kernel<KB, 8, 8, true, T>), kGemmLds)  \
  QTIP_ALLOW((gemm_rows_kernel<KB, 8, 4, false, T>), kGemmLds) \
  QTIP_ALLOW((gemm_rows_kernel<KB, 8, 4, true, T>), kGemmLds)  \
  QTIP_ALLOW((gemm_rows_kernel<KB, 6, 8, false, T>), kGemmLds) \
  QTIP_ALLOW((gemm_rows_kernel<KB, 6, 8, true, T>), kGemmLds)  \
  QTIP_ALLOW((gemm_rows_kernel<KB, 4, 8, false, T>), kGemmLds) \
  QTIP_ALLOW((gemm_rows_kernel<KB, 4, 8, true, T>), kGemmLds)  \
  QTIP_ALLOW((gemm_rows_kernel<KB, 4, 4, false, T>), kGemmLds) \
  QTIP_ALLOW((gemm_rows_kernel<KB, 4, 4, true, T>), kGemmLds)  \
  QTIP_ALLOW((gemm_rows_kernel<KB, 4, 2, false, T>), kGemmLds) \
  QTIP_ALLOW((gemm_rows_kernel<KB, 4, 2, true, T>), kGemmLds)  \
  QTIP_ALLOW((gemm_rows_kernel<KB, 2, 4, false, T>), kGemmLds) \
  QTIP_ALLOW((gemm_rows_kernel<KB, 2, 4, true, T>), kGemmLds)  \
  QTIP_ALLOW((gemm_rows_kernel<KB, 2, 2, false, T>), kGemmLds) \
  QTIP_ALLOW((gemm_rows_kernel<KB, 2, 2, true, T>), kGemmLds)
  QTIP_ALLOW_GEMM(2, float)
  QTIP_ALLOW_GEMM(3, float)
  QTIP_ALLOW_GEMM(4, float)
  QTIP_ALLOW_GEMM(2, _Float16)
  QTIP_ALLOW_GEMM(3, _Float16)
  QTIP_ALLOW_GEMM(4, _Float16)
#define QTIP_ALLOW_SHARED(KB, CUTV)                     \
  QTIP_ALLOW((gemm_kernel<KB, 1, CUTV, float>), kGemmLds) \
  QTIP_ALLOW((gemm_kernel<KB, 1, CUTV, _Float16>), kGemmLds)
  QTIP_ALLOW_SHARED(3, false)
  QTIP_ALLOW_SHARED(3, true)
  QTIP_ALLOW_SHARED(4, false)
  QTIP_ALLOW_SHARED(4, true)
#undef QTIP_ALLOW_SHARED
#undef QTIP_ALLOW_GEMM
#undef QTIP_ALLOW
  return hipSuccess;
}

int qtip_gemm_ranges(int m, int k, int bits, int batch, bool fine) {
  const int cus = qtip_device_cus();
  if (!cus || next_pass(m, k, bits, batch, cus, true, fine) != batch) return 1;
  const GemmParts p = gemm_plan(m, k, bits, batch, cus, true, fine);
  return p.m0 == m ? p.first.S : 1;
}

int qtip_gemm_parts(float* parts, int nparts, const void* packed, const void* x_f16, const void* tlut, int m, int k, int bits,
                    int batch, bool fine, void* stream) {
  int rc = check_common(parts, packed, x_f16, tlut, m, k, bits);
  if (rc) return rc;
  if (!aligned16(packed) || !aligned16(x_f16) || !aligned16(parts) || (reinterpret_cast<uintptr_t>(tlut) & 3u)) return QTIP_E_ALIGN;
  int cus = 0;
  rc = qtip_device_ready(stream, &cus);
  if (rc) return rc;
  if (next_pass(m, k, bits, batch, cus, true, fine) != batch) return QTIP_E_SHAPE;
  const GemmParts p = gemm_plan(m, k, bits, batch, cus, true, fine);
  if (p.m0 != m || p.first.S < 2 || p.first.S != nparts) return QTIP_E_SHAPE;
  launch_gemm<float>(bits, p.first, parts, m, (const uint8_t*)packed, (const uint16_t*)x_f16, (const uint32_t*)tlut, m, k, batch, 0, cus,
                     (hipStream_t)stream);
  return (int)hipGetLastError();
}

size_t qtip_gemm_scratch(int m, int k, int bits, int batch, bool fine) {
  if (m <= 0 || k <= 0 || (m & 31) || (k & 31) || bits < 2 || bits > 4 || batch < 1) return 0;
  const int cus = qtip_device_cus();
  if (!cus) return 0;
  size_t need = 0;
  for (int b0 = 0, nb, seen = 0; b0 < batch; b0 += nb) {
    nb = next_pass(m, k, bits, batch - b0, cus, true, fine);
    if (nb == seen) continue;
    seen = nb;
    const GemmParts p = gemm_plan(m, k, bits, nb, cus, true, fine);
    for (size_t bytes : {parts_bytes(p.first, p.m0, nb), p.m0 < m ? parts_bytes(p.rest, m - p.m0, nb) : 0})
      need = bytes > need ? bytes : need;
  }
  return need;
}

extern "C" {

size_t qtip_gemm_workspace_bytes(int m, int k, int bits, int batch) { return qtip_gemm_scratch(m, k, bits, batch, true); }

size_t qtip_gemm_long_workspace_bytes(int m, int k, int bits, int batch) { return qtip_gemm_scratch(m, k, bits, batch, false); }

int qtip_decompress_gemm(float* out, const void* packed, const void* x_f16, const void* tlut, int m, int k, int bits,
                         int batch, int round_f16, void* workspace, size_t workspace_bytes, void* stream) {
  return run_gemm<float>(out, packed, x_f16, tlut, m, k, bits, batch, round_f16, workspace, workspace_bytes, stream);
}

int qtip_decompress_gemm_f16(void* out_f16, const void* packed, const void* x_f16, const void* tlut, int m, int k, int bits,
                             int batch, void* workspace, size_t workspace_bytes, void* stream) {
  return run_gemm<_Float16>((_Float16*)out_f16, packed, x_f16, tlut, m, k, bits, batch, 1, workspace, workspace_bytes,
                            stream);
}

int qtip_decompress_gemm_long_f16(void* out_f16, const void* packed, const void* x_f16, const void* tlut, int m, int k,
                                  int bits, int batch, void* workspace, size_t workspace_bytes, void* stream) {
  return run_gemm<_Float16, false>((_Float16*)out_f16, packed, x_f16, tlut, m, k, bits, batch, 1, workspace, workspace_bytes,
                                   stream);
}

}  // extern "C"
