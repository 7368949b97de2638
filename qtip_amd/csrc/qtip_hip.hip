// libqtip_hip.so: gfx950 kernels and C ABI for QTIP's quantized-linear
// inference path.  Declarations and the reference interfaces each entry
// point replaces are in include/qtip_hip.h.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <mutex>
#include <type_traits>

#include "../../include/qtip_hip.h"
#include "qtip_device.h"
#include "qtip_matvec_half.h"
#include "qtip_setup.h"
#include "qtip_shares.h"
#include "qtip_wht.h"

#ifdef QTIP_STAMPS  // (the timeline build, see QTIP_STAMP)
// inside the layer boundary of the prologue (sv = the kernel's stamp_v): 6 entered, 7 / 8 / 9 past its
// first / second / third barrier (first transform, RMSNorm sum, second transform), 10 left
#define QTIP_STAMP_SV(i) if (wave == 0 && sv) sv[i] = __builtin_amdgcn_s_memrealtime();
#endif
#include "qtip_chain.h"
#include "qtip_mix.h"

using namespace qtip;
using namespace qtip_chain;

namespace {

// kThreads = 1024: 16 waves per workgroup, one workgroup per CU
constexpr int kMaxSplit = 16;
constexpr int kApartShift = 16;  // upw_r of half units that lie apart holds their workgroups and, from this bit on, half_apart

__device__ __forceinline__ float dpp_xor1(float v) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1 /* quad_perm 1,0,3,2 */,
                                         0xF, 0xF, false));
}
// ---------------------------------------------------------------------------
// decode: packed stream -> dense fp16 (m, k)
//
// Write-bound (2 bytes out per K/8 bytes in), so what matters is the shape of the stores.  A lane
// decodes 4-column pieces of 16 different rows; stored as they come, a row of the matrix receives
// 8 bytes per lane and the memory system sees partial cache lines (measured 2.4 TB/s against
// 6.9 TB/s for a fill).  Each wave therefore turns its wave-load (32 rows x 128 columns) round
// in LDS, a quarter (8 rows x 256 bytes) at a time: pieces go in with the 16-byte chunk index
// xor-ed with the row (conflict free both ways), come back as one 16-byte chunk per lane, and a
// store instruction writes four 256-byte row segments - whole cache lines only.  The 128 KiB
// table of the matvec (32 replicas, one bank per lane) serves the lookups; the next wave-load
// of the stream is requested before the current one is decoded.
// ---------------------------------------------------------------------------
constexpr size_t kDecodeLds = kLut128Bytes + kWaves * 2048;

template <int K>
__global__ __launch_bounds__(kThreads, 1) void decode_kernel(uint16_t* __restrict__ out,
                                                             const uint8_t* __restrict__ packed,
                                                             const uint32_t* __restrict__ tlut,
                                                             int m, int k) {
  extern __shared__ __align__(16) uint8_t smem[];
  uint32_t* lut = reinterpret_cast<uint32_t*>(smem);
  build_lut128(lut, tlut, threadIdx.x, kThreads);
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int a = lane & 15, g = lane >> 4;
  const uint32_t slot4 = lds_address(lut) + ((uint32_t)(lane & 31) << 2);
  uint8_t* stage = smem + kLut128Bytes + wave * 2048;  // this wave's [8 rows][256 bytes]
  const int nkb = k >> 5;
  const int nwl = (nkb + 3) >> 2;
  const long total = (long)(m >> 5) * nwl;  // wave-loads in the matrix
  const size_t rb_bytes = (size_t)nkb * 128 * K;
  const long step = (long)gridDim.x * kWaves;
  auto fetch = [&](long ww) {
    const long wc = ww < total ? ww : total - 1;
    const int rb = (int)(wc / nwl), wl = (int)(wc - (long)rb * nwl);
    int kb = 4 * wl + g;
    kb = kb < nkb ? kb : nkb - 1;  // blocks past the row's end (k / 32 not a multiple of 4) are decoded but not stored
    return load_lane<K>(packed + (size_t)rb * rb_bytes + (size_t)kb * 128 * K + a * 8 * K);
  };
  // The stream is requested NB wave-loads ahead.  (Loads and stores share one in-order completion
  // counter, so a wait for a requested wave-load also waits for the stores issued before the
  // request; requesting 2, 4 or 8 wave-loads at a time to meet that wait less often measured no
  // faster - the memory system, not the wave, holds the stores back.)
  constexpr int NB = 1;
  long w = (long)blockIdx.x * kWaves + wave;
  LaneData<K> cur[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) cur[b] = fetch(w + b * step);
  // piece (kh, jh) of this lane inside a quarter, and the chunk it reads back
  const int r8 = a >> 1;
  const int row_rd = lane >> 4, c_rd = lane & 15;
  for (; w < total; w += NB * step) {
    LaneData<K> nxt[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) nxt[b] = fetch(w + (NB + b) * step);
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const long wb = w + b * step;
      if (wb >= total) break;  // the same for every lane of the wave
      const int rb = (int)(wb / nwl), wl = (int)(wb - (long)rb * nwl);
      uint32_t P[16], W[32];
      packed_states<K>(cur[b], P);
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const uint32_t q = pk_hash(P[i]) & 0xFFC0FFC0u;
        W[2 * i] = lds_word_abs(lut128_addr_lo(q, slot4));
        W[2 * i + 1] = lds_word_abs(lut128_addr_hi(q, slot4));
      }
      const bool store_ok = 4 * wl + (c_rd >> 2) < nkb;
#pragma unroll
      for (int mh = 0; mh < 2; ++mh)
#pragma unroll
        for (int rh = 0; rh < 2; ++rh) {
#pragma unroll
          for (int kh = 0; kh < 2; ++kh)
#pragma unroll
            for (int jh = 0; jh < 2; ++jh) {
              const int t = 2 * kh + mh, j = 2 * jh + rh;
              const int chunk = 4 * g + 2 * kh + jh;
              u32x2 v = {W[w_index<K>(0, t, j)], W[w_index<K>(1, t, j)]};
              *reinterpret_cast<u32x2*>(stage + r8 * 256 + ((chunk ^ r8) << 4) + 8 * (a & 1)) = v;
            }
          // the wave reads what its other lanes wrote: LDS serves a wave's requests in order
          __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
          __builtin_amdgcn_wave_barrier();
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            const int r = row_rd + 4 * i;
            const u32x4 v = *reinterpret_cast<const u32x4*>(stage + r * 256 + ((c_rd ^ r) << 4));
            const size_t row = (size_t)rb * 32 + 16 * mh + 8 * rh + r;
            const size_t col = (size_t)wl * 128 + c_rd * 8;
            if (store_ok) __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(out + row * k + col));
          }
          __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
          __builtin_amdgcn_wave_barrier();
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) cur[b] = nxt[b];
  }
}

// ---------------------------------------------------------------------------
// decompress + matvec
// ---------------------------------------------------------------------------
constexpr size_t kMatvecLds = kLut128Bytes + 2 * kWaves * 32 * sizeof(float);
constexpr size_t kMatvecXBytes = 28 * 1024;  // LDS left for the x values of a workgroup's k range

// x for a lane's columns of a wave-load: 4 x (4 consecutive fp16), 16 bytes apart
__device__ __forceinline__ void load_x_buf(__amdgpu_buffer_rsrc_t rsrc, uint32_t voff, uint32_t soff,
                                           u32x2 xv[4]) {
#pragma unroll
  for (int q = 0; q < 4; ++q) xv[q] = __builtin_amdgcn_raw_buffer_load_b64(rsrc, voff + 16 * q, soff, 0);
}

// Input transform of the layer inside the matvec prologue (k = 1024 * EPT a power of two):
// xs[e] = fp16(scale * (H_k (su * x))[e]) for the whole vector, written to LDS where the
// kernel keeps its activations.  Every workgroup computes the whole transform (a few thousand
// butterflies per thread, hidden behind the latency of the first weight loads) - it replaces
// a separate transform launch.  `xchg`: k + k/64 floats.
// Natural to swapped layout (qtip_chain.h).
template <int EPT>
__device__ __forceinline__ void xform_compute(float (&v)[EPT], float scale, float* xchg, _Float16 (&xo)[EPT], int place,
                                              int wave) {
  using namespace qtip_wht;
  wht_regs<EPT>(v);
  wht_places<EPT>(v, 6, place);
  st_f32<EPT>(xchg + xidx<EPT>(nat_index<EPT>(place, wave)), v);
  __syncthreads();
  ld_f32<EPT>(xchg + xidx<EPT>(swp_index<EPT>(place, wave)), v);
  wht_places<EPT>(v, 4, place);
#pragma unroll
  for (int i = 0; i < EPT; ++i) xo[i] = (_Float16)(v[i] * scale);
}

// Transformed activations lie in LDS with 16 bytes between wave-loads: a transform ends in the swapped layout, whose
// sixteen lanes store 64 * EPT elements apart, on one bank without them.
constexpr uint32_t kXsStride = 256 + 16;
// LDS of a matvec with a transform in front: where the table leaves room (k <= 4096) the exchange buffer is beside it
// and the table is written while the operands are on their way; at 8192 it lies under the table, whose first items
// wait for it.
constexpr uint32_t xform_lds_bytes(int k) { return (uint32_t)k / 128 * kXsStride; }
constexpr bool xform_beside(int k) { return k <= 4096; }
constexpr size_t xform_lds(int k) {
  return kMatvecLds + xform_lds_bytes(k) + (xform_beside(k) ? chain_floats(k) * sizeof(float) : 0);
}
constexpr int kLateItems = 3;  // items of 16 KiB of the table that the exchange buffer of 8192 covers
static_assert(qtip_mix::mix_in_lds(qtip_mix::kMixInMaxRows, 4).bytes <= kMatvecLds + kMatvecXBytes - 7 * 16 * kThreads &&
              qtip_mix::mix_in_lds(qtip_mix::kMixInMaxRows, 4).bytes % 16 == 0, "a mix leaves the table but for its last item");
static_assert(xform_lds(4096) <= kMatvecLds + kMatvecXBytes && xform_lds(8192) <= kMatvecLds + kMatvecXBytes &&
              chain_floats(8192) * sizeof(float) <= kLateItems * 16 * kThreads, "the transform's buffers fit");

// XFORM == 2: the whole boundary between two linear layers of a decoder (qtip_chain.h) in front of the matvec, what
// rht_chain_kernel does in a launch of its own.  Every workgroup recomputes the k-point boundary - a few microseconds of
// work on 1024 threads, most of it while the first stream requests are in flight - and workgroup (0, 0) stores x_new for
// the layers that follow.

// Up to three matrices with the same k and bit width in one launch (the separate q / k / v or
// gate / up projections of a decoder layer): the workgroups blockIdx.y in
// [wg_begin[g], wg_begin[g + 1]) serve matrix g with its own stream, table, sign vector and
// output rows; everything else (k split, layer boundary, x_out) is shared.
struct GroupArgs {
  float* dst[3];              // first output row of the matrix inside a partial result
  const uint8_t* packed[3];
  const uint32_t* tlut[3];
  const uint16_t* su[3];
  const uint16_t* x[3];       // the matrices' own inputs (plain form; unused with a layer boundary)
  int m[3];
  int wg_begin[4];
  int upw_q[3], upw_r[3];
  size_t part_stride;         // floats between partial results
};
// Timeline build (-DQTIP_STAMPS, used by `bench.py --timeline` through a library of its own; the
// product library is built without it): waves 0 and 15 of every matvec workgroup keep a few
// readings of the 100 MHz constant clock in registers and wave 0 stores them when it ends, into
// the slot of its launch's shape, so that after a graph replay the buffer holds the last launch
// of every shape.
//   0 first instruction   1 table words picked   2 at the first barrier   3 past it
//   4 end of the kernel   5 first instruction of wave 15   15 first wave-load of wave 0 in registers
//   6-10 the transform / layer boundary of the prologue (see QTIP_STAMP_SV)
// (nothing is read inside the loop: a clock reading there makes every wait in it a full one; and
// only two waves read the clock: 4096 waves reading it at once queue up behind each other)
#ifdef QTIP_STAMPS
constexpr int kStampSlots = 64, kStampWgs = 256, kStampN = 16;
__device__ unsigned long long g_stamps[kStampSlots][kStampWgs][kStampN];
#define QTIP_STAMP_DECL unsigned long long stamp_v[kStampN] = {};
#define QTIP_STAMP(i) if (wave == 0 || (i == 0 && wave == kWaves - 1)) stamp_v[i] = __builtin_amdgcn_s_memrealtime();
#define QTIP_STAMP_FIRST_LOAD() if (wave == 0) { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(DEPTH - 1)); stamp_v[15] = __builtin_amdgcn_s_memrealtime(); }
#define QTIP_STAMP_PTR stamp_v
#else
#define QTIP_STAMP_DECL
#define QTIP_STAMP(i)
#define QTIP_STAMP_FIRST_LOAD()
#define QTIP_STAMP_PTR nullptr
#endif
// (read and selected: left to itself the compiler selects an address and reads there, a round trip more)
__device__ __forceinline__ int pick3(const int (&a)[3], int g) {
  int x = a[0], y = a[1], z = a[2];
  asm("" : "+s"(x), "+s"(y), "+s"(z));
  return g == 0 ? x : (g == 1 ? y : z);
}
template <typename T>
__device__ __forceinline__ T* pick3(T* const (&a)[3], int g) {
  uint64_t x = (uint64_t)a[0], y = (uint64_t)a[1], z = (uint64_t)a[2];
  asm("" : "+s"(x), "+s"(y), "+s"(z));
  // (device memory, which the statement above hides from the compiler)
  return (T*)(__attribute__((address_space(1))) T*)(g == 0 ? x : (g == 1 ? y : z));
}

// Work unit = (32-row block rb, k split s).  The 16 waves of a workgroup take
// the unit's wave-loads round-robin (so the workgroup streams one contiguous
// run of bytes), reduce across the four blocks of a wave-load inside the MFMA, across the two
// column halves with one DPP exchange and across waves through LDS in a fixed order, and store 32 sums to
// dst[s*m + 32*rb ...]: the result itself when S == 1, else one of S partial
// vectors that the consumer adds in order (deterministic either way).
//
// The launcher's grid is (S, workgroups per k range): a workgroup keeps one k range
// [wl0, wl1) and walks row blocks rb0, rb0 + rb_step, ...  A wave sees its work
// as a flat sequence of items (unit i, j) with wave-load wl0 + wave + 16*j;
// every unit has npw items per wave of which the first nvj are real (the same
// count in every unit).  DEPTH items are in flight; the prefetch runs ahead
// across unit boundaries and every load in the loop is unconditional (a
// conditional prefetch makes the compiler wait for it at once): padding items
// use an out-of-range lane offset (the load returns zeros without a memory
// access) and are skipped by the arithmetic.
// XLDS: the x values of the workgroup's k range are staged in LDS once
// (needs 256 bytes per wave-load of the range) and read from there.
// XFORM: 0 = x is the matvec's fp16 input, 1 = x is the layer's raw input (input transform in the
// prologue), 2 = the previous layer's partial results (whole layer boundary in the prologue).
// 3 = as 1, for a table order times a power of two (qtip_mix.h); every workgroup makes the range of the vector that it reads
// and x is staged as in the plain form.  EPT is a sixteenth of the columns there.
// 4 = as 1, on the attention output that the shares of the key ranges give (qtip_shares.h).
// EPT = k / 1024 with 1, 2 and 4, a kernel each: behind a switch over it the compiler waits for everything in flight.
// XHALF: the k range needs up to twice the staging area and every workgroup has exactly one unit:
// x is staged in two halves, the second replacing the first in the middle of the unit (two more
// barriers per launch instead of x travelling through vector loads with every wave-load, which
// made the 28672-wide matrices 15-20 % slower).
// HALF: the row blocks that do not fill a last round of whole units (at most half a round of
// them) are cut by row half instead: a workgroup w < upw_r takes the rows of one rh of one of them after its upw_q whole units.  Such a half unit reads the block's
// whole stream but decodes half of its states (about 0.55 of a unit's time), and its rows are
// complete sums, so nothing has to be combined across workgroups: 320 row blocks on 256
// workgroups take 1.55 units of time instead of 2, 128 row blocks 0.55 instead of 1.
// HALF = 1: the halves of a block lie side by side, 2: 1 << half_apart workgroups apart, but for the last ones, less than a round of pairs
// (a form of its own: its dozen scalar instructions in a row in front of the first stream load cost the other 1 to 2 %).
template <int K, int DEPTH, bool XLDS, int XFORM = 0, bool XHALF = false, bool GROUP = false, int HALF = 0,
          int EPT = 0>
__global__ __launch_bounds__(kThreads, 1) void matvec_kernel(
    float* __restrict__ dst_, const uint8_t* __restrict__ packed_, const uint16_t* __restrict__ x_,
    const uint32_t* __restrict__ tlut_, int m_, int k_, int wl_per, int upw_q_, int upw_r_,
    const uint16_t* __restrict__ su_ = nullptr, float xscale = 1.f, const ChainArgs chain = ChainArgs{},
    const GroupArgs grp = GroupArgs{}, const qtip_mix::MixArgs mix = qtip_mix::MixArgs{},
    const qtip_shares::ShareArgs sh = qtip_shares::ShareArgs{}) {
  static_assert(!XFORM || XLDS, "the transformed activations live in LDS");
  static_assert((XFORM != 0) == (EPT != 0), "a transform in front knows its size");
  constexpr bool POW2 = XFORM != 0 && XFORM != 3;  // the whole transformed vector, in padded wave-loads
  const int k = POW2 ? 1024 * EPT : k_;
  static_assert(!GROUP || XFORM == 2 || (XFORM == 0 && XLDS && !XHALF),
                "grouped launches exist for the layer-boundary form and the plain form with x in LDS");
  // the matrix this workgroup serves (uniform: scalar selects on kernel arguments)
  int gi = 0;
  if constexpr (GROUP) gi = (int)blockIdx.y >= grp.wg_begin[2] ? 2 : ((int)blockIdx.y >= grp.wg_begin[1] ? 1 : 0);
  float* __restrict__ dst = GROUP ? pick3(grp.dst, gi) : dst_;
  const uint8_t* __restrict__ packed = GROUP ? pick3(grp.packed, gi) : packed_;
  const uint32_t* __restrict__ tlut = GROUP ? pick3(grp.tlut, gi) : tlut_;
  const uint16_t* __restrict__ su = GROUP ? pick3(grp.su, gi) : su_;
  const uint16_t* __restrict__ x = (GROUP && XFORM == 0) ? pick3(grp.x, gi) : x_;
  const int m = GROUP ? pick3(grp.m, gi) : m_;
  const int upw_q = GROUP ? pick3(grp.upw_q, gi) : upw_q_;
  const int upw_r = GROUP ? pick3(grp.upw_r, gi) : (HALF == 2 ? upw_r_ & ((1 << kApartShift) - 1) : upw_r_);
  static_assert(!XHALF || (XLDS && !XFORM), "two-half staging is a form of the plain staged x");
  static_assert(!HALF || (XLDS && !POW2 && !XHALF && !GROUP), "half units exist for the plain form with x in LDS and behind a mix");
  // wave-loads requested before the table is built.  With half units both: a half wave-load is
  // decoded in half the time, which no longer covers the latency of a load requested after the barrier.
  constexpr int FIRST = (DEPTH > 2 || HALF) ? 2 : 1;
  extern __shared__ __align__(16) uint8_t smem[];
  uint32_t* lut = reinterpret_cast<uint32_t*>(smem);
  float* part = reinterpret_cast<float*>(smem + kLut128Bytes);  // [2][kWaves][32]
  uint8_t* xs_lds = smem + kLut128Bytes + 2 * kWaves * 32 * sizeof(float);  // [wl_per][256] when XLDS
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform, lives in an SGPR
  QTIP_STAMP_DECL
  QTIP_STAMP(0)
  const int a = lane & 15, g = lane >> 4;
  const uint32_t slot4 = lds_address(lut) + ((uint32_t)(lane & 31) << 2);
  const int nkb = k >> 5;
  const int nwl = (nkb + 3) >> 2;  // wave-loads per row block, the last may be partial
  const int nfull = nkb >> 2;      // full wave-loads per row block
  const int nrb = m >> 5;
  const uint32_t rb_bytes = (uint32_t)nkb * 128 * K;
  constexpr uint32_t WL_BYTES = 512 * K;
  const uint32_t loff = (uint32_t)lane * 8 * K;                // lane's bytes inside a wave-load
  const uint32_t xoff = (uint32_t)(32 * g + 4 * (a & 1)) * 2;  // lane's x bytes inside a wave-load

  // grid = (S, workgroups per k range): no integer division on the way to the first loads
  const int s = blockIdx.x;
  const int wg0 = GROUP ? (gi == 0 ? 0 : (gi == 1 ? grp.wg_begin[1] : grp.wg_begin[2])) : 0;
  const int rb0 = (int)blockIdx.y - wg0;
  const int rb_step = GROUP ? (gi == 0 ? grp.wg_begin[1] : (gi == 1 ? grp.wg_begin[2] : grp.wg_begin[3])) - wg0
                            : (int)gridDim.y;
  const int wl0 = s * wl_per;
  const int wl1 = wl0 + wl_per < nwl ? wl0 + wl_per : nwl;
  const int wl1f = wl1 < nfull ? wl1 : nfull;           // end of the full wave-loads
  const int npw = (wl_per + kWaves - 1) / kWaves;       // items per wave and unit (padded)
  // whole units of this workgroup: ceil((nrb - rb0) / rb_step), quotient and remainder from the host;
  // with HALF the remainder counts half units instead
  const int upw = HALF ? upw_q : upw_q + (rb0 < upw_r ? 1 : 0);
  const int T_full = upw * npw;
  const bool has_half = HALF && rb0 < upw_r;
  const int apart = HALF == 2 ? upw_r_ >> kApartShift : 0;
  const int lg = HALF == 2 && rb0 < (upw_r >> (apart + 1)) << (apart + 1) ? apart : 0;
  const int half_rh = (rb0 >> lg) & 1;
  const int half_rb = upw_q * rb_step + (HALF == 2 ? ((rb0 >> (lg + 1)) << lg) + (rb0 & ((1 << lg) - 1)) : rb0 >> 1);
  const int T = T_full + (has_half ? npw : 0);
  const int w_first = wl0 + wave;
  const int nvj = w_first < wl1f ? (wl1f - w_first + kWaves - 1) / kWaves : 0;  // real items per unit
  const bool tail_wave = wl1 > nfull && ((nfull - wl0) % kWaves) == wave;
  float* out_s = dst + (size_t)s * (GROUP ? grp.part_stride : (size_t)m);

  const __amdgpu_buffer_rsrc_t rs_w = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(packed), 0, (int)((size_t)nrb * rb_bytes), 0x00020000);
  const __amdgpu_buffer_rsrc_t rs_x =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(x), 0, k * 2, 0x00020000);

  // load cursor: unit l_i (row block l_rb), item l_j
  int l_j = 0, l_t = 0;
  uint32_t l_rboff = (uint32_t)((HALF && upw == 0) ? half_rb : rb0) * rb_bytes;
  const uint32_t rb_step_bytes = (uint32_t)rb_step * rb_bytes;
  LaneData<K> buf[DEPTH];
  u32x2 xbuf[XLDS ? 1 : DEPTH][4];
  auto issue = [&](int d) {
    const bool valid = l_j < nvj && l_t < T;
    const uint32_t wl = (uint32_t)(w_first + l_j * kWaves);
    const uint32_t woff = valid ? l_rboff + wl * WL_BYTES : 0u;
    const uint32_t xw = valid ? wl * 256u : 0u;
    // padding items: a lane offset past the end of the descriptor returns zeros without touching
    // memory (reading offset 0 instead cost the small shapes up to 2 us: thousands of waves
    // hammering the same few cache lines)
    buf[d] = load_lane_buf<K>(rs_w, valid ? loff : 0x7FFFFF00u, woff);
    if constexpr (!XLDS) load_x_buf(rs_x, valid ? xoff : 0x7FFFFF00u, xw, xbuf[d]);
    ++l_t;
    if (++l_j == npw) {
      l_j = 0;
      l_rboff = (HALF && l_t == T_full) ? (uint32_t)half_rb * rb_bytes : l_rboff + rb_step_bytes;
    }
  };
  // Prologue loads in the order they are needed: the table words and x first, then the first
  // FIRST wave-loads of the stream; the other DEPTH - FIRST follow once the table is built and the
  // workgroup is past its barrier.  A CU serves requests in order from a finite queue: with all
  // DEPTH wave-loads of all 16 waves requested up front (25 MB over the chip at K = 2) the last
  // waves stall on issuing theirs until most of that data has arrived, and reach the table they
  // have yet to write - and the barrier every wave waits at - thousands of cycles late.
  // (Measured: 2 before / rest after is 3-10 % faster than all before on every shape tried; 1, 3
  // and 4 before are in between.)
  static_assert(kLutEntries * 8 == 8 * kThreads, "table build assumes 8 16-byte items per thread");
  uint32_t tw[4];  // item it*1024 + tid belongs to entry it*128 + tid/8; entries e and e+512 share a word
  // the wave's eight words of a pass come through the scalar cache (uniform address), which
  // keeps them out of the vector-memory queue that the stream requests fill
  if constexpr (!XFORM) {
#pragma unroll
    for (int it = 0; it < 4; ++it) {
      const uint32_t* tp = tlut + it * 128 + wave * 8;
      // one 32-byte scalar load (the table needs dword alignment only).  Loaded word by word, the
      // compiler may fold the first select below into a per-lane load of tp[lane >> 3], and the wait
      // for that vector load also waits for the stream loads requested before it.
      typedef uint32_t u32x8_dw __attribute__((ext_vector_type(8), aligned(4)));
      const u32x8_dw sw = *reinterpret_cast<const u32x8_dw*>(tp);
      uint32_t v = sw[0];
#pragma unroll
      for (int j = 1; j < 8; ++j) v = ((lane >> 3) == j) ? sw[j] : v;
      tw[it] = v;
    }
  }
  QTIP_STAMP(1)
  u32x4 xstage[2] = {{0u, 0u, 0u, 0u}, {0u, 0u, 0u, 0u}};
  u32x4 xstage2[XHALF ? 2 : 1] = {};
  const int jh = XHALF ? (npw + 1) >> 1 : npw;  // items per wave served by the first staging
  // wave-loads of the first staging (all of the range unless XHALF)
  const int wlx = XHALF ? ((wl1 - wl0) < jh * kWaves ? (wl1 - wl0) : jh * kWaves) : (wl1 - wl0);
  if constexpr (XLDS && !XFORM) {
    // x of wave-loads [wl0, wl0 + wlx): 16 bytes per thread and pass, at most 2 passes (28 KiB)
    const int xbytes = wlx * 256;
    const int kbytes = k * 2;
#pragma unroll
    for (int ps = 0; ps < 2; ++ps) {
      const int o = (ps * kThreads + tid) * 16;
      if (o < xbytes && wl0 * 256 + o < kbytes)
        xstage[ps] = *reinterpret_cast<const u32x4*>(reinterpret_cast<const uint8_t*>(x) + (size_t)wl0 * 256 + o);
    }
    if constexpr (XHALF) {
      const int xbytes2 = (wl1 - wl0 - wlx) * 256;
      const int base2 = (wl0 + wlx) * 256;
#pragma unroll
      for (int ps = 0; ps < 2; ++ps) {
        const int o = (ps * kThreads + tid) * 16;
        if (o < xbytes2 && base2 + o < kbytes)
          xstage2[ps] = *reinterpret_cast<const u32x4*>(reinterpret_cast<const uint8_t*>(x) + (size_t)base2 + o);
      }
    }
  }
  auto table_item = [&](int it) {
    const uint32_t w = tw[it & 3] ^ ((uint32_t)(it >> 2) << 15);
    const u32x4 v = {w, w, w, w};
    reinterpret_cast<u32x4*>(lut)[it * kThreads + tid] = v;
  };
  if constexpr (XFORM == 3) {
#pragma unroll
    for (int it = 0; it < 4; ++it) tw[it] = tlut[it * 128 + (tid >> 3)];
    const int row0 = wl0 * (8 / EPT), row1 = wl1 * (8 / EPT);  // of the range
    qtip_mix::MixInRegs<EPT> r;
    const _Float16* xr = reinterpret_cast<const _Float16*>(x);
    const _Float16* sr = reinterpret_cast<const _Float16*>(su);
    qtip_mix::mix_in_load<EPT>(r, mix, xr, sr, row0, tid);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int d = 0; d < FIRST; ++d) issue(d);
    // The transform's buffers end where the LDS does: on the staging area and the waves' sums, which are free, and, from 224
    // rows of 64 on, a part of the table's last item, which is written behind the transform then.
    const int buffers = (int)(kMatvecLds + kMatvecXBytes) - qtip_mix::mix_in_lds(mix.on, EPT).bytes;
    const bool all = buffers >= 8 * 16 * kThreads;
#pragma unroll
    for (int it = 0; it < 7; ++it) table_item(it);
    if (all) table_item(7);
    __builtin_amdgcn_sched_barrier(0);
    qtip_mix::mix_in_compute<EPT>(r, mix, xscale, smem + buffers, reinterpret_cast<_Float16*>(xs_lds), xr, sr, row0, row1, tid,
                                  QTIP_STAMP_PTR);
    QTIP_STAMP(10)
    if (!all) table_item(7);
  } else if constexpr (XFORM) {
    constexpr bool BESIDE = xform_beside(1024 * EPT);
    const int place = qtip_wht::wht_place(lane);
    // (vector loads: the scalar ones of the plain form are four round trips in a row where registers are short)
#pragma unroll
    for (int it = 0; it < 4; ++it) tw[it] = tlut[it * 128 + (tid >> 3)];
    const _Float16* sr = reinterpret_cast<const _Float16*>(su);
    float* xbuf = reinterpret_cast<float*>(BESIDE ? xs_lds + xform_lds_bytes(1024 * EPT) : smem);
    _Float16 xo[EPT];
    auto requested = [&] {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int d = 0; d < FIRST; ++d) issue(d);
#pragma unroll
      for (int it = BESIDE ? 0 : kLateItems; it < 8; ++it) table_item(it);
      __builtin_amdgcn_sched_barrier(0);  // (the table's writes wait for its words only)
      QTIP_STAMP(6)
    };
    if constexpr (XFORM == 2) {
      ChainRegs<EPT> cr;
      chain_load<EPT>(chain, sr, place, wave, cr);
      requested();
      chain_compute<EPT>(cr, chain, xscale, xbuf, xo, lane, place, wave, blockIdx.x == 0 && blockIdx.y == 0, QTIP_STAMP_PTR);
    } else if constexpr (XFORM == 4) {
      typedef _Float16 hvec __attribute__((ext_vector_type(EPT)));
      const int e = nat_index<EPT>(place, wave), dim = 1 << sh.log_dim, step = qtip_shares::floats(dim);
      const float* w = sh.shares + (size_t)(e >> sh.log_dim) * sh.ranges * step;
      const int d = e & (dim - 1);
      const hvec sv = *reinterpret_cast<const hvec*>(sr + e);
      constexpr int R = qtip_shares::kMaxRanges;
      float o[R][EPT] = {};
      float2 ml[R] = {};
      qtip_wht::ld_f32<EPT>(w + d, o[0]);
      ml[0] = *reinterpret_cast<const float2*>(w + dim);
      const int pos = (int)sh.pos[0], nkeys = pos + 1 < sh.max_len ? pos + 1 : sh.max_len;
      const int used = qtip_shares::active(nkeys, sh.ranges, k >> sh.log_dim);
      if (used > 1) {  // (the position is as far away as the first share: short contexts wait for nothing more)
#pragma unroll
        for (int z = 1; z < R; ++z) {
          const float* wz = w + (z < used ? z : 0) * step;
          qtip_wht::ld_f32<EPT>(wz + d, o[z]);
          ml[z] = *reinterpret_cast<const float2*>(wz + dim);
        }
      }
      requested();
      float v[EPT];
      if (used == 1) {
        const float f = 1.f / ml[0].y;
#pragma unroll
        for (int i = 0; i < EPT; ++i) v[i] = (float)(_Float16)(o[0][i] * f) * (float)sv[i];
      } else {
        float M = ml[0].x;
#pragma unroll
        for (int z = 1; z < R; ++z) M = z < used ? fmaxf(M, ml[z].x) : M;
        float num[EPT] = {}, den = 0.f;
#pragma unroll
        for (int z = 0; z < R; ++z) {
          const float f = z < used && ml[z].x != -INFINITY ? __expf(ml[z].x - M) : 0.f;
          den += z < used ? f * ml[z].y : 0.f;
#pragma unroll
          for (int i = 0; i < EPT; ++i) num[i] += z < used ? f * o[z][i] : 0.f;
        }
#pragma unroll
        for (int i = 0; i < EPT; ++i) v[i] = (float)(_Float16)(num[i] / den) * (float)sv[i];
      }
      xform_compute<EPT>(v, xscale, xbuf, xo, place, wave);
    } else {
      // the raw activations and the sign vector of the layer
      typedef _Float16 hvec __attribute__((ext_vector_type(EPT)));
      const int e = nat_index<EPT>(place, wave);
      const hvec xr = *reinterpret_cast<const hvec*>(reinterpret_cast<const _Float16*>(x) + e);
      const hvec sv = *reinterpret_cast<const hvec*>(sr + e);
      requested();
      float v[EPT];
#pragma unroll
      for (int i = 0; i < EPT; ++i) v[i] = (float)xr[i] * (float)sv[i];
      xform_compute<EPT>(v, xscale, xbuf, xo, place, wave);
    }
    const int e = swp_index<EPT>(place, wave);
    qtip_wht::st_f16<EPT>(reinterpret_cast<_Float16*>(xs_lds) + e + 8 * (e >> 7), xo);
    QTIP_STAMP(10)
    if constexpr (!BESIDE) {
      __syncthreads();  // the exchange buffer has been read
#pragma unroll
      for (int it = 0; it < kLateItems; ++it) table_item(it);
    }
  } else {
#pragma unroll
    for (int d = 0; d < FIRST; ++d) issue(d);
#pragma unroll
    for (int it = 0; it < 8; ++it) table_item(it);
  }
  if constexpr (XLDS && !XFORM) {
    const int xbytes = wlx * 256;
#pragma unroll
    for (int ps = 0; ps < 2; ++ps) {
      const int o = (ps * kThreads + tid) * 16;
      if (o < xbytes) *reinterpret_cast<u32x4*>(xs_lds + o) = xstage[ps];
    }
  }
  QTIP_STAMP(2)
  __syncthreads();
  QTIP_STAMP(3)
#pragma unroll
  for (int d = FIRST; d < DEPTH; ++d) issue(d);
  QTIP_STAMP_FIRST_LOAD()

  // wave-load w_first (the transformed vector is stored whole, a staged one from wl0 on)
  constexpr uint32_t xs_stride = POW2 ? kXsStride : 256u;
  const uint32_t xs_lane = lds_address(xs_lds) + xoff + (uint32_t)(POW2 ? w_first : wave) * xs_stride;

  float4_t acc[4];  // [2*mh + rh]: rows 16*mh + 8*rh + a/2 of the unit's 32-row block
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i] = float4_t{0.f, 0.f, 0.f, 0.f};
  int parity = 0, c_j = 0, c_rb = (HALF && upw == 0) ? half_rb : rb0;
  int c_jbase = 0;  // first item of the staging that is in LDS
  int prio_phase = wave >> 2;  // waves w, w + 4, w + 8, w + 12 share a SIMD
  // items [t0, t1) of the workgroup's item sequence, decoding all states (RH = -1) or one row half.
  // Whole and half units run in loops of their own: with both forms behind a branch in one loop
  // body the compiler loses track of the loads in flight and waits for all of them at every item.
  auto run = [&](auto rh_tag, const int t0, const int t1) {
  constexpr int RH = decltype(rh_tag)::value;
  auto accumulate = [&](const LaneData<K>& ld, const u32x2 xv[4]) {
    matvec_accumulate<K, RH>(ld, xv, slot4, acc);
  };
  for (int t = t0; t < t1; t += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      // The hardware serves the waves of a SIMD oldest first, so the oldest finishes its share of a
      // unit long before the youngest and the SIMD ends every unit on too few waves to hide
      // latencies: the top issue priority rotates through the four waves, item by item.
      switch ((prio_phase++) & 3) {
        case 0: __builtin_amdgcn_s_setprio(0); break;
        case 1: __builtin_amdgcn_s_setprio(1); break;
        case 2: __builtin_amdgcn_s_setprio(2); break;
        default: __builtin_amdgcn_s_setprio(3); break;
      }
      if (t + d < t1) {
        if (c_j < nvj) {
          if constexpr (XLDS) {
            typedef __attribute__((address_space(3))) const u32x2 lds_u32x2_t;
            u32x2 xv[4];
            const uint32_t xa = xs_lane + (uint32_t)(c_j - c_jbase) * (kWaves * xs_stride);
#pragma unroll
            for (int q = 0; q < 4; ++q) xv[q] = *(lds_u32x2_t*)(uintptr_t)(xa + 16u * q);
            accumulate(buf[d], xv);
          } else {
            accumulate(buf[d], xbuf[d]);
          }
        }
      }
      // the stage's registers are refilled only after their last use, so the
      // refill reuses them in place (no copies, no wait on the new load)
      issue(d);
      if (t + d < t1) ++c_j;
      if constexpr (XHALF) {
        // middle of the (only) unit: every wave has read its last x of the first half
        if (t + d < t1 && c_j == jh && jh < npw) {
          __syncthreads();
          const int xbytes2 = (wl1 - wl0 - wlx) * 256;
#pragma unroll
          for (int ps = 0; ps < 2; ++ps) {
            const int o = (ps * kThreads + tid) * 16;
            if (o < xbytes2) *reinterpret_cast<u32x4*>(xs_lds + o) = xstage2[ps];
          }
          __syncthreads();
          c_jbase = jh;
        }
      }
      if (t + d < t1 && c_j == npw) {
        // ---- end of a unit: ragged tail, reductions, store
        // k/32 not a multiple of 4: one wave takes the partial wave-load.  Every lane takes part
        // in an MFMA, so the lanes of the missing tile blocks (g >= nkb % 4) load x and the stream
        // with a lane offset that is out of range by itself: both come back as zeros without a
        // memory access, whatever the range check makes of the scalar offset.
        if (tail_wave) {
          const bool in_row = g < nkb - 4 * nfull;
          u32x2 xt[4];
          load_x_buf(rs_x, in_row ? xoff : 0x7FFFFF00u, (uint32_t)nfull * 256u, xt);
          const LaneData<K> tail = load_lane_buf<K>(rs_w, in_row ? loff : 0x7FFFFF00u,
                                                    (uint32_t)c_rb * rb_bytes + (uint32_t)nfull * WL_BYTES);
          accumulate(tail, xt);
        }
        float* pp = part + parity * (kWaves * 32);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          // element a % 2 holds the lane's sum over the four blocks: an even lane adds its element 0
          // and element 1 of its odd neighbour (the other column half).  Written without a
          // per-lane choice of the element on purpose: with `v = odd ? e1 : e0; v += exchange(v)`
          // the compiler, knowing that only even lanes store, fed e0 into the exchange for every lane.
          const float v = acc[i][0] + dpp_xor1(acc[i][1]);
          acc[i] = float4_t{0.f, 0.f, 0.f, 0.f};
          if (g == 0 && (a & 1) == 0) pp[wave * 32 + (i >> 1) * 16 + (i & 1) * 8 + (a >> 1)] = v;
        }
        __syncthreads();
        // (a half unit owns the rows 16*mh + 8*rh + 0..7 of its rh only)
        if (tid < 32 && (RH < 0 || ((tid >> 3) & 1) == RH)) {
          float sum = 0.f;
#pragma unroll
          for (int w = 0; w < kWaves; ++w) sum += pp[w * 32 + tid];
          out_s[c_rb * 32 + tid] = sum;
        }
        parity ^= 1;  // the other buffer is free: its readers passed the barrier above
        c_j = 0;
        c_rb = (HALF && t + d + 1 == T_full) ? half_rb : c_rb + rb_step;
      }
    }
  }
  };
  run(std::integral_constant<int, -1>{}, 0, T_full);
  if constexpr (HALF) {
    if (has_half) {
      if (half_rh) run(std::integral_constant<int, 1>{}, T_full, T);
      else run(std::integral_constant<int, 0>{}, T_full, T);
    }
  }
#ifdef QTIP_STAMPS
  {
    QTIP_STAMP(4)
    const int wg = (int)blockIdx.x + (int)gridDim.x * (int)blockIdx.y;
    const int slot = ((m ^ k) >> 10) & (kStampSlots - 1);
    if (wg < kStampWgs && lane == 0) {
      if (wave == 0) {
#pragma unroll
        for (int i = 0; i < kStampN; ++i)
          if (i != 5) g_stamps[slot][wg][i] = stamp_v[i];
      } else if (wave == kWaves - 1) {
        g_stamps[slot][wg][5] = stamp_v[0];
      }
    }
  }
#endif
}

// out[i] = parts[0][i] + parts[1][i] + ... in that order
__global__ __launch_bounds__(256) void sum_parts_kernel(float* __restrict__ out,
                                                        const float* __restrict__ parts, int m,
                                                        int S) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= m) return;
  float sum = parts[i];
  for (int s = 1; s < S; ++s) sum += parts[(size_t)s * m + i];
  out[i] = sum;
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
// Device memory the allocation-free entry point keeps its split-k partial sums in: one copy per
// GPU the library runs on, held until the process ends.  In host code this name is only a handle
// for hipGetSymbolAddress (never a device address): launches take DeviceState::scratch_ptr.
constexpr size_t kScratchFloats = 64 * 1024;  // 256 KiB
static __device__ __align__(256) float scratch[kScratchFloats];


template <typename F>
hipError_t allow_lds(F* fn, size_t bytes) {
  return hipFuncSetAttribute(reinterpret_cast<const void*>(fn),
                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

hipError_t allow_lds_all() {
  hipError_t e;
#define QTIP_ALLOW(fn, bytes) \
  if ((e = allow_lds(fn, bytes)) != hipSuccess) return e;
  QTIP_ALLOW((decode_kernel<2>), kDecodeLds)
  QTIP_ALLOW((decode_kernel<3>), kDecodeLds)
  QTIP_ALLOW((decode_kernel<4>), kDecodeLds)
  QTIP_ALLOW((matvec_kernel<2, 2, false>), kMatvecLds)
  QTIP_ALLOW((matvec_kernel<3, 2, false>), kMatvecLds)
  QTIP_ALLOW((matvec_kernel<4, 2, false>), kMatvecLds)
  QTIP_ALLOW((matvec_kernel<2, 2, true>), kMatvecLds + kMatvecXBytes)
  QTIP_ALLOW((matvec_kernel<3, 2, true>), kMatvecLds + kMatvecXBytes)
  QTIP_ALLOW((matvec_kernel<4, 2, true>), kMatvecLds + kMatvecXBytes)
  QTIP_ALLOW((matvec_kernel<2, 2, true, 0, false, false, 1>), kMatvecLds + kMatvecXBytes)
  QTIP_ALLOW((matvec_kernel<2, 2, true, 0, false, false, 2>), kMatvecLds + kMatvecXBytes)
  QTIP_ALLOW((matvec_kernel<3, 2, true, 0, false, false, 2>), kMatvecLds + kMatvecXBytes)
  QTIP_ALLOW((matvec_kernel<4, 2, true, 0, false, false, 2>), kMatvecLds + kMatvecXBytes)
  QTIP_ALLOW((matvec_kernel<2, 2, true, 0, false, true>), kMatvecLds + kMatvecXBytes)
  QTIP_ALLOW((matvec_kernel<3, 2, true, 0, false, true>), kMatvecLds + kMatvecXBytes)
  QTIP_ALLOW((matvec_kernel<4, 2, true, 0, false, true>), kMatvecLds + kMatvecXBytes)
  QTIP_ALLOW((matvec_kernel<2, 2, true, 0, true>), kMatvecLds + kMatvecXBytes)
  QTIP_ALLOW((matvec_kernel<3, 2, true, 0, true>), kMatvecLds + kMatvecXBytes)
  QTIP_ALLOW((matvec_kernel<4, 2, true, 0, true>), kMatvecLds + kMatvecXBytes)
#define QTIP_ALLOW_XFORM(BITS, EPT)                                                                       \
  QTIP_ALLOW((matvec_kernel<BITS, 2, true, 1, false, false, 0, EPT>), xform_lds(1024 * EPT))           \
  QTIP_ALLOW((matvec_kernel<BITS, 2, true, 2, false, false, 0, EPT>), xform_lds(1024 * EPT))           \
  QTIP_ALLOW((matvec_kernel<BITS, 2, true, 2, false, true, 0, EPT>), xform_lds(1024 * EPT))            \
  QTIP_ALLOW((matvec_kernel<BITS, 2, true, 4, false, false, 0, EPT>), xform_lds(1024 * EPT))
  QTIP_ALLOW_XFORM(2, 2) QTIP_ALLOW_XFORM(2, 4) QTIP_ALLOW_XFORM(2, 8)
  QTIP_ALLOW_XFORM(3, 2) QTIP_ALLOW_XFORM(3, 4) QTIP_ALLOW_XFORM(3, 8)
  QTIP_ALLOW_XFORM(4, 2) QTIP_ALLOW_XFORM(4, 4) QTIP_ALLOW_XFORM(4, 8)
#undef QTIP_ALLOW_XFORM
#define QTIP_ALLOW_MIX(BITS, HALF)                                                                         \
  QTIP_ALLOW((matvec_kernel<BITS, 2, true, 3, false, false, HALF, 2>), kMatvecLds + kMatvecXBytes)         \
  QTIP_ALLOW((matvec_kernel<BITS, 2, true, 3, false, false, HALF, 4>), kMatvecLds + kMatvecXBytes)
  QTIP_ALLOW_MIX(2, 0) QTIP_ALLOW_MIX(2, 1) QTIP_ALLOW_MIX(2, 2) QTIP_ALLOW_MIX(3, 0) QTIP_ALLOW_MIX(4, 0)
#undef QTIP_ALLOW_MIX
#undef QTIP_ALLOW
  return hipSuccess;
}

// Per-device set-up: CU count, LDS opt-in of every kernel, address of this device's copy of
// `scratch`.  qtip_init() runs it for the current device; a launcher that meets a device for the
// first time runs it too (none of it allocates or synchronises, but hipFuncSetAttribute is not
// a call to make while a stream is being captured: callers that record graphs call qtip_init()
// first).
struct DeviceState {
  int cus = 0;
  float* scratch_ptr = nullptr;
  std::atomic<bool> done{false};  // set last, read first: the fields above are complete when it is true
};
constexpr int kMaxDevices = 64;
DeviceState g_devices[kMaxDevices];
std::mutex g_devices_mutex;

// What a launcher learns about its device in one look: rc = 0, QTIP_E_NOT_INIT (first use of the
// device inside a stream capture: the set-up is not run there and nothing is launched) or the
// hipError_t of a failed set-up (tried again by the next call).
struct Ready {
  int rc;
  int cus;
  float* scratch;
};

// State of the current device, set up on first use.  `launching`: the caller is about to
// enqueue work on `st`.  One hipGetDevice per call; the mutex only on the first use of a device.
Ready ready(bool launching, hipStream_t st) {
  int dev = -1;
  const hipError_t ge = hipGetDevice(&dev);
  if (ge != hipSuccess || dev < 0 || dev >= kMaxDevices)
    return Ready{(int)(ge != hipSuccess ? ge : hipErrorInvalidDevice), 0, nullptr};
  DeviceState& d = g_devices[dev];
  if (d.done.load(std::memory_order_acquire)) return Ready{0, d.cus, d.scratch_ptr};
  std::lock_guard<std::mutex> lock(g_devices_mutex);
  if (d.done.load(std::memory_order_relaxed)) return Ready{0, d.cus, d.scratch_ptr};
  if (launching) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    const hipError_t ce = hipStreamIsCapturing(st, &cs);
    if (ce == hipErrorStreamCaptureImplicit || (ce == hipSuccess && cs != hipStreamCaptureStatusNone))
      return Ready{QTIP_E_NOT_INIT, 0, nullptr};
    if (ce != hipSuccess) (void)hipGetLastError();  // the query's own error is not the caller's
  }
  int cus = 0;
  hipError_t e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  if (e == hipSuccess) e = allow_lds_all();
  if (e == hipSuccess) e = qtip_rht_allow_lds();
  if (e == hipSuccess) e = qtip_gemm_allow_lds();
  float* sp = nullptr;
  if (e == hipSuccess) e = hipGetSymbolAddress(reinterpret_cast<void**>(&sp), HIP_SYMBOL(scratch));
  if (e == hipSuccess && !sp) e = hipErrorInvalidSymbol;
  if (e != hipSuccess) return Ready{(int)e, 0, nullptr};
  d.cus = cus > 0 ? cus : 256;
  d.scratch_ptr = sp;
  d.done.store(true, std::memory_order_release);
  return Ready{0, d.cus, d.scratch_ptr};
}
Ready ready(void* stream) { return ready(true, (hipStream_t)stream); }

// CU count of the current device for the size queries: no set-up (they may be a process's first
// call on the device and may come while a stream is being captured), 0 when there is no device.
int query_cus() {
  int dev = -1, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return 0;
  const DeviceState& d = g_devices[dev];
  if (d.done.load(std::memory_order_acquire)) return d.cus;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
  return cus > 0 ? cus : 256;
}

// k split S for the shape: a workgroup walks `rounds` units of nwl/S wave-loads, and when the
// caller wants the summed vector (not the parts) a split costs one more small launch.
// Cost model of the k split, in units of one wave-load per wave (~0.08 us), fitted to launch times
// measured with cold weights: a unit costs its wave-loads per wave plus ~8 of fixed work (flush,
// barrier, stores; ~2 more when the output is a partial vector), a k range longer than the x
// staging area of LDS makes every wave-load ~20 % dearer (x then travels through vector loads),
// and a launch does not get shorter than ~24 however little each workgroup has to do.
int choose_split(int m, int k, int bits, int cus, bool summed) {
  (void)bits;
  const int nrb = m >> 5;
  const int nwl = ((k >> 5) + 3) >> 2;
  int best = 1;
  double best_cost = 1e30;
  for (int S = 1; S <= kMaxSplit; S *= 2) {
    if (nwl / S < kWaves && S > 1) break;  // keep at least one wave-load per wave
    const long units = (long)nrb * S;
    const long rounds = (units + cus - 1) / cus;
    const int wl_per = (nwl + S - 1) / S;
    const bool x_in_lds = (size_t)wl_per * 256 <= kMatvecXBytes;
    const double per_unit = (double)nwl / S * (x_in_lds ? 1.0 : 1.2) + 8.0 + (S > 1 ? 2.0 : 0.0);
    double cost = rounds * per_unit;
    if (cost < 24.0) cost = 24.0;
    if (S > 1 && summed) cost += 53.0;
    if (cost < best_cost * 0.97) {
      best_cost = cost;
      best = S;
    }
  }
  return best;
}

}  // namespace

int qtip_device_cus() { return query_cus(); }

int qtip_device_ready(void* stream, int* cus) {
  const Ready r = ready(stream);
  *cus = r.cus;
  return r.rc;
}

extern "C" {

int qtip_abi_version(void) { return QTIP_ABI_VERSION; }

int qtip_init(void) { return ready(false, nullptr).rc; }

const char* qtip_error_string(int code) {
  switch (code) {
    case QTIP_OK: return "ok";
    case QTIP_E_SHAPE: return "qtip: unsupported shape (need m % 32 == 0, k % 32 == 0, bits in 2..4, sizes in range)";
    case QTIP_E_NULL: return "qtip: null pointer argument";
    case QTIP_E_ALIGN: return "qtip: pointer not 16-byte aligned";
    case QTIP_E_WORKSPACE: return "qtip: workspace too small";
    case QTIP_E_DTYPE: return "qtip: unknown dtype code";
    case QTIP_E_NOT_INIT:
      return "qtip: first call on this device came inside a stream capture; call qtip_init() (or any "
             "launcher) on the device before capturing";
    case QTIP_E_SCRATCH:
      return "qtip: the partial sums of this call exceed the library's static scratch (256 KiB); use "
             "qtip_decompress_matvec with a caller workspace";
    default: return code > 0 ? hipGetErrorString((hipError_t)code) : "qtip: unknown error";
  }
}

int qtip_decode(void* out_f16, const void* packed, const void* tlut, int m, int k, int bits,
                void* stream) {
  int rc = check_common(out_f16, packed, tlut, tlut, m, k, bits);
  if (rc) return rc;
  if (!aligned16(out_f16) || !aligned16(packed) || (reinterpret_cast<uintptr_t>(tlut) & 3u))
    return QTIP_E_ALIGN;
  const Ready di = ready(stream);
  if (di.rc) return di.rc;
  const long total = (long)(m >> 5) * (((k >> 5) + 3) >> 2);
  long want = (total + kWaves - 1) / kWaves;
  const int grid = (int)(want < di.cus ? want : di.cus);
  hipStream_t st = (hipStream_t)stream;
  auto* o = (uint16_t*)out_f16;
  auto* p = (const uint8_t*)packed;
  auto* t = (const uint32_t*)tlut;
  switch (bits) {
    case 2: decode_kernel<2><<<grid, kThreads, kDecodeLds, st>>>(o, p, t, m, k); break;
    case 3: decode_kernel<3><<<grid, kThreads, kDecodeLds, st>>>(o, p, t, m, k); break;
    default: decode_kernel<4><<<grid, kThreads, kDecodeLds, st>>>(o, p, t, m, k); break;
  }
  return (int)hipGetLastError();
}

int qtip_matvec_split(int m, int k, int bits) {
  if (m <= 0 || k <= 0 || (m & 31) || (k & 31) || bits < 2 || bits > 4) return 0;
  const int cus = query_cus();
  return cus ? choose_split(m, k, bits, cus, false) : 0;
}

size_t qtip_matvec_workspace_bytes(int m, int k, int bits) {
  if (m <= 0 || k <= 0 || (m & 31) || (k & 31) || bits < 2 || bits > 4) return 0;
  const int cus = query_cus();
  if (!cus) return 0;
  const int S = choose_split(m, k, bits, cus, true);
  return S > 1 ? (size_t)S * m * sizeof(float) : 0;
}

// the kernel with a transform in front for `bits` and k = 2048, 4096 or 8192, on grid g2 with lds bytes
#define QTIP_XFORM(MODE, GROUP, ARGS)                                                       \
  switch (16 * bits + (k >> 10)) {                                                          \
    case 34: matvec_kernel<2, 2, true, MODE, false, GROUP, 0, 2><<<g2, kThreads, lds, st>>>ARGS; break; \
    case 36: matvec_kernel<2, 2, true, MODE, false, GROUP, 0, 4><<<g2, kThreads, lds, st>>>ARGS; break; \
    case 40: matvec_kernel<2, 2, true, MODE, false, GROUP, 0, 8><<<g2, kThreads, lds, st>>>ARGS; break; \
    case 50: matvec_kernel<3, 2, true, MODE, false, GROUP, 0, 2><<<g2, kThreads, lds, st>>>ARGS; break; \
    case 52: matvec_kernel<3, 2, true, MODE, false, GROUP, 0, 4><<<g2, kThreads, lds, st>>>ARGS; break; \
    case 56: matvec_kernel<3, 2, true, MODE, false, GROUP, 0, 8><<<g2, kThreads, lds, st>>>ARGS; break; \
    case 66: matvec_kernel<4, 2, true, MODE, false, GROUP, 0, 2><<<g2, kThreads, lds, st>>>ARGS; break; \
    case 68: matvec_kernel<4, 2, true, MODE, false, GROUP, 0, 4><<<g2, kThreads, lds, st>>>ARGS; break; \
    default: matvec_kernel<4, 2, true, MODE, false, GROUP, 0, 8><<<g2, kThreads, lds, st>>>ARGS; break; \
  }

static int launch_matvec(const Ready& di, float* dst, const void* packed, const void* x_f16, const void* tlut,
                         int m, int k, int bits, int S, hipStream_t st, const void* su_f16 = nullptr,
                         float xscale = 1.f, const ChainArgs* chain = nullptr, const qtip_mix::MixArgs* mix = nullptr,
                         const qtip_shares::ShareArgs* shares = nullptr) {
  const long units = (long)(m >> 5) * S;
  long grid = units < di.cus ? units : di.cus;
  grid -= grid % S;  // a workgroup keeps one k range (units is a multiple of S, so grid >= S)
  const int nwl = ((k >> 5) + 3) >> 2;
  const int wl_per = (nwl + S - 1) / S;
  auto* p = (const uint8_t*)packed;
  auto* xx = (const uint16_t*)x_f16;
  auto* t = (const uint32_t*)tlut;
  const int per_range = (int)(grid / S);  // workgroups per k range, each walks row blocks rb0, rb0 + per_range, ...
  const dim3 g2((unsigned)S, (unsigned)per_range);
  const int uq = (m >> 5) / per_range, ur = (m >> 5) % per_range;
  if (su_f16 && !mix) {
    // input transform inside the prologue: the whole transformed vector lives in LDS
    const size_t lds = xform_lds(k);
    auto* sg = (const uint16_t*)su_f16;
    if (chain) {
      QTIP_XFORM(2, false, (dst, p, xx, t, m, k, wl_per, uq, ur, sg, xscale, *chain))
      return (int)hipGetLastError();
    }
    if (shares) {
      QTIP_XFORM(4, false, (dst, p, xx, t, m, k, wl_per, uq, ur, sg, xscale, ChainArgs{}, GroupArgs{}, qtip_mix::MixArgs{}, *shares))
      return (int)hipGetLastError();
    }
    QTIP_XFORM(1, false, (dst, p, xx, t, m, k, wl_per, uq, ur, sg, xscale))
    return (int)hipGetLastError();
  }
  const size_t xbytes = (size_t)wl_per * 256;
  // row blocks left over by the rounds of whole units may be cut into their row halves
  const int full_range = di.cus / S;
  const int left = full_range > 0 ? (m >> 5) % full_range : 0;
  const int whole = full_range > 0 ? (m >> 5) / full_range : 0;
  const bool half = half_units(bits, left, whole, full_range, S, wl_per, di.cus);
  const int apart = half_apart(bits, left, whole, S, wl_per, di.cus);
  const bool aside = bits == 2 && apart == 0;  // (3 and 4 bits have the form of halves that lie apart alone)
  const int half_r = aside ? 2 * left : 2 * left | apart << kApartShift;
  if (mix) {
    const int cols = k / mix->on;
    const size_t lds = kMatvecLds + kMatvecXBytes;
    auto* sg = (const uint16_t*)su_f16;
    const bool halves = half && bits == 2;  // (not measured at 3 and 4)
    const dim3 gh = halves ? dim3((unsigned)S, (unsigned)(whole > 0 ? full_range : 2 * left)) : g2;
    const int q = halves ? whole : uq, r = halves ? half_r : ur;
#define QTIP_MIX(BITS, HALF)                                                                                                     \
  if (cols == 64) matvec_kernel<BITS, 2, true, 3, false, false, HALF, 4><<<gh, kThreads, lds, st>>>(                            \
      dst, p, xx, t, m, k, wl_per, q, r, sg, xscale, ChainArgs{}, GroupArgs{}, *mix);                                            \
  else matvec_kernel<BITS, 2, true, 3, false, false, HALF, 2><<<gh, kThreads, lds, st>>>(                                        \
      dst, p, xx, t, m, k, wl_per, q, r, sg, xscale, ChainArgs{}, GroupArgs{}, *mix)
    if (halves && aside) {
      QTIP_MIX(2, 1);
    } else if (halves) {
      QTIP_MIX(2, 2);
    } else {
      switch (bits) {
        case 2: QTIP_MIX(2, 0); break;
        case 3: QTIP_MIX(3, 0); break;
        default: QTIP_MIX(4, 0); break;
      }
    }
#undef QTIP_MIX
    return (int)hipGetLastError();
  }
  if (xbytes <= kMatvecXBytes && half) {
    const dim3 gh((unsigned)S, (unsigned)(whole > 0 ? full_range : 2 * left));
    const size_t lds = kMatvecLds + xbytes;
    switch (bits) {
      case 2:
        if (aside) matvec_kernel<2, 2, true, 0, false, false, 1><<<gh, kThreads, lds, st>>>(dst, p, xx, t, m, k, wl_per, whole, half_r);
        else matvec_kernel<2, 2, true, 0, false, false, 2><<<gh, kThreads, lds, st>>>(dst, p, xx, t, m, k, wl_per, whole, half_r);
        break;
      case 3: matvec_kernel<3, 2, true, 0, false, false, 2><<<gh, kThreads, lds, st>>>(dst, p, xx, t, m, k, wl_per, whole, half_r); break;
      default: matvec_kernel<4, 2, true, 0, false, false, 2><<<gh, kThreads, lds, st>>>(dst, p, xx, t, m, k, wl_per, whole, half_r); break;
    }
    return (int)hipGetLastError();
  }
  if (xbytes <= kMatvecXBytes) {
    const size_t lds = kMatvecLds + xbytes;
    switch (bits) {
      case 2: matvec_kernel<2, 2, true><<<g2, kThreads, lds, st>>>(dst, p, xx, t, m, k, wl_per, uq, ur); break;
      case 3: matvec_kernel<3, 2, true><<<g2, kThreads, lds, st>>>(dst, p, xx, t, m, k, wl_per, uq, ur); break;
      default: matvec_kernel<4, 2, true><<<g2, kThreads, lds, st>>>(dst, p, xx, t, m, k, wl_per, uq, ur); break;
    }
  } else if (uq == 1 && ur == 0 && (size_t)((((wl_per + kWaves - 1) / kWaves) + 1) >> 1) * kWaves * 256 <= kMatvecXBytes) {
    // one unit per workgroup and a k range of at most twice the staging area: x in two halves
    const size_t lds = kMatvecLds + kMatvecXBytes;
    switch (bits) {
      case 2: matvec_kernel<2, 2, true, 0, true><<<g2, kThreads, lds, st>>>(dst, p, xx, t, m, k, wl_per, uq, ur); break;
      case 3: matvec_kernel<3, 2, true, 0, true><<<g2, kThreads, lds, st>>>(dst, p, xx, t, m, k, wl_per, uq, ur); break;
      default: matvec_kernel<4, 2, true, 0, true><<<g2, kThreads, lds, st>>>(dst, p, xx, t, m, k, wl_per, uq, ur); break;
    }
  } else {
    switch (bits) {
      case 2: matvec_kernel<2, 2, false><<<g2, kThreads, kMatvecLds, st>>>(dst, p, xx, t, m, k, wl_per, uq, ur); break;
      case 3: matvec_kernel<3, 2, false><<<g2, kThreads, kMatvecLds, st>>>(dst, p, xx, t, m, k, wl_per, uq, ur); break;
      default: matvec_kernel<4, 2, false><<<g2, kThreads, kMatvecLds, st>>>(dst, p, xx, t, m, k, wl_per, uq, ur); break;
    }
  }
  return (int)hipGetLastError();
}

// Columns (32 or 64) of a transform of k elements in front of a matvec cut in S ranges of k, or 0: at most 256 rows (few columns
// are many rows, which more waves share), whole wave-loads in every range and a range that fits the staging area.  With
// 128 columns, for k up to 32768, the launch is slower than its two: one wave a tile goes through eight values of four rows.  us from cold
// memory at 2 bits, two launches / one with 128 columns: 5120 x 5120 9.0 / 10.5, 14336 -> 4096 10.5 / 12.1, 28672 -> 8192 23.6 / 25.9.
static int matvec_mix_cols(int k, int order, int S) {
  if (order < 1 || k < 128 || (k & 127) || k % order || S < 1 || S > kMaxSplit || S > (k >> 7)) return 0;
  const int p2 = k / order;
  if ((p2 & (p2 - 1)) || p2 < 32 || (size_t)(((k >> 7) + S - 1) / S) * 256 > kMatvecXBytes) return 0;
  if (k / 32 <= qtip_mix::kMixInMaxRows) return 32;
  return p2 >= 64 && k / 64 <= qtip_mix::kMixInMaxRows ? 64 : 0;
}

static int check_matvec(const void* out, const void* packed, const void* x_f16, const void* tlut,
                        int m, int k, int bits) {
  int rc = check_common(out, packed, x_f16, tlut, m, k, bits);
  if (rc) return rc;
  if (!aligned16(packed) || (reinterpret_cast<uintptr_t>(x_f16) & 7u) ||
      (reinterpret_cast<uintptr_t>(tlut) & 3u) || (reinterpret_cast<uintptr_t>(out) & 3u))
    return QTIP_E_ALIGN;
  return QTIP_OK;
}

#ifdef QTIP_STAMPS
// copies the clock readings of the timeline build (64 x 256 x 16 x 8 bytes) to host memory;
// synchronises the device
int qtip_debug_stamps(void* host_buf) {
  hipError_t e = hipDeviceSynchronize();
  if (e == hipSuccess) e = hipMemcpyFromSymbol(host_buf, HIP_SYMBOL(g_stamps), sizeof(g_stamps));
  return (int)e;
}
#endif

int qtip_decompress_matvec_parts(float* parts, const void* packed, const void* x_f16,
                                 const void* tlut, int m, int k, int bits, int nparts,
                                 void* stream) {
  int rc = check_matvec(parts, packed, x_f16, tlut, m, k, bits);
  if (rc) return rc;
  if (nparts < 1 || nparts > kMaxSplit || nparts > ((((k >> 5) + 3) >> 2))) return QTIP_E_SHAPE;
  const Ready rd = ready(stream);
  if (rd.rc) return rd.rc;
  return launch_matvec(rd, parts, packed, x_f16, tlut, m, k, bits, nparts, (hipStream_t)stream);
}

int qtip_decompress_matvec_parts_rht(float* parts, const void* packed, const void* x_raw_f16,
                                     const void* su_f16, float scale, const void* tlut, int m, int k,
                                     int bits, int nparts, void* stream) {
  int rc = check_matvec(parts, packed, x_raw_f16, tlut, m, k, bits);
  if (rc) return rc;
  if (!su_f16) return QTIP_E_NULL;
  if (k != 2048 && k != 4096 && k != 8192) return QTIP_E_SHAPE;
  if (nparts < 1 || nparts > kMaxSplit || nparts > (k >> 7)) return QTIP_E_SHAPE;
  if (!aligned16(x_raw_f16) || !aligned16(su_f16)) return QTIP_E_ALIGN;
  const Ready rd = ready(stream);
  if (rd.rc) return rd.rc;
  return launch_matvec(rd, parts, packed, x_raw_f16, tlut, m, k, bits, nparts, (hipStream_t)stream, su_f16, scale);
}

int qtip_decompress_matvec_parts_shares(float* parts, const void* packed, const float* shares, int ranges, int head_dim,
                                        const void* pos_i64, int max_len, const void* su_f16, float scale, const void* tlut, int m,
                                        int k, int bits, int nparts, void* stream) {
  int rc = check_matvec(parts, packed, shares, tlut, m, k, bits);
  if (rc) return rc;
  if (!su_f16 || !pos_i64) return QTIP_E_NULL;
  if ((k != 2048 && k != 4096 && k != 8192) || (head_dim != 64 && head_dim != 128)) return QTIP_E_SHAPE;
  if (nparts < 1 || nparts > kMaxSplit || nparts > (k >> 7) || ranges < 1 || ranges > qtip_shares::kMaxRanges || max_len < 1)
    return QTIP_E_SHAPE;
  if (!aligned16(shares) || !aligned16(su_f16)) return QTIP_E_ALIGN;
  const qtip_shares::ShareArgs sh = {shares, (const long*)pos_i64, ranges, head_dim == 64 ? 6 : 7, max_len};
  const Ready rd = ready(stream);
  if (rd.rc) return rd.rc;
  return launch_matvec(rd, parts, packed, shares, tlut, m, k, bits, nparts, (hipStream_t)stream, su_f16, scale, nullptr, nullptr, &sh);
}

int qtip_matvec_mix_columns(int k, int order, int nparts) { return matvec_mix_cols(k, order, nparts); }

int qtip_decompress_matvec_parts_mix(float* parts, const void* packed, const void* x_raw_f16, const void* su_f16, float scale,
                                     const uint32_t* sign_rows, int order, const void* tlut, int m, int k, int bits, int nparts,
                                     void* stream) {
  int rc = check_matvec(parts, packed, x_raw_f16, tlut, m, k, bits);
  if (rc) return rc;
  if (!su_f16 || !sign_rows) return QTIP_E_NULL;
  const int cols = matvec_mix_cols(k, order, nparts);
  if (!cols) return QTIP_E_SHAPE;
  if (!aligned16(x_raw_f16) || !aligned16(su_f16) || !aligned16(sign_rows)) return QTIP_E_ALIGN;
  const qtip_mix::MixArgs mix = {sign_rows, k / cols};
  const Ready rd = ready(stream);
  if (rd.rc) return rd.rc;
  return launch_matvec(rd, parts, packed, x_raw_f16, tlut, m, k, bits, nparts, (hipStream_t)stream, su_f16, scale, nullptr, &mix);
}

int qtip_decompress_matvec_parts_chain(float* parts, const void* packed, const void* tlut, int m, int k,
                                       int bits, int nparts, const float* prev_parts, int prev_nparts,
                                       size_t prev_part_stride, const float* post, float scale_out,
                                       const void* residual_f16, const void* norm_w_f16, float eps,
                                       const void* su_f16, float scale_in, void* x_out_f16,
                                       void* stream) {
  int rc = check_matvec(parts, packed, su_f16, tlut, m, k, bits);
  if (rc) return rc;
  if (!prev_parts || !post || !residual_f16 || !norm_w_f16 || !x_out_f16) return QTIP_E_NULL;
  if (k != 2048 && k != 4096 && k != 8192) return QTIP_E_SHAPE;
  if (nparts < 1 || nparts > kMaxSplit || nparts > (k >> 7)) return QTIP_E_SHAPE;
  if (prev_nparts < 1 || prev_nparts > kMaxSplit || x_out_f16 == residual_f16) return QTIP_E_SHAPE;
  if (!aligned16(prev_parts) || !aligned16(post) || !aligned16(residual_f16) || !aligned16(norm_w_f16) ||
      !aligned16(su_f16) || !aligned16(x_out_f16) || ((prev_part_stride * sizeof(float)) & 15u))
    return QTIP_E_ALIGN;
  ChainArgs c;
  c.parts = prev_parts;
  c.post = post;
  c.residual = (const _Float16*)residual_f16;
  c.norm_w = (const _Float16*)norm_w_f16;
  c.x_out = (_Float16*)x_out_f16;
  c.part_stride = prev_part_stride;
  c.scale_out = scale_out;
  c.eps = eps;
  c.in_parts = prev_nparts;
  const Ready rd = ready(stream);
  if (rd.rc) return rd.rc;
  return launch_matvec(rd, parts, packed, su_f16, tlut, m, k, bits, nparts, (hipStream_t)stream, su_f16, scale_in, &c);
}

}  // extern "C"

// Workgroups per k range shared out among the matrices of a grouped launch in proportion to
// their row blocks (at least one each, never more than a matrix has row blocks); fills every
// field of GroupArgs except the pointers' meaning-specific ones (su / x).  Returns the number of
// workgroups per k range, 0 if the device is too small for the group.
static int share_out_group(int cus, GroupArgs& ga, float* parts, int ngroups, const void* const* packed,
                           const void* const* tlut, const int* m, int S, long m_total) {
  const int P = cus / S;
  if (P < ngroups) return 0;
  int nrb[3] = {0, 0, 0}, wg[3] = {0, 0, 0};
  long nrb_total = 0;
  for (int g = 0; g < ngroups; ++g) {
    nrb[g] = m[g] >> 5;
    nrb_total += nrb[g];
  }
  int used = 0;
  for (int g = 0; g < ngroups; ++g) {
    long w = (long)P * nrb[g] / nrb_total;
    if (w < 1) w = 1;
    if (w > nrb[g]) w = nrb[g];
    wg[g] = (int)w;
    used += wg[g];
  }
  while (used > P) {  // the minimum of one per matrix can overshoot
    int big = 0;
    for (int g = 1; g < ngroups; ++g)
      if (wg[g] > wg[big]) big = g;
    --wg[big];
    --used;
  }
  for (bool grown = true; used < P && grown;) {  // leftovers go where a workgroup has the most units
    grown = false;
    int best = -1;
    double most = 1.0;
    for (int g = 0; g < ngroups; ++g) {
      const double load = (double)nrb[g] / wg[g];
      if (wg[g] < nrb[g] && load > most) {
        most = load;
        best = g;
      }
    }
    if (best >= 0) {
      ++wg[best];
      ++used;
      grown = true;
    }
  }
  int begin = 0;
  long col = 0;
  for (int g = 0; g < 3; ++g) {
    const int gg = g < ngroups ? g : ngroups - 1;
    ga.dst[g] = parts + (g < ngroups ? col : 0);
    ga.packed[g] = (const uint8_t*)packed[gg];
    ga.tlut[g] = (const uint32_t*)tlut[gg];
    ga.su[g] = nullptr;
    ga.x[g] = nullptr;
    ga.m[g] = m[gg];
    ga.wg_begin[g] = g < ngroups ? begin : used;
    ga.upw_q[g] = g < ngroups ? nrb[g] / wg[g] : 0;
    ga.upw_r[g] = g < ngroups ? nrb[g] % wg[g] : 0;
    if (g < ngroups) {
      begin += wg[g];
      col += m[g];
    }
  }
  ga.wg_begin[3] = used;
  ga.part_stride = (size_t)m_total;
  return used;
}

extern "C" {

int qtip_decompress_matvec_group_chain(float* parts, int ngroups, const void* const* packed,
                                       const void* const* tlut, const void* const* su_f16, const int* m,
                                       int k, int bits, int nparts, const float* prev_parts,
                                       int prev_nparts, size_t prev_part_stride, const float* post,
                                       float scale_out, const void* residual_f16, const void* norm_w_f16,
                                       float eps, float scale_in, void* x_out_f16, void* stream) {
  if (!parts || !packed || !tlut || !su_f16 || !m) return QTIP_E_NULL;
  if (ngroups < 1 || ngroups > 3) return QTIP_E_SHAPE;
  long m_total = 0;
  for (int g = 0; g < ngroups; ++g) {
    int rc = check_matvec(parts, packed[g], su_f16[g], tlut[g], m[g], k, bits);
    if (rc) return rc;
    if (!aligned16(su_f16[g])) return QTIP_E_ALIGN;
    m_total += m[g];
  }
  if (!prev_parts || !post || !residual_f16 || !norm_w_f16 || !x_out_f16) return QTIP_E_NULL;
  if (k != 2048 && k != 4096 && k != 8192) return QTIP_E_SHAPE;
  if (nparts < 1 || nparts > kMaxSplit || nparts > (k >> 7)) return QTIP_E_SHAPE;
  if (prev_nparts < 1 || prev_nparts > kMaxSplit || x_out_f16 == residual_f16) return QTIP_E_SHAPE;
  if (!aligned16(prev_parts) || !aligned16(post) || !aligned16(residual_f16) || !aligned16(norm_w_f16) ||
      !aligned16(x_out_f16) || ((prev_part_stride * sizeof(float)) & 15u))
    return QTIP_E_ALIGN;
  ChainArgs c;
  c.parts = prev_parts;
  c.post = post;
  c.residual = (const _Float16*)residual_f16;
  c.norm_w = (const _Float16*)norm_w_f16;
  c.x_out = (_Float16*)x_out_f16;
  c.part_stride = prev_part_stride;
  c.scale_out = scale_out;
  c.eps = eps;
  c.in_parts = prev_nparts;

  const int S = nparts;
  const Ready rd = ready(stream);
  if (rd.rc) return rd.rc;
  GroupArgs ga;
  const int used = share_out_group(rd.cus, ga, parts, ngroups, packed, tlut, m, S, m_total);
  if (used == 0) return QTIP_E_SHAPE;
  for (int g = 0; g < 3; ++g) ga.su[g] = (const uint16_t*)su_f16[g < ngroups ? g : ngroups - 1];
  const int nwl = ((k >> 5) + 3) >> 2;
  const int wl_per = (nwl + S - 1) / S;
  const dim3 g2((unsigned)S, (unsigned)used);
  const size_t lds = xform_lds(k);
  hipStream_t st = (hipStream_t)stream;
  QTIP_XFORM(2, true, (nullptr, nullptr, nullptr, nullptr, 0, k, wl_per, 0, 0, nullptr, scale_in, c, ga))
  return (int)hipGetLastError();
}

int qtip_decompress_matvec_group(float* parts, int ngroups, const void* const* packed,
                                 const void* const* x_f16, const void* const* tlut, const int* m, int k,
                                 int bits, int nparts, void* stream) {
  if (!parts || !packed || !tlut || !x_f16 || !m) return QTIP_E_NULL;
  if (ngroups < 1 || ngroups > 3) return QTIP_E_SHAPE;
  long m_total = 0;
  for (int g = 0; g < ngroups; ++g) {
    int rc = check_matvec(parts, packed[g], x_f16[g], tlut[g], m[g], k, bits);
    if (rc) return rc;
    if (!aligned16(x_f16[g])) return QTIP_E_ALIGN;
    m_total += m[g];
  }
  const int nwl = ((k >> 5) + 3) >> 2;
  if (nparts < 1 || nparts > kMaxSplit || nparts > nwl) return QTIP_E_SHAPE;
  const int S = nparts;
  const int wl_per = (nwl + S - 1) / S;
  const size_t xbytes = (size_t)wl_per * 256;
  if (xbytes > kMatvecXBytes) return QTIP_E_SHAPE;  // the grouped plain form keeps x in LDS
  const Ready rd = ready(stream);
  if (rd.rc) return rd.rc;
  GroupArgs ga;
  const int used = share_out_group(rd.cus, ga, parts, ngroups, packed, tlut, m, S, m_total);
  if (used == 0) return QTIP_E_SHAPE;
  for (int g = 0; g < 3; ++g) ga.x[g] = (const uint16_t*)x_f16[g < ngroups ? g : ngroups - 1];
  const dim3 g2((unsigned)S, (unsigned)used);
  const size_t lds = kMatvecLds + xbytes;
  hipStream_t st = (hipStream_t)stream;
  switch (bits) {
    case 2: matvec_kernel<2, 2, true, 0, false, true><<<g2, kThreads, lds, st>>>(nullptr, nullptr, nullptr, nullptr, 0, k, wl_per, 0, 0, nullptr, 1.f, ChainArgs{}, ga); break;
    case 3: matvec_kernel<3, 2, true, 0, false, true><<<g2, kThreads, lds, st>>>(nullptr, nullptr, nullptr, nullptr, 0, k, wl_per, 0, 0, nullptr, 1.f, ChainArgs{}, ga); break;
    default: matvec_kernel<4, 2, true, 0, false, true><<<g2, kThreads, lds, st>>>(nullptr, nullptr, nullptr, nullptr, 0, k, wl_per, 0, 0, nullptr, 1.f, ChainArgs{}, ga); break;
  }
  return (int)hipGetLastError();
}

int qtip_decompress_matvec(float* out, const void* packed, const void* x_f16, const void* tlut,
                           int m, int k, int bits, void* workspace, size_t workspace_bytes,
                           void* stream) {
  int rc = check_matvec(out, packed, x_f16, tlut, m, k, bits);
  if (rc) return rc;
  const Ready rd = ready(stream);
  if (rd.rc) return rd.rc;
  int S = 1;
  if (workspace) {
    S = choose_split(m, k, bits, rd.cus, true);
    if (S > 1 && workspace_bytes < (size_t)S * m * sizeof(float)) return QTIP_E_WORKSPACE;
    if (!aligned16(workspace)) return QTIP_E_ALIGN;
  }
  hipStream_t st = (hipStream_t)stream;
  if (S == 1) return launch_matvec(rd, out, packed, x_f16, tlut, m, k, bits, 1, st);
  rc = launch_matvec(rd, (float*)workspace, packed, x_f16, tlut, m, k, bits, S, st);
  if (rc) return rc;
  sum_parts_kernel<<<(m + 255) / 256, 256, 0, st>>>(out, (const float*)workspace, m, S);
  return (int)hipGetLastError();
}

int qtip_decompress_matvec_noalloc(float* out, const void* packed, const void* x_f16, const void* tlut,
                                   int m, int k, int bits, int nparts, void* stream) {
  int rc = check_matvec(out, packed, x_f16, tlut, m, k, bits);
  if (rc) return rc;
  const Ready rd = ready(stream);
  if (rd.rc) return rd.rc;
  const int nwl = ((k >> 5) + 3) >> 2;
  if (nparts < 0 || nparts > kMaxSplit || nparts > nwl) return QTIP_E_SHAPE;
  int S = nparts;
  if (S == 0) {
    // the library's own choice, halved until its partial sums fit the scratch (S = 1 needs none)
    S = choose_split(m, k, bits, rd.cus, true);
    while (S > 1 && (size_t)S * m > kScratchFloats) S >>= 1;
  }
  hipStream_t st = (hipStream_t)stream;
  if (S == 1) return launch_matvec(rd, out, packed, x_f16, tlut, m, k, bits, 1, st);
  if ((size_t)S * m > kScratchFloats) return QTIP_E_SCRATCH;  // only a split the caller asked for
  // every one of the S * m partial sums is written before it is read: nothing to clear
  float* parts = rd.scratch;
  rc = launch_matvec(rd, parts, packed, x_f16, tlut, m, k, bits, S, st);
  if (rc) return rc;
  sum_parts_kernel<<<(m + 255) / 256, 256, 0, st>>>(out, parts, m, S);
  return (int)hipGetLastError();
}

}  // extern "C"
