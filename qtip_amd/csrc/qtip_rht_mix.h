// Randomised Hadamard transform of many rows, every table order: the mix on the matrix cores.
// Included by qtip_rht.hip inside its namespace (RhtParams, Raw8, the PRE_* modes).
//
// A row of n = order * S * A * pp elements is, for each of the S slices of its power-of-two part,
// the (order*A) x pp matrix v[j][c], and its transform is (table (x) H_A) v H_pp.  The left factor
// is a matrix of +-1, so the product runs on the matrix cores without losing a bit:
//   one fp16 plane    fp16 values under a sign vector of +-1 (or none): v is fp16 as it stands
//   three bf16 planes everything else: v's 24 mantissa bits cut into 8 + 8 + 8 by truncation, one
//                     plane at a time through the same LDS; a third plane of zeros is skipped
// Products are exact, sums fp32.  H_pp is butterflies on the accumulators: three levels over
// registers, the rest over the low lane bits.
//
// A workgroup of two waves per k tile (KT = ceil(order*A / 32) tiles) takes 128 columns (128 / pp
// rows) at a time.  Wave w, lane (g, a) loads rows 16w + 4g .. + 3 of v at columns 8a .. 8a + 7
// (16-byte loads, 256 contiguous bytes per row of v) and writes them to LDS transposed: for column
// 8a + e the four values are 8 contiguous bytes of column position 16e + a.  Wave w then owns
// output rows 16w .. 16w + 15: operand A the signs (a byte per k tile and row, expanded on use),
// operand B the columns 8a + e over all KT row blocks.  So a lane ends with eight consecutive
// columns of four output rows and stores 16 bytes at a time.  Columns are padded to an odd number
// of 16-byte units, which keeps the 16-byte reads of a phase on distinct banks.  The next 128
// columns are requested before the products of the current ones.
//
// KTC = 2, 4, 8 (at least KT) fixes the column stride, so that the LDS addresses are one register and
// immediate offsets: computed from a run-time stride they cost 32 registers, and the kernel spilled.
//
// Bound by a wave's instructions, so 16-row waves with 128 registers, four to a SIMD (32-row waves of
// 256 registers read LDS half as often and took 45 instead of 41 us below).  us per launch, fp16 rows
// under a +-1 sign vector, with the one-workgroup-set-per-row form (or, at order 172, the best of it
// and fp32 library products) before: 28672 = 28 * 1024, 1000 rows 772 -> 39 (2.9 TB/s), 45 rows
// 38 -> 7.7; 11008 = 172 * 64, 1000 rows ~150 -> 19, 45 rows 67 -> 7.5; 12288, 1000 rows 471 -> 17.
// fp32 rows: 28672, 1000 rows 811 -> 82; 11008, 2048 rows ~240 -> 64.  Few rows: the workgroups of a pass share its
// output rows (launch_mix), each with all of the plane.

using qtip_mix::bf16x8;
using qtip_mix::half8m;
using qtip_mix::u32x4m;
using qtip_mix::expand_signs;
using qtip_mix::mix_signs;
constexpr int kMixCols = 128;
constexpr int kMixMaxKT = 8;
constexpr int kMixMaxOrder = 32 * kMixMaxKT;  // table orders, built in or a caller's own

struct MixShape {
  int logpp, logA2, logS;  // n = order << (logS + logA2 + logpp)
  int npass;               // 128-column groups
  int share;               // waves of a workgroup that produce output rows: from share * blockIdx.y on
};

constexpr uint32_t mix_stride(int ktc) { return 64 * ktc + 16; }  // bytes per column

// the plane, the table bits, the row sums and the flags
constexpr size_t mix_lds(int ktc, int order) {
  return (size_t)kMixCols * mix_stride(ktc) + (((size_t)order * order + 31) / 32 * 4 + 15) / 16 * 16 +
         32 * kMixMaxKT * sizeof(float) + 16;
}

template <typename TIn, typename TOut, int MODE, int KTC>
__global__ __launch_bounds__(128 * KTC, 4) void rht_mix_kernel(const RhtParams P, const MixShape M, int rows) {
  extern __shared__ __align__(16) uint8_t mix_smem[];
  constexpr bool F16 = sizeof(TIn) == 2;
  constexpr bool PARTS = MODE == PRE_PARTS;  // rows of fp32 partial sums, summed and rounded to fp16 on load
  constexpr bool AUX = MODE != PRE_NONE && !PARTS;
  static_assert(MODE == PRE_NONE || F16, "the element-wise prologues take fp16 rows");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int KT = blockDim.x >> 7;
  const int a = lane & 15, g = lane >> 4;
  const int logA2 = M.logA2, logpp = M.logpp, logS = M.logS;
  const int order = P.order, S = 1 << logS, on = order << logA2;
  const int n = P.n;
  // grid (8, shares, eights of passes * slices): the workgroups that read the same rows are on one XCD
  const int s = blockIdx.z & (S - 1), step = 8 * (gridDim.z >> logS);
  constexpr uint32_t stride = mix_stride(KTC);
  uint32_t* hb = reinterpret_cast<uint32_t*>(mix_smem + kMixCols * stride);
  const int nw = (order * order + 31) >> 5;
  float* wsum = reinterpret_cast<float*>(hb + ((nw + 3) & ~3));  // [2 KT][16] sums of squares
  uint32_t* flag = reinterpret_cast<uint32_t*>(wsum + 32 * kMixMaxKT);  // a third plane is needed, the sign vector is not +-1
  const TIn* in = reinterpret_cast<const TIn*>(P.in);

  // ---- this lane's patch of v: row j = 16 * wave + 4 * g + i, columns c0 .. c0 + 7 of row rsub of the pass
  const int lrows = 7 - logpp;  // log2 of the rows per pass
  const int rsub = (8 * a) >> logpp, c0 = (8 * a) & ((1 << logpp) - 1);
  // a result's columns are those of the lane's place, which the operands are read for
  int pa = wht_place(lane) & 15, rsub_out = (8 * pa) >> logpp, c0_out = (8 * pa) & ((1 << logpp) - 1);
  const int Am = (1 << logA2) - 1;
  // element j, slice part sl inside a row
  auto element = [&](int j, int sl) {
    return (uint32_t)((((((j >> logA2) << logS) + sl) << logA2) + (j & Am)) << logpp) + (uint32_t)c0;
  };
  const int j0 = 16 * wave + 4 * g;
  uint32_t eoff[4];  // element offset of patch row i inside a row, slice part 0 (row 0 for padding)
#pragma unroll
  for (int i = 0; i < 4; ++i) eoff[i] = element(j0 + i < on ? j0 + i : 0, 0);
  const int nlive = on - j0;                          // patch rows i < nlive are rows of v
  const bool edge = 16 * wave + 16 > on;              // the wave holds padding rows
  // no output rows here: padding (the second wave of the last k tile), or another workgroup's share
  const bool idle = 16 * wave >= on || (unsigned)(wave - (int)blockIdx.y * M.share) >= (unsigned)M.share;
  const uint32_t slice_step = 1u << (logA2 + logpp);  // elements between slices

  // Addresses are a uniform base (the pass's first row) and a 32-bit lane offset.
  // a patch's raw operands: input, sign vector, norm weight or up half
  struct Patch {
    Raw8<TIn> x[4];
    Raw8<_Float16> f[4], u[AUX ? 4 : 1];
  };
  auto first_row = [&](int ps) { return (size_t)ps << lrows; };
  auto lane_row = [&](int ps) { return (int)first_row(ps) + rsub < rows ? (uint32_t)rsub : 0u; };  // (a row to read)
  auto load_patch = [&](Patch& p, int ps, uint32_t add, bool vectors = true) {
    const TIn* src = in + first_row(ps) * P.in_row_stride;
    const uint32_t lr = lane_row(ps) * (uint32_t)P.in_row_stride + add;
    if constexpr (PARTS) {
      const float* parts = reinterpret_cast<const float*>(P.in) + first_row(ps) * P.in_row_stride;
#pragma unroll
      for (int i0 = 0; i0 < 4; i0 += 2) {  // (two rows at a time: registers)
        float t[2][8];
#pragma unroll
        for (int i = 0; i < 2; ++i) ld_f32<8>(parts + (lr + eoff[i0 + i]), t[i]);
        for (int w = 1; w < P.in_parts; ++w) {
          const float* more = parts + w * P.part_stride;
          float q[2][8];
#pragma unroll
          for (int i = 0; i < 2; ++i) ld_f32<8>(more + (lr + eoff[i0 + i]), q[i]);
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int e = 0; e < 8; ++e) t[i][e] += q[i][e];
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          half8m h;
#pragma unroll
          for (int e = 0; e < 8; ++e) h[e] = (_Float16)t[i][e];
          p.x[i0 + i] = __builtin_bit_cast(Raw8<TIn>, h);
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) p.x[i].load(src + (lr + eoff[i]));
    }
    if (!vectors) return;
    if (P.pre) {
      const _Float16* f = P.pre + first_row(ps) * P.pre_row_stride;
      const uint32_t lf = lane_row(ps) * (uint32_t)P.pre_row_stride + add;
#pragma unroll
      for (int i = 0; i < 4; ++i) p.f[i].load(f + (lf + eoff[i]));
    }
    if constexpr (MODE == PRE_RMSNORM) {
#pragma unroll
      for (int i = 0; i < 4; ++i) p.u[i].load(P.norm_w + (add + eoff[i]));
    } else if constexpr (MODE == PRE_SILU_MUL) {
      const _Float16* up = reinterpret_cast<const _Float16*>(src) + n;
#pragma unroll
      for (int i = 0; i < 4; ++i) p.u[i].load(up + (lr + eoff[i]));
    }
  };
  Patch cur;
  int ps = blockIdx.x + 8 * (blockIdx.z >> logS);
  if (ps >= M.npass) return;
  if (F16) load_patch(cur, ps, 0);

  // the output vector is needed last, behind a chain as long as a cold read: its cache lines are asked for now
  // (a dword of each: rows 16 * wave + lane / 4 of the mix, 32 columns a lane)
  float line = 0.f;
  if (!AUX && P.post && !idle) {
    const int i = 16 * wave + (lane >> 2), c = 32 * (lane & 3) & ((1 << logpp) - 1);
    line = P.post[first_row(ps) * P.post_row_stride + element(i < on ? i : 0, s) - c0 + c];
  }

  for (int i = tid; i < nw; i += blockDim.x) hb[i] = order > 1 ? P.had_bits[i] : 0u;
  if (tid < 2) flag[tid] = 0;
  __syncthreads();
  // ---- signs of output row 16 * wave + a against v rows 32 * kt + 8 * g + e: byte kt of sb, bit e
  uint32_t sb0 = 0, sb1 = 0;
  if (!idle) mix_signs<KTC>(sb0, sb1, hb, order, logA2, 16 * wave, on, lane);
  auto signs = [&](int kt, uint32_t one) {
    return expand_signs(((KTC > 4 && (kt & 4) ? sb1 : sb0) >> (8 * (kt & 3))) & 0xFFu, one);
  };
  // the wave's reciprocal RMS of the lane's row: every slice, all waves, the lanes of the row
  auto row_rs = [&](const Patch& p, int ps) {
    float ss = 0.f;
    auto squares = [&](const Raw8<TIn> y[4]) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float t[8];
        y[i].get(t);
        float q = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) q += t[e] * t[e];
        ss += i < nlive ? q : 0.f;
      }
    };
    squares(p.x);
    for (int sj = 1; sj < S; ++sj) {
      Raw8<TIn> y[4];
      const uint32_t lr = lane_row(ps) * (uint32_t)P.in_row_stride + sj * slice_step;
#pragma unroll
      for (int i = 0; i < 4; ++i) y[i].load(in + first_row(ps) * P.in_row_stride + (lr + eoff[i]));
      squares(y);
    }
    // lane bits 4, 5 and the low logpp - 3 bits of a
#pragma unroll
    for (int b = 0; b < 6; ++b)
      if (b >= 4 || b < logpp - 3) ss += lane_xor(ss, b);
    if (g == 0) wsum[wave * 16 + a] = ss;
    __syncthreads();
    float tot = 0.f;
    for (int w = 0; w < 2 * KT; ++w) tot += wsum[w * 16 + a];
    return __builtin_amdgcn_rsqf(tot / (float)n + P.eps);
  };
  // the element-wise prologue on eight fp16 values of a patch row
  auto prologue = [&](const Raw8<_Float16>& px, const Raw8<_Float16>& pu, float rs) {
    half8m x = __builtin_bit_cast(half8m, px);
    if constexpr (MODE == PRE_RMSNORM) {
      half8m h;
#pragma unroll
      for (int e = 0; e < 8; ++e) h[e] = (_Float16)((float)x[e] * rs);
      x = __builtin_bit_cast(half8m, pu) * h;
    } else if constexpr (MODE == PRE_SILU_MUL) {
      half8m h;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float gt = (float)x[e];
        h[e] = (_Float16)(gt * __builtin_amdgcn_rcpf(1.f + __expf(-gt)));
      }
      x = h * __builtin_bit_cast(half8m, pu);
    }
    return x;
  };
  // H_pp on the products (register e is column bits 0..2, bit b of a lane's place column bit 3 + b) and the results
  auto finish = [&](float4v acc[8], int ps) {
    if (idle) return;
    if constexpr (!AUX) asm volatile("" ::"v"(line));
    if constexpr (MODE == PRE_SILU_MUL && KTC == 8) {
      // (Taken again: kept over the products they cost this form a register to scratch, 16 rows of 28672 9.8 us, so 9.3.  The
      // other forms have the registers for them; taken again there, 1000 rows are 1 to 4 % slower.)
      int own = lane;
      asm("" : "+v"(own));
      pa = wht_place(own) & 15, rsub_out = (8 * pa) >> logpp, c0_out = (8 * pa) & ((1 << logpp) - 1);
    }
#pragma unroll
    for (int h = 1; h < 8; h <<= 1)
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (!(e & h)) {
          const float4v u = acc[e], w = acc[e + h];
          acc[e] = u + w;
          acc[e + h] = u - w;
        }
#pragma unroll
    for (int b = 0; b < 4; ++b)
      if (b < logpp - 3) {
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
          for (int q = 0; q < 4; ++q) acc[e][q] = wht_place_stage(acc[e][q], b, pa);
      }
    // output rows 16 * wave + 4 * g + q of the mix
    const bool row_ok = (int)first_row(ps) + rsub_out < rows;
    const uint32_t lr = row_ok ? (uint32_t)rsub_out : 0u;
    const float* post = P.post ? P.post + first_row(ps) * P.post_row_stride : nullptr;
    const _Float16* res = P.residual ? P.residual + first_row(ps) * n : nullptr;
    TOut* out = reinterpret_cast<TOut*>(P.out) + first_row(ps) * n;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int i = j0 + q;
      const uint32_t o = element(i < on ? i : 0, s) - c0 + c0_out;
      float y[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] = acc[e][q] * P.scale;
      if (post) {
        Raw8<float> pv;
        pv.load(post + (lr * (uint32_t)P.post_row_stride + o));
        float t[8];
        pv.get(t);
#pragma unroll
        for (int e = 0; e < 8; ++e) y[e] *= t[e];
      }
      TOut* dst = out + (lr * (uint32_t)n + o);
      if constexpr (sizeof(TOut) == 2) {
        if (res) {
          float t[8];
          ld_f16<8>(res + (lr * (uint32_t)n + o), t);
#pragma unroll
          for (int e = 0; e < 8; ++e) y[e] = t[e] + (float)(_Float16)y[e];
        }
        _Float16 h[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) h[e] = (_Float16)y[e];
        if (row_ok && i < on) st_f16<8>(reinterpret_cast<_Float16*>(dst), h);
      } else if (row_ok && i < on) {
        *reinterpret_cast<float4v*>(dst) = float4v{y[0], y[1], y[2], y[3]};
        *reinterpret_cast<float4v*>(dst + 4) = float4v{y[4], y[5], y[6], y[7]};
      }
    }
  };
  uint8_t* wr = mix_smem + (uint32_t)a * stride + (uint32_t)(4 * wave + g) * 8;
  const uint8_t* rd = mix_smem + (uint32_t)pa * stride + (uint32_t)g * 16;
  // the plane's products: a column group's next operand is requested as soon as its present one is used
  auto products = [&](float4v acc[8], uint32_t one, auto mfma) {
    if (idle) return;
    u32x4m b[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) b[e] = *reinterpret_cast<const u32x4m*>(rd + e * 16 * stride);
    for (int kt = 0; kt < KT; ++kt) {
      const u32x4m fa = signs(kt, one);
      const uint8_t* next = rd + (kt + 1 < KT ? kt + 1 : kt) * 64;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        acc[e] = mfma(fa, b[e], acc[e]);
        b[e] = *reinterpret_cast<const u32x4m*>(next + e * 16 * stride);
      }
    }
  };

  // ---- one plane of fp16 values: no slices or partial sums to add, and a sign vector of nothing but
  // +-1 (the same for every pass)
  if constexpr (F16) {
    bool fast = S == 1 && (PARTS || P.in_parts == 1) && (!P.pre || P.pre_row_stride == 0);
    if (fast && P.pre) {
      uint32_t off = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const u32x4m f = __builtin_bit_cast(u32x4m, cur.f[i].a);
#pragma unroll
        for (int q = 0; q < 4; ++q) off |= (f[q] & 0x7FFF7FFFu) ^ 0x3C003C00u;
      }
      if (__any(off != 0) && lane == 0) flag[1] = 1;
      __syncthreads();
      fast = flag[1] == 0;
    }
    if (fast) {
      // behind a norm the signs go into its weights, which every pass has in common: read again for each and kept beside the
      // products' operands they cost 13 to 16 registers of scratch (us, 1000 rows, then / now: 28672 51.1/41.4, 4096 9.5/8.5)
      constexpr bool NORM = MODE == PRE_RMSNORM;
      if (NORM && P.pre) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          cur.u[AUX ? i : 0].a = __builtin_bit_cast(uint4, __builtin_bit_cast(u32x4m, cur.u[AUX ? i : 0].a) ^
                                                      (__builtin_bit_cast(u32x4m, cur.f[i].a) & 0x80008000u));
      }
      for (; ps < M.npass; ps += step) {
        float rs = 1.f;
        if constexpr (MODE == PRE_RMSNORM) rs = row_rs(cur, ps);
        u32x4m h[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          h[i] = __builtin_bit_cast(u32x4m, prologue(cur.x[i], cur.u[AUX ? i : 0], rs));
          if (!NORM && P.pre) h[i] ^= __builtin_bit_cast(u32x4m, cur.f[i].a) & 0x80008000u;
        }
        if (edge) {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (i >= nlive) h[i] = u32x4m{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          uint2 w;
          w.x = __builtin_amdgcn_perm(h[1][e >> 1], h[0][e >> 1], (e & 1) ? 0x07060302u : 0x05040100u);
          w.y = __builtin_amdgcn_perm(h[3][e >> 1], h[2][e >> 1], (e & 1) ? 0x07060302u : 0x05040100u);
          *reinterpret_cast<uint2*>(wr + e * 16 * stride) = w;
        }
        if (ps + step < M.npass) load_patch(cur, ps + step, 0, !NORM);
        __syncthreads();
        float4v acc[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] = float4v{0.f, 0.f, 0.f, 0.f};
        products(acc, 0x3C003C00u, [](u32x4m fa, u32x4m b, float4v c) {
          return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8m, fa), __builtin_bit_cast(half8m, b), c, 0, 0, 0);
        });
        __syncthreads();  // the plane is free
        finish(acc, ps);
      }
      return;
    }
  }

  // ---- three bf16 planes of fp32 values
  for (; ps < M.npass; ps += step) {
    float v[4][8];
    {
      float rs = 1.f;
      if constexpr (MODE == PRE_RMSNORM) {
        load_patch(cur, ps, 0);
        rs = row_rs(cur, ps);
      }
      for (int sj = 0; sj < S; ++sj) {
        const uint32_t add = sj * slice_step;
        load_patch(cur, ps, add);
        const uint32_t lr = lane_row(ps) * (uint32_t)P.in_row_stride + add;
        const uint32_t flip = ((uint32_t)__builtin_popcount(s & sj) & 1u) << 31;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float t[8];
          if constexpr (AUX) {
            const half8m x = prologue(cur.x[i], cur.u[i], rs);
#pragma unroll
            for (int e = 0; e < 8; ++e) t[e] = (float)x[e];
          } else {
            cur.x[i].get(t);
            for (int w = 1; w < (PARTS ? 1 : P.in_parts); ++w) {
              Raw8<TIn> y;
              y.load(in + w * P.part_stride + first_row(ps) * P.in_row_stride + (lr + eoff[i]));
              float q[8];
              y.get(q);
#pragma unroll
              for (int e = 0; e < 8; ++e) t[e] += q[e];
            }
          }
          if (P.pre) {
            float f[8];
            cur.f[i].get(f);
#pragma unroll
            for (int e = 0; e < 8; ++e) t[e] *= f[e];
          }
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float u = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, t[e]) ^ flip);
            v[i][e] = sj ? v[i][e] + u : u;
          }
        }
      }
    }
    if (edge) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (i >= nlive) {
#pragma unroll
          for (int e = 0; e < 8; ++e) v[i][e] = 0.f;
        }
    }
    float4v acc[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = float4v{0.f, 0.f, 0.f, 0.f};
    for (int p = 0; p < 3; ++p) {
      // the leading eight bits of what is left of every value
      uint32_t left = 0;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        uint32_t b[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          b[i] = __builtin_bit_cast(uint32_t, v[i][e]);
          // (nothing is left of an infinity: the difference would turn it into a NaN)
          const float rest = v[i][e] - __builtin_bit_cast(float, b[i] & 0xFFFF0000u);
          v[i][e] = __builtin_isinf(v[i][e]) ? 0.f : rest;
          left |= __builtin_bit_cast(uint32_t, v[i][e]);
        }
        uint2 w;
        w.x = __builtin_amdgcn_perm(b[1], b[0], 0x07060302u);
        w.y = __builtin_amdgcn_perm(b[3], b[2], 0x07060302u);
        *reinterpret_cast<uint2*>(wr + e * 16 * stride) = w;
      }
      if (p == 1 && __any((left & 0x7FFFFFFFu) != 0) && lane == 0) flag[0] = 1;
      __syncthreads();
      products(acc, 0x3F803F80u, [](u32x4m fa, u32x4m b, float4v c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, fa), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
      });
      const bool last = p == 2 || (p == 1 && flag[0] == 0);  // the same for the whole workgroup
      if (p == 2 && tid == 0) flag[0] = 0;                   // (everyone read it before the barrier of this plane)
      __syncthreads();                                       // the plane is free
      if (last) break;
    }
    finish(acc, ps);
  }
}
