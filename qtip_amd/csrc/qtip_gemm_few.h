// Batched decompress + fp16 MFMA GEMM up to 16 batch rows.  Included by qtip_gemm.hip inside its namespace.
//
// Up to 16 rows of activations are 2 KiB beside the 512 * K bytes of weights of a wave-load, so every wave reads its own
// from L2 and walks its stream freely, four waves to a SIMD covering for each other as in the matvec; nothing but the
// end of a unit holds them together.  (Shared through LDS, as gemm_kernel has them, they cost a barrier per wave-load: the
// four waves decode, multiply and wait at the same time, 1.6 us per round of wave-loads against 1.0 to 1.3 here and
// 1.06 of the matvec.)  A lane loads eight consecutive columns of one batch row, 16 bytes; v_permlane16_swap makes them the
// four and four of an MFMA operand.  Loads of the four and four, 8 bytes each, were bound by the address rate
// (28672x8192 at 2 bits, 16 rows: 38 us).
//
// 16 waves of 128 registers: RG row-block pairs by KS = 16 / RG column slices, which meet in LDS at a unit's end.  One
// wave-load of weights in flight per wave instead of two: 10 % more from cold memory at 4 bits.  us per product of 16 rows from
// cold memory, launches and sums of ranges included, gemm_kernel / here with fine sums, 2 bits: 28672x8192 27.6 / 24.6,
// 22016x4096 15.9 / 13.0, 4096x4096 10.5 / 9.7, 4096x11008 13.8 / 12.2, 8192x28672 26.8 / 26.7.  At 4 bits 4096x4096 10.8 / 9.9,
// 4096x11008 15.2 / 14.2, but of the largest (launch alone) 22016x4096 15.9 / 16.8 and 28672x8192 28.0 / 34.2: there the
// stream is the bound, and requests for 16 rows of activations are in its way (shared_rows).

template <int K, int RG, typename TOut>
__global__ __launch_bounds__(64 * kFewWaves, 1) void gemm_few_kernel(
    TOut* __restrict__ dst, const uint8_t* __restrict__ packed, const uint16_t* __restrict__ x,
    const uint32_t* __restrict__ tlut, int m, int k, int batch, long ldo, int round_f16, int wl_per, int upw_q, int upw_r) {
  constexpr int WAVES = kFewWaves, THREADS = 64 * WAVES, KS = WAVES / RG;
  extern __shared__ __align__(16) uint8_t smem[];
  uint32_t* lut = reinterpret_cast<uint32_t*>(smem);
  float* xch = reinterpret_cast<float*>(smem + kLut128Bytes);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rg = wave % RG, ks = wave / RG;
  const int r8 = lane & 7, pb = (lane >> 3) & 1, ch = (lane >> 4) & 1, g0 = lane >> 5;
  const uint32_t slot4 = lds_address(lut) + ((uint32_t)(lane & 31) << 2);
  const int nkb = k >> 5, nwl = (nkb + 1) >> 1, nrb = m >> 5, npair = (nrb + 1) >> 1;
  const uint32_t rb_bytes = (uint32_t)nkb * 128 * K;
  constexpr uint32_t WL_BYTES = 256 * K, OUT = kOutOfRange;
  const uint32_t loff = (uint32_t)pb * rb_bytes + (uint32_t)g0 * (128 * K) + (uint32_t)(2 * r8 + ch) * (8 * K);
  const int nxt4 = (ch ? ((lane & ~23) | ((r8 + 1) & 7)) : (lane | 16)) << 2;
  const __amdgpu_buffer_rsrc_t rs_w = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(packed), 0, (int)((size_t)nrb * rb_bytes), 0x00020000);
  const __amdgpu_buffer_rsrc_t rs_x =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(x), 0, (int)((size_t)batch * k * 2), 0x00020000);
  auto uni = [](auto v) { return __builtin_amdgcn_readfirstlane(v); };

  const int s = blockIdx.x, u0 = blockIdx.y, ustep = gridDim.y;
  const int wl0 = s * wl_per;
  const int wl1 = wl0 + wl_per < nwl ? wl0 + wl_per : nwl;
  const int upw = upw_q + (u0 < upw_r ? 1 : 0);
  const int nst = wl1 - wl0 > ks ? (wl1 - wl0 - ks + KS - 1) / KS : 0;  // wave-loads of this wave per unit
  TOut* out_s = dst + (size_t)s * batch * ldo;

  // ---- stream: two wave-loads of weights in flight, their place refilled as soon as the states of one are in registers;
  // the activations one ahead, asked for before the weights of the next (loads return in order)
  LaneData<K> buf[2];
  u32x4 xr[2][2];  // [parity of the wave-load][column half]
  const bool last_half = (nkb & 1) && nst > 0 && wl0 + KS * (nst - 1) + ks == nwl - 1;
  int w_left = nst, w_u = u0, w_n = upw, x_left = nst, x_n = upw;
  uint32_t w_so = 0, w_vo = OUT, x_so = 0, x_vo = OUT;
  auto w_unit = [&]() {
    const int pair = w_u * RG + rg;
    const bool ok = w_n > 0 && nst > 0 && pair < npair;
    w_so = ok ? (uint32_t)(2 * pair) * rb_bytes + (uint32_t)(wl0 + ks) * WL_BYTES : 0u;
    w_vo = ok && 2 * pair + pb < nrb && !(last_half && nst == 1 && g0) ? loff : OUT;
    w_left = nst;
  };
  auto x_unit = [&]() {
    const FewPlace p = few_activations(lane, batch, k, wl0 + ks, x_n, nst, last_half);
    x_so = p.so;
    x_vo = p.vo;
    x_left = nst;
  };
  auto load_x = [&](int d) {
#pragma unroll
    for (int i = 0; i < 2; ++i) xr[d][i] = __builtin_amdgcn_raw_buffer_load_b128(rs_x, x_vo + 32 * i, uni(x_so), 0);
    x_so += KS * 128;
    --x_left;
  };
  auto load_w = [&](int d) { buf[d] = load_lane_buf<K>(rs_w, w_vo, uni(w_so)); };
  auto x_next = [&]() {
    if (uni(x_left) <= 1) {
      if (uni(x_left) <= 0) {
        --x_n;
        x_unit();
      } else if (last_half && g0) {
        x_vo = OUT;
      }
    }
  };
  auto w_next = [&]() {
    w_so += KS * WL_BYTES;
    if (uni(--w_left) <= 1) {
      if (uni(w_left) <= 0) {
        --w_n;
        w_u += ustep;
        w_unit();
      } else if (last_half && g0) {
        w_vo = OUT;
      }
    }
  };
  w_unit();
  x_unit();
  constexpr int NTW = kLutEntries * 4 / THREADS;
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
  load_x(0);
  x_next();
  load_w(0);
  w_next();
#pragma unroll
  for (int it = 0; it < 2 * NTW; ++it) {
    const uint32_t w = tw[it % NTW] ^ ((uint32_t)(it / NTW) << 15);
    const u32x4 v = {w, w, w, w};
    reinterpret_cast<u32x4*>(lut)[it * THREADS + tid] = v;
  }
  __syncthreads();

  load_w(1);
  w_next();
  float4_t acc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i] = float4_t{0.f, 0.f, 0.f, 0.f};
  auto work = [&](int d, bool cut) {  // cut: the wave-load ends after 32 columns
    load_x(d ^ 1);
    x_next();
    uint32_t P[16], W[2][16];
    packed_states<K>(buf[d], P, [&](uint32_t v) { return (uint32_t)__builtin_amdgcn_ds_bpermute(nxt4, (int)v); });
    __builtin_amdgcn_sched_barrier(0);
    load_w(d);
    w_next();
#pragma unroll
    for (int kh = 0; kh < 2; ++kh)
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        const uint32_t q = pk_hash(P[SlotMap<K>::reg(kh, r)]) & 0xFFC0FFC0u;
        W[kh][SlotMap<K>::word(r, 0)] = lds_word_abs(lut128_addr_lo(q, slot4));
        W[kh][SlotMap<K>::word(r, 1)] = lds_word_abs(lut128_addr_hi(q, slot4));
      }
    __builtin_amdgcn_sched_barrier(0);
    if (uni(cut)) {  // (what the missing block decodes to, table entry 0, may be infinite)
#pragma unroll
      for (int i = 0; i < 32; ++i) (&W[0][0])[i] = g0 ? 0u : (&W[0][0])[i];
    }
#pragma unroll
    for (int kh = 0; kh < 2; ++kh) {
      // a lane's eight consecutive columns to the operand's four and four
      const u32x4 v = xr[d][kh];
      const auto a = __builtin_amdgcn_permlane16_swap(v[0], v[2], false, false);
      const auto b = __builtin_amdgcn_permlane16_swap(v[1], v[3], false, false);
      const u32x4 xa = {a[0], b[0], a[1], b[1]};
#pragma unroll
      for (int mr = 0; mr < 4; ++mr) {
        const u32x4 wv = {W[kh][4 * mr], W[kh][4 * mr + 1], W[kh][4 * mr + 2], W[kh][4 * mr + 3]};
        acc[mr] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, wv), __builtin_bit_cast(half8_t, xa), acc[mr],
                                                         0, 0, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  int u = u0;
  int par = 0;  // parity of the next wave-load: a unit may hold an odd number
  for (int un = 0; un < upw; ++un, u += ustep) {
    int t = nst;
    if (par && t > 0) {
      work(1, last_half && t == 1);
      --t;
    }
    for (; t > 1; t -= 2) {
      work(0, false);
      work(1, last_half && t == 2);
    }
    par = 0;
    if (t == 1) {
      work(0, last_half);
      par = 1;
    }
    par = uni(par);
    // ---- the slices of the unit meet
    constexpr int VEC = 4, V = kGemmTileBytes / (WAVES * 1024);  // accumulator vectors, those that fit at a time
#pragma unroll
    for (int f0 = 0; f0 < VEC; f0 += V) {
#pragma unroll
      for (int f = 0; f < V; ++f)
        *reinterpret_cast<float4_t*>(xch + ((wave * V + f) * 64 + lane) * 4) = acc[f0 + f];
      __syncthreads();
      if (wave < RG * V) {
        const int f = wave / RG, g = wave % RG;
        float4_t sum = *reinterpret_cast<const float4_t*>(xch + ((g * V + f) * 64 + lane) * 4);
#pragma unroll
        for (int z = 1; z < KS; ++z) sum += *reinterpret_cast<const float4_t*>(xch + (((z * RG + g) * V + f) * 64 + lane) * 4);
        const int row = 64 * (u * RG + g) + 32 * g0 + 8 * (f0 + f) + 4 * ch, bb = lane & 15;
        if (bb < batch && row < m) {
          typedef TOut out4_t __attribute__((ext_vector_type(4), aligned(sizeof(TOut))));
          out4_t y;
#pragma unroll
          for (int e = 0; e < 4; ++e) y[e] = (TOut)(sizeof(TOut) == 4 && round_f16 ? (float)(_Float16)sum[e] : sum[e]);
          *reinterpret_cast<out4_t*>(out_s + (size_t)bb * ldo + row) = y;
        }
      }
      __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = float4_t{0.f, 0.f, 0.f, 0.f};
  }
}
