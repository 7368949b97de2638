// Batched decompress + fp16 MFMA GEMM from 33 batch rows on.  Included by qtip_gemm.hip inside its namespace.
//
// The matrix cores do not wait for the decode: a wave multiplies one column half (16 of the 32
// columns of either tile block, 16 table words) while it looks up the words of the next, and the instructions of
// both, with the LDS reads of the activations two groups ahead, are issued in turn.  (Decoding, then
// multiplying, between two barriers reached 0.67 PFLOP/s at 128 rows of 28672x8192.)
//
// A workgroup is eight waves of up to 256 registers, two to a SIMD: RG row-block pairs by KS = 8 / RG column slices
// of 64, a batch tile of 16 * NB rows.  The 128 KiB table leaves 32 KiB: two tiles of activations, one stage
// (a wave-load of every slice, or half of one where a whole stage takes more than 16 KiB) read while the next
// is written: one barrier a stage.  It stands before the last group of a step, whose operands are in registers by then.  A
// tile is laid out by operand: [16 columns][column half][batch row][16 bytes], batch rows xor-ed with the column tile:
// reads and writes without bank conflicts.  Operand A is the matrix, B the activations: a lane ends with four
// consecutive matrix rows of one batch row and stores 8 bytes.
//
// Unit = (group of RG pairs, batch tile); a workgroup keeps one k range and walks its units with the pipeline running
// across their boundaries.  The slices of a unit meet in LDS at its end, each wave adding up a share.  S > 1 (few
// units): fp32 partial results.
//
// A wave-load of NB batch tiles takes about 0.64 + 0.099 NB us on a full chip, where the matrix cores alone need
// 0.107 NB at 2.4 GHz and the decode by itself 0.53: it is bound by issue (95 vector instructions beside 8 NB products
// a wave-load, a product taking the slots of two) and, with every CU busy, by the clock: 1024 rows of 8192x8192 run at
// 1.18 PFLOP/s, the library's product of the decoded matrix at 1.20.  us per product from cold memory, launches
// and sums of ranges included, 2 bits: a kernel that decodes, then multiplies between two barriers, in passes of 128 rows / here
// with fine sums / with long ones (qtip_gemm_plan.h):
//   4096x4096     45 rows 15.4 / 15.1 / 12.5, 128 31 / 19 / 17, 250 60 / 30 / 20, 1000 242 / 115 / 42
//   22016x4096    45 rows 28.7 / 24.8 / 24.4, 128 53 / 42 / 37, 250 105 / 72 / 55, 1000 420 / 286 / 181
//   28672x8192    45 rows 51 / 45 / 46, 128 92 / 69 / 70, 250 178 / 127 / 111, 1000 701 / 510 / 419
//   4096x11008    45 rows 20.9 / 19.6 / 18.4, 128 38 / 28 / 27, 250 73 / 46 / 39, 1000 289 / 183 / 93
//   8192x28672    45 rows 51 / 46 / 45, 128 85 / 68 / 69, 250 166 / 122 / 115, 1000 653 / 479 / 409

template <int K>
struct SlotMap {  // slot r = 0..7 of a column half kh: register of P, and where its two halves' words go
  static constexpr __device__ int reg(int kh, int r) {
    if (K == 4) return ((r >> 2) * 4 + 2 * kh + ((r >> 1) & 1)) * 2 + (r & 1);
    return ((r >> 2) * 2 + kh) * 4 + (r & 3);
  }
  static constexpr __device__ int word(int r, int h) {  // 4 * (2 mh + rh) + w
    if (K == 4) return 4 * (2 * ((r >> 1) & 1) + (r & 1)) + (r >> 2) + 2 * (1 - h);
    return 4 * (2 * h + (r & 1)) + (r >> 2) + 2 * ((r & 3) >> 1);
  }
};

// CUT: k ends inside a stage (k no multiple of 64 KS).
template <int K, int NB, int RG, bool CUT, typename TOut>
__global__ __launch_bounds__(64 * kRowsWaves, 1) void gemm_rows_kernel(
    TOut* __restrict__ dst, const uint8_t* __restrict__ packed, const uint16_t* __restrict__ x,
    const uint32_t* __restrict__ tlut, int m, int k, int batch, int nbt, long ldo, int round_f16, int wl_per, int upw_q,
    int upw_r) {
  constexpr int WAVES = kRowsWaves, THREADS = 64 * WAVES, KS = WAVES / RG, BT = 16 * NB;
  constexpr int HS = rows_stage_halves(NB, RG);      // column halves of a wave-load in a stage
  constexpr uint32_t OCB = BT * 16;                  // bytes of one operand chunk over the rows of a tile
  constexpr uint32_t TILE = KS * 2 * HS * 2 * OCB;
  constexpr int CPR = KS * HS * 4;                   // 16-byte pieces of a row per stage
  constexpr int CHUNKS = BT * CPR;
  constexpr int NX = (CHUNKS + THREADS - 1) / THREADS;  // pieces per thread
  static_assert(2 * TILE <= kGemmTileBytes, "two tiles");
  extern __shared__ __align__(16) uint8_t smem[];
  uint32_t* lut = reinterpret_cast<uint32_t*>(smem);
  uint8_t* tile = smem + kLut128Bytes;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rg = wave % RG, ks = wave / RG;
  const int r8 = lane & 7, pb = (lane >> 3) & 1, ch = (lane >> 4) & 1, g0 = lane >> 5;
  const uint32_t slot4 = lds_address(lut) + ((uint32_t)(lane & 31) << 2);
  const int nkb = k >> 5, nwl = (nkb + 1) >> 1, nrb = m >> 5, npair = (nrb + 1) >> 1;
  const uint32_t rb_bytes = (uint32_t)nkb * 128 * K;
  constexpr uint32_t WL_BYTES = 256 * K;
  const uint32_t loff = (uint32_t)pb * rb_bytes + (uint32_t)g0 * (128 * K) + (uint32_t)(2 * r8 + ch) * (8 * K);
  const int nxt4 = (ch ? ((lane & ~23) | ((r8 + 1) & 7)) : (lane | 16)) << 2;
  const __amdgpu_buffer_rsrc_t rs_w = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(packed), 0, (int)((size_t)nrb * rb_bytes), 0x00020000);
  const __amdgpu_buffer_rsrc_t rs_x =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(x), 0, (int)((size_t)batch * k * 2), 0x00020000);

  const int s = blockIdx.x;
  const int u0 = blockIdx.y, ustep = gridDim.y;
  const int wl0 = s * wl_per;
  const int wl1 = wl0 + wl_per < nwl ? wl0 + wl_per : nwl;
  const int nst = (wl1 - wl0 + KS - 1) / KS;  // wave-loads of a wave per unit
  const int upw = upw_q + (u0 < upw_r ? 1 : 0);
  const int T = upw * nst;
  TOut* out_s = dst + (size_t)s * batch * ldo;
  const int kend = 64 * wl1 < k ? 64 * wl1 : k;
  const int last_cols = CUT ? kend - 64 * (wl0 + KS * (nst - 1)) : 64 * KS;  // columns of the last stage

  // ---- units of this workgroup; the weights, the activations and the products each have a place of their own in
  // them, one ahead of the other.  Inside a unit only a scalar offset changes.  (The compiler takes what comes
  // out of these closures for values of a lane: without `uni` every load of activations was a loop over lanes.)
  const int dg = __builtin_amdgcn_readfirstlane(ustep / nbt), db = ustep - dg * nbt;
  auto uni = [](auto v) { return __builtin_amdgcn_readfirstlane(v); };
  struct Unit {
    int left, g, b;  // units to go, group, batch tile
  };
  auto advance = [&](Unit& u) {
    --u.left;
    u.g += dg;
    u.b += db;
    if (u.b >= nbt) {
      u.b -= nbt;
      ++u.g;
    }
  };
  const int g_first = __builtin_amdgcn_readfirstlane(u0 / nbt);
  const Unit first = {upw, g_first, u0 - g_first * nbt};
  constexpr uint32_t OUT = 0x7FFFFF00u;  // a lane offset that is out of range by itself
  // ---- weight stream of this wave, two wave-loads in flight
  LaneData<K> buf[2];
  // Where a range ends inside a stage, weights and activations there are zeros without a memory access: of every lane in a
  // slice past the end, of the second column block where that is missing.  Such weights would decode to table entry 0,
  // which may be infinite: see cut_words.
  const bool w_over = CUT && wl0 + KS * (nst - 1) + ks >= wl1;
  const bool w_half = CUT && !w_over && (nkb & 1) && wl0 + KS * (nst - 1) + ks == nwl - 1;
  const int cut_left = w_over || w_half ? 1 : 0;  // wave-loads to go in a unit where that is so, 0: nowhere
  Unit wu = first;
  int w_left;
  uint32_t w_so, w_vo;
  auto w_last = [&]() {  // before the last wave-load of a unit
    if (w_over) w_so -= (uint32_t)(KS * (nst - 1) + ks) * WL_BYTES;  // (a place that is there)
    if (w_over || (w_half && g0)) w_vo = OUT;
  };
  auto w_unit = [&]() {
    const int pair = wu.g * RG + rg;
    const bool ok = wu.left > 0 && pair < npair;
    w_so = ok ? (uint32_t)(2 * pair) * rb_bytes + (uint32_t)(wl0 + ks) * WL_BYTES : (uint32_t)(wl0 + ks) * WL_BYTES;
    w_vo = ok && 2 * pair + pb < nrb ? loff : OUT;
    w_left = nst;
    if (nst == 1) w_last();
  };
  auto issue = [&](int d) {
    buf[d] = load_lane_buf<K>(rs_w, w_vo, uni(w_so));
    w_so += KS * WL_BYTES;
    --w_left;
  };
  auto w_next = [&]() {  // after an issue()
    if (uni(w_left) <= 1) {
      if (uni(w_left) == 0) {
        advance(wu);
        w_unit();
      } else {
        w_last();
      }
    }
  };
  w_unit();
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
  issue(0);
  w_next();

  // ---- activation tiles
  u32x4 xg[NX];
  uint32_t xv[NX], xlds[NX];
  Unit xu = first;
  int x_left;
  uint32_t x_so;
  auto x_offsets = [&](int cols) {  // lane offsets of the unit's rows and the first `cols` columns of the stage
    const int rows_left = xu.left > 0 ? batch - xu.b * BT : 0;
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const int idx = i * THREADS + tid;
      const int bb = idx / CPR, c = idx % CPR, q = c >> 1;
      const int col = HS == 2 ? 8 * c : 32 * q + 8 * (c & 1);
      xlds[i] = (uint32_t)(2 * q) * OCB + ((uint32_t)(bb ^ (2 * (q & 7))) << 4) + 8 * (c & 1);
      xv[i] = bb < rows_left && col < cols && (CHUNKS % THREADS == 0 || idx < CHUNKS) ? ((uint32_t)bb * (uint32_t)k + (uint32_t)col) * 2 : OUT;
    }
  };
  auto x_unit = [&]() {
    x_so = xu.left > 0 ? ((uint32_t)(xu.b * BT) * (uint32_t)k + (uint32_t)(64 * wl0)) * 2 : 0u;
    x_left = nst;
    x_offsets(nst == 1 ? last_cols : 64 * KS);
  };
  auto load_tile = [&](int h) {  // (h: column half, HS == 1)
#pragma unroll
    for (int i = 0; i < NX; ++i) xg[i] = __builtin_amdgcn_raw_buffer_load_b128(rs_x, xv[i], uni(x_so), 0);
    x_so += HS == 2 ? KS * 128 : (h ? KS * 128 - 32 : 32);
    if (HS == 2 || h) --x_left;
  };
  auto x_next = [&]() {  // after the load of a stage's last tile
    if (uni(x_left) <= 1) {
      if (uni(x_left) == 0) {
        advance(xu);
        x_unit();
      } else if (last_cols < 64 * KS) {
        x_offsets(last_cols);
      }
    }
  };
  x_unit();
  auto store_tile = [&](uint32_t base) {
#pragma unroll
    for (int i = 0; i < NX; ++i)
      if (CHUNKS % THREADS == 0 || i * THREADS + tid < CHUNKS) {
        *reinterpret_cast<u32x2*>(tile + base + xlds[i]) = u32x2{xg[i][0], xg[i][1]};
        *reinterpret_cast<u32x2*>(tile + base + xlds[i] + OCB) = u32x2{xg[i][2], xg[i][3]};
      }
  };
  load_tile(0);
  if (HS == 2) x_next();
#pragma unroll
  for (int it = 0; it < 2 * NTW; ++it) {
    const uint32_t w = tw[it % NTW] ^ ((uint32_t)(it / NTW) << 15);
    const u32x4 v = {w, w, w, w};
    reinterpret_cast<u32x4*>(lut)[it * THREADS + tid] = v;
  }
  store_tile(0);
  load_tile(1);
  x_next();
  issue(1);
  w_next();
  __syncthreads();

  float4_t acc[4][NB];  // [2 mh + rh][batch tile]
#pragma unroll
  for (int i = 0; i < 4 * NB; ++i) (&acc[0][0])[i] = float4_t{0.f, 0.f, 0.f, 0.f};
  // read addresses of the two column halves
  uint32_t ra[HS];
#pragma unroll
  for (int h = 0; h < HS; ++h) {
    const uint32_t q = (uint32_t)((ks * 2 + g0) * HS + h);
    ra[h] = lds_address(tile) + (2 * q + ch) * OCB + ((uint32_t)((lane & 15) ^ (2 * (q & 7))) << 4);
  }
  typedef __attribute__((address_space(3))) const u32x4 lds_u32x4_t;
  auto read_x = [&](int kh, uint32_t cb, int nb) {
    return *(lds_u32x4_t*)(uintptr_t)(ra[HS == 2 ? kh : 0] + cb + (uint32_t)nb * 256);
  };
  uint32_t P[16];
  uint32_t W[2][16];
  // the successors' pieces are asked for ahead of the states that need them
  uint32_t nv[4];
  auto fetch_next = [&](int d) {
    int c = 0;
    uint32_t unused[16];
    packed_states<K>(buf[d], unused, [&](uint32_t v) {
      nv[c++] = (uint32_t)__builtin_amdgcn_ds_bpermute(nxt4, (int)v);
      return 0u;
    });
  };
  auto states = [&](int d) {
    int c = 0;
    packed_states<K>(buf[d], P, [&](uint32_t) { return nv[c++]; });
  };
  auto lookup = [&](int kh, int r, uint32_t* w) {
    const uint32_t q = pk_hash(P[SlotMap<K>::reg(kh, r)]) & 0xFFC0FFC0u;
    w[SlotMap<K>::word(r, 0)] = lds_word_abs(lut128_addr_lo(q, slot4));
    w[SlotMap<K>::word(r, 1)] = lds_word_abs(lut128_addr_hi(q, slot4));
  };
  // Before a wave-load that is cut short, with its first half looked up and its states at hand: finite words in place of
  // what meets no activations.  (Words cleared before the products of either half cost every wave-load two branches: 1 % on
  // average, 5 % at 128 rows of 5120x13824; this costs 0.7 % at 1000 rows of 4096x22016, so whole stages have kernels without.)
  uint32_t finite = 0;  // a state of a finite table entry, in both halves
  if (CUT && cut_left) {
    for (uint32_t s2 = 0; s2 < 4096u * 0x10001u; s2 += 0x10001u) {
      const uint32_t w = uni(lds_word_abs(lut128_addr_lo(pk_hash(s2) & 0xFFC0FFC0u, slot4)));
      if ((w & 0x7C00u) != 0x7C00u && (w & 0x7C000000u) != 0x7C000000u) {
        finite = s2;
        break;
      }
    }
  }
  auto cut_words = [&]() {
    const bool none = w_over || g0;
#pragma unroll
    for (int i = 0; i < 16; ++i) W[0][i] = none ? 0u : W[0][i];
#pragma unroll
    for (int r = 0; r < 8; ++r) P[SlotMap<K>::reg(1, r)] = none ? finite : P[SlotMap<K>::reg(1, r)];
  };
  constexpr int GN = NB >= 4 ? 2 : 1, NG = NB / GN;  // batch tiles per group of instructions
  u32x4 xa[2 * GN];
  fetch_next(0);
  states(0);
#pragma unroll
  for (int r = 0; r < 8; ++r) lookup(0, r, W[0]);
#pragma unroll
  for (int i = 0; i < GN; ++i) xa[i] = read_x(0, 0, i);
  // slots looked up before group gr: none in the last group, the first two of a wave-load after its states
  auto slot_at = [](int kh, int gr) constexpr -> int {
    if (gr >= NG - 1) return 8;
    if (NG == 4) return kh == 0 ? 3 * gr : (gr == 0 ? 0 : (gr == 1 ? 2 : 5));
    return gr == 0 ? 0 : 8 * gr / (NG - 1);
  };
  Unit cu = first;
  int c_left = nst;
  if (CUT && nst == cut_left) cut_words();
  for (int left = T; left > 0; left -= 2) {
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      if (d == 1 && left == 1) break;
#pragma unroll
      for (int kh = 0; kh < 2; ++kh) {
        const int st = HS == 2 ? d : kh;  // parity of the stage
        const uint32_t cb = (uint32_t)st * TILE, nbuf = (uint32_t)(st ^ 1) * TILE;
        const bool stage_end = HS == 1 || kh == 1;
#pragma unroll
        for (int gr = 0; gr < NG; ++gr) {
          if (kh == 1 && gr == 0) states(d ^ 1);
          if (kh == 0 && gr == 0) issue(d);
          if (kh == 0 && gr == NG - 1) fetch_next(d ^ 1);
          if (stage_end && gr == (NG > 2 ? 1 : 0)) store_tile(nbuf);
          if (stage_end && gr == NG - 1) {
            // every wave has read this tile and written the next (no reads or lookups of the products to come are
            // in flight here, so the wait costs nothing)
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(0xF | (3 << 14) | (7 << 4));  // lgkmcnt(0)
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
          }
#pragma unroll
          for (int i = 0; i < GN; ++i)
            xa[GN + i] = gr + 1 < NG ? read_x(kh, cb, (gr + 1) * GN + i) : read_x(kh ^ 1, stage_end ? nbuf : cb, i);
          if (stage_end && gr == (NG > 2 ? 2 : NG - 1)) load_tile(kh);
#pragma unroll
          for (int r = 0; r < 8; ++r)
            if (r >= slot_at(kh, gr) && r < slot_at(kh, gr + 1)) lookup(kh ^ 1, r, W[kh ^ 1]);
#pragma unroll
          for (int i = 0; i < GN; ++i)
#pragma unroll
            for (int mr = 0; mr < 4; ++mr) {
              const u32x4 wv = {W[kh][4 * mr], W[kh][4 * mr + 1], W[kh][4 * mr + 2], W[kh][4 * mr + 3]};
              acc[mr][gr * GN + i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                  __builtin_bit_cast(half8_t, wv), __builtin_bit_cast(half8_t, xa[i]), acc[mr][gr * GN + i], 0, 0, 0);
            }
#pragma unroll
          for (int i = 0; i < GN; ++i) xa[i] = xa[GN + i];
#pragma unroll
          for (int i = 0; i < 4 * GN; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x080, 1, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      w_next();
      x_next();
      if (uni(--c_left) > (CUT ? cut_left : 0)) continue;
      if (c_left == 0) {
        c_left = nst;
        const int pair = cu.g * RG + rg;
        const int row = 64 * pair + 32 * g0 + 4 * ch;
        const int b0 = cu.b * BT + (lane & 15);
        const uint32_t cb = (HS == 2 ? (uint32_t)d : 1u) * TILE;  // (a tile every wave is done with)
        auto put = [&](float4_t v, int bb, int r) {
          if (bb < batch && r < m) {
            typedef TOut out4_t __attribute__((ext_vector_type(4), aligned(sizeof(TOut))));  // (out may start anywhere)
            out4_t y;
#pragma unroll
            for (int e = 0; e < 4; ++e) y[e] = (TOut)(sizeof(TOut) == 4 && round_f16 ? (float)(_Float16)v[e] : v[e]);
            *reinterpret_cast<out4_t*>(out_s + (size_t)bb * ldo + r) = y;
          }
        };
        if constexpr (KS == 1) {
#pragma unroll
          for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int mr = 0; mr < 4; ++mr) put(acc[mr][nb], b0 + 16 * nb, row + 8 * mr);
        } else {
          // the k slices: wave ks keeps the vectors mr of its share, the others send theirs through LDS that is free
          constexpr int OWN = 4 / KS;  // values of mr a wave keeps
          constexpr bool SPARE = kGemmTileBytes - 2 * TILE > TILE;
          constexpr uint32_t ROOM = SPARE ? kGemmTileBytes - 2 * TILE : TILE;
          constexpr int V = ROOM >= WAVES * 2048u ? 2 : 1;  // vectors a wave sends per step
          static_assert(ROOM >= WAVES * 1024u * V, "the exchange does not fit");
          float* xch = reinterpret_cast<float*>(tile + (SPARE ? 2 * TILE : cb));
#pragma unroll
          for (int f0 = 0; f0 < OWN * NB; f0 += V) {
            float4_t mine[V];
#pragma unroll
            for (int t = 0; t < V; ++t) {
              const int o = (f0 + t) % OWN, nb = (f0 + t) / OWN;
              mine[t] = acc[o][nb];
#pragma unroll
              for (int z = 1; z < KS; ++z) mine[t] = ks == z ? acc[z * OWN + o][nb] : mine[t];
            }
#pragma unroll
            for (int z = 1; z < KS; ++z) {  // to wave ks ^ z
#pragma unroll
              for (int t = 0; t < V; ++t) {
                const int o = (f0 + t) % OWN, nb = (f0 + t) / OWN;
                float4_t v = acc[z * OWN + o][nb];
#pragma unroll
                for (int y = 1; y < KS; ++y) v = ks == y ? acc[(y ^ z) * OWN + o][nb] : v;
                *reinterpret_cast<float4_t*>(xch + ((wave * V + t) * 64 + lane) * 4) = v;
              }
              __syncthreads();
              const int from = (ks ^ z) * RG + rg;
#pragma unroll
              for (int t = 0; t < V; ++t)
                mine[t] += *reinterpret_cast<const float4_t*>(xch + ((from * V + t) * 64 + lane) * 4);
              __syncthreads();
            }
#pragma unroll
            for (int t = 0; t < V; ++t)
              put(mine[t], b0 + 16 * ((f0 + t) / OWN), row + 8 * (ks * OWN + (f0 + t) % OWN));
          }
        }
#pragma unroll
        for (int i = 0; i < 4 * NB; ++i) (&acc[0][0])[i] = float4_t{0.f, 0.f, 0.f, 0.f};
        advance(cu);
      }
      if (CUT && uni(c_left) == cut_left) cut_words();
    }
  }
}
