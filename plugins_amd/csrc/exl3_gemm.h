// exl3_gemm.h -- the EXL3 GEMM for MI355X (gfx950, wave64): more than 16
// rows, weights decoded in the registers of the waves that multiply them.
// Included by exl3_kern.h.  Paths in citations are relative to
// /root/reference/plugins/.
#pragma once

namespace exl3 {

// A workgroup is CW x KP waves over 32 MR rows x 64 CW columns: wave w takes
// columns 64 (w % CW) .. + 63 over k-part w / CW of the workgroup's k range.  A
// step of a wave is 32 k (two k-tile rows): lane l = 32 h + 8 t + c decodes
// chunk c of tile t in k-tile row 2 s + h -- 32 weights, columns 16 t + c and
// 16 t + c + 8 over the row's 16 k -- into four 8 x f16 operands of
// v_mfma_f32_32x32x16_f16, each used against the MR row blocks.  The weights
// are the first operand, so the accumulators hold z^T: lane l has row l % 32
// of a block and, in register r of column set j, column 16 (r / 4) + 8 j +
// 4 h + r % 4 of the wave's 64.
//
// Decoding into operand registers leaves LDS to the activations and the
// packed words (no store and no barrier between a weight's decode and its
// use), and the wave's own MFMAs run beside the decode of its next operand.
// Both come by direct global-to-LDS loads, 64 k (a stage) at a time, one
// barrier a stage: the activations (shared by the CW waves of a k-part) a
// stage ahead, the words (one wave's own) two.
//
// What bounds it: issue slots.  A decoded weight costs ~4 VALU instructions a
// wave (mul1, the whole kernel's) however many rows use it, an MFMA 32 matrix
// cycles, so the decode outweighs the MFMAs up to 64 rows and equals them at
// 128.  Of the SIMDs' busy cycles VALU instructions issue in 90 % and MFMAs run
// in 32 % for routed experts of 32 slots each (256 of 7168 x 2048, K = 3, gate +
// up); in 45 and 35 % for 4096 -> 2 x 12288 at 203 rows, 43 and 17 % for 4096 ->
// 12288 at 40, whose single round of workgroups waits for its first data and
// its finish.
constexpr int RD_BK = 64;
// The dense GEMM's workgroup shapes (gemm_rd_plan chooses).
struct RdShape {
  int mr, cw, kp;
};
constexpr RdShape RD_SHAPES[] = {{1, 4, 2}, {2, 4, 2}, {4, 4, 2}};
__host__ __device__ constexpr int rd_threads(int CW, int KP) { return 64 * CW * KP; }
// finish exchange: 32 rows of the 64 CW columns (f32), rows padded so that a
// 16-row run of 16-byte stores touches distinct banks; rd_pass of them (with
// two k-parts each part's waves own a row block)
__host__ __device__ constexpr int rd_fld(int CW) { return 64 * CW + 4; }
__host__ __device__ constexpr int rd_pass(int MR, int KP) { return MR > 1 && KP > 1 ? 2 : 1; }
__host__ __device__ constexpr int rd_fbytes(int CW) { return 32 * rd_fld(CW) * 4; }

// Dwords of a tile at rate K, or (FR > 0) at the half-integer rate n = 8 FR.
template <int K, int FR>
__host__ __device__ constexpr int rd_nw() { return FR > 0 ? 4 * FR : 8 * K; }
// Direct loads (1 KiB each) of a wave's words of a stage: 16 tiles.
template <int K, int FR>
__host__ __device__ constexpr int rd_wi() { return (rd_nw<K, FR>() * 4 + 63) / 64; }
template <int K, int FR, int MR, int CW, int KP>
__host__ __device__ constexpr int rd_main_bytes(int wr) {
  return 2 * KP * MR * 4096 + CW * KP * wr * rd_wi<K, FR>() * 1024;
}
// Word stages in LDS: three, or two where three leave the tile past 160 KiB
// (or a rate above 6 bits).
template <int K, int FR, int MR, int CW, int KP>
__host__ __device__ constexpr int rd_wr() {
  return rd_wi<K, FR>() <= 3 && rd_main_bytes<K, FR, MR, CW, KP>(3) <= 160 * 1024 ? 3 : 2;
}
template <int K, int FR, int MR, int CW, int KP>
__host__ __device__ constexpr int rd_lds_bytes() {
  const int main = rd_main_bytes<K, FR, MR, CW, KP>(rd_wr<K, FR, MR, CW, KP>());
  const int fin = rd_pass(MR, KP) * rd_fbytes(CW);
  return main > fin ? main : fin;
}
// Waves a SIMD the registers are budgeted for: four where the accumulators
// leave it (MR <= 2), two at MR 4; fewer where the workgroups' LDS allows
// fewer.
template <int K, int FR, int MR, int CW, int KP>
__host__ __device__ constexpr int rd_waves() {
  static_assert(MR <= 4, "two waves a SIMD hold the accumulators");
  const int regs = MR <= 2 ? 4 : 2, wg = CW * KP / 4;  // wg: waves a SIMD each
  const int lds = 160 * 1024 / rd_lds_bytes<K, FR, MR, CW, KP>() * wg;
  return lds < regs ? lds : regs;
}

// A pointer that is the same in every lane, in scalar registers.
__device__ __forceinline__ const char *uniform_ptr(const char *p) {
  const uint64_t v = (uint64_t)(uintptr_t)p;
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
  return (const char *)(uintptr_t)(((uint64_t)hi << 32) | lo);
}

// Where a workgroup's k-part reads: byte addresses, uniform within a wave
// but for the per-lane offsets.
struct RdSrc {
  const char *x;    // activations at the k-part's first stage
  const char *tw;   // words at the k-part's first stage and the wave's tiles
  uint32_t wrow;    // bytes of a k-tile row
  int stages;       // stages of the k-part (>= 1)
};

// The main loop: acc += W^T x over the wave's k-part.  va[u]: byte offset of
// the lane's piece of activation load u (rows 8 (NA cw + u) + l / 8, piece
// (l % 8) ^ ((row / 2) % 8) at place l % 8: a fragment read of 16 consecutive
// rows of one piece touches 16 distinct bank groups).
template <int K, int CB, bool MASKED, int MR, int CW, int KP, int FR>
__device__ __forceinline__ void rd_main(f16v_t (&acc)[MR][2], char *smem, const RdSrc &src,
                                        const uint32_t (&va)[4 * MR / CW], const CbRow &dec) {
  constexpr int NW = rd_nw<K, FR>(), WI = rd_wi<K, FR>(), WR = rd_wr<K, FR, MR, CW, KP>();
  constexpr int NA = 4 * MR / CW;          // activation loads a wave makes a stage
  constexpr int ABYTES = MR * 4096;        // one k-part's activations of a stage
  constexpr int ABUF = KP * ABYTES;
  constexpr int W0 = 2 * ABUF;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int cw = wave % CW, kp = wave / CW;
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
  const int NS = src.stages;

  // the lane's 16-byte pieces of the wave's words: 4 k-tile rows of NW pieces
  // (4 tiles), in order
  uint32_t vw[WI];
#pragma unroll
  for (int u = 0; u < WI; ++u) {
    const int p = min(64 * u + lane, 4 * NW - 1);
    vw[u] = (uint32_t)(p / NW) * src.wrow + (uint32_t)(p % NW) * 16u;
  }
  const uint32_t la = lds0 + kp * ABYTES + cw * (NA * 1024);
  const uint32_t lw = lds0 + W0 + wave * (WR * WI * 1024);
  // (stages past the last read the last one again: every stage issues the
  // same loads, so the waits stay exact)
  auto load_a = [&](int st, int u) {
    const char *b = uniform_ptr(src.x + (size_t)min(st, NS - 1) * (RD_BK * 2));
    lds_dma16(b, va[u], la + (st & 1) * ABUF + u * 1024);
  };
  auto load_w = [&](int st, int slot, int u) {
    const char *b = uniform_ptr(src.tw + (size_t)min(st, NS - 1) * (4 * (size_t)src.wrow));
    lds_dma16(b, vw[u], lw + slot * (WI * 1024) + u * 1024);
  };

  // per-lane LDS offsets: activation fragment f (k rows 0-7, 8-15 of the
  // lane half's k-tile row) of step s; the words of the lane's chunk
  const int h = lane >> 5, r = lane & 31;
  uint32_t ax[2][2];
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int f = 0; f < 2; ++f)
      ax[s][f] = kp * ABYTES + r * 128 + 16 * ((4 * s + 2 * h + f) ^ ((r >> 1) & 7));
  const uint32_t wt = W0 + wave * (WR * WI * 1024) + (h * 4 + ((lane >> 3) & 3)) * (NW * 4);
  const int c = lane & 7;

  // a chunk's words as the decode takes them
  constexpr int WN = FR > 0 ? gf_nb<FR>() : K + 1;
  // FR: the dword offsets of the chunk in its tile and the realigning shift
  constexpr int LW = FR > 0 ? gf_nb<FR>() + 1 : 1;
  uint32_t foff[LW];
  uint32_t fsh = 0;
  if constexpr (FR > 0) {
    // the chunk's history halfword hs (stream order: halfword s is the high
    // half of dword s / 2 when s is even, the low half when odd)
    const int hs = (c * FR - 1 + 8 * FR) % (8 * FR);
    const bool low = (hs & 1) != 0;
    const int b0 = (hs >> 1) - (low ? 0 : 1);
    fsh = low ? 16u : 0u;
#pragma unroll
    for (int j = 0; j < LW; ++j) foff[j] = (uint32_t)((b0 + j + NW) % NW) * 4u;
  }
  const uint32_t coff = FR > 0 ? 0u : (uint32_t)(c * K) * 4u;
  const uint32_t hoff = FR > 0 ? 0u : (uint32_t)(((c + 7) & 7) * K + K - 1) * 4u;
  auto read_words = [&](uint32_t (&wd)[WN], uint32_t slot_off, int s) {
    const char *p = smem + wt + slot_off + s * (8 * NW * 4);
    if constexpr (FR > 0) {
      uint32_t raw[LW];
#pragma unroll
      for (int j = 0; j < LW; ++j) raw[j] = *reinterpret_cast<const uint32_t *>(p + foff[j]);
#pragma unroll
      for (int j = 0; j < WN; ++j) wd[j] = __builtin_amdgcn_alignbit(raw[j], raw[j + 1], fsh);
    } else {
      wd[0] = *reinterpret_cast<const uint32_t *>(p + hoff);
      // a chunk of 4 or 8 dwords sits at a multiple of 16 bytes, of 2 or 6
      // at one of 8
      if constexpr (K % 4 == 0) {
#pragma unroll
        for (int i = 0; i < K; i += 4) {
          const u4_t v = *reinterpret_cast<const u4_t *>(p + coff + 4 * i);
          wd[i + 1] = v[0], wd[i + 2] = v[1], wd[i + 3] = v[2], wd[i + 4] = v[3];
        }
      } else if constexpr (K % 2 == 0) {
#pragma unroll
        for (int i = 0; i < K; i += 2) {
          const u2_t v = *reinterpret_cast<const u2_t *>(p + coff + 4 * i);
          wd[i + 1] = v[0], wd[i + 2] = v[1];
        }
      } else {
#pragma unroll
        for (int i = 0; i < K; ++i)
          wd[i + 1] = *reinterpret_cast<const uint32_t *>(p + coff + 4 * i);
      }
    }
  };
  auto operand = [&](auto F, const uint32_t (&wd)[WN]) {
    constexpr int f = decltype(F)::value;
    uint32_t v[4];
    static_for<4>([&](auto J) {
      constexpr int pr = gm_pair(f, decltype(J)::value);
      if constexpr (FR > 0)
        v[J] = decode_pair_cw<CB, MASKED>(chunk_cw_frac<FR, 2 * pr>(wd),
                                          chunk_cw_frac<FR, 2 * pr + 1>(wd), dec);
      else
        v[J] = chunk_pair_cw<K, CB, MASKED, pr>(wd, dec);
    });
    const u4_t u = {v[0], v[1], v[2], v[3]};
    return bits<h8_t>(u);
  };
  // The stage in eight slots, one per operand o = 4 s + 2 f + j (step s,
  // fragment f, column set j): the MR MFMAs of operand o, decoded in the slot
  // before, issue between the instructions that decode operand o + 1.  The
  // activation fragments of a pair of slots are read two slots ahead.  The
  // stage's barrier stands before its last pair, whose fragments are in
  // registers by then: behind it the next stage's first fragments and words
  // are read, and the loads of two (words: WR) stages on start into the
  // buffers just freed, a few each slot over six slots (issued together they
  // hold every wave at the address unit: 8 waves x 6 KiB at 64 bytes a cycle).
  h8_t af[2][MR], op[2];
  uint32_t wd[2][WN];
  auto read_a = [&](auto Q, uint32_t abuf) {  // fragments of slots 2 q, 2 q + 1
    constexpr int q = decltype(Q)::value;
#pragma unroll
    for (int i = 0; i < MR; ++i)
      af[q & 1][i] =
          *reinterpret_cast<const h8_t *>(smem + ax[q >> 1][q & 1] + abuf + i * 4096);
  };
  // the wait leaves the newest words (two stages on) in flight: loads
  // complete in issue order
  auto stage_end = [&] {
    if constexpr (WR == 2)
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else if constexpr (WI == 1)
      asm volatile("s_waitcnt vmcnt(1) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else if constexpr (WI == 2)
      asm volatile("s_waitcnt vmcnt(2) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else
      asm volatile("s_waitcnt vmcnt(3) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
  // loads of position p (0..5: slots 6, 7 and the next stage's 0..3), the
  // activations of stage sa first, then the words of stage sw into `slot`
  auto issue = [&](auto P, int sa, int sw, int slot) {
    constexpr int p = decltype(P)::value, N = NA + WI;
#pragma unroll
    for (int u = 0; u < N; ++u)
      if (u * 6 / N == p) {
        if (u < NA)
          load_a(sa, u);
        else
          load_w(sw, slot, u - NA);
      }
  };
#pragma unroll
  for (int u = 0; u < WI; ++u) load_w(0, 0, u);
#pragma unroll
  for (int u = 0; u < NA; ++u) load_a(0, u);
#pragma unroll
  for (int u = 0; u < WI; ++u) load_w(1, 1, u);
  stage_end();  // (stage 0's loads; with two word slots stage 1's words too)
  int slot = 0;
  issue(std::integral_constant<int, 0>{}, 1, WR - 1, WR - 1);
  issue(std::integral_constant<int, 1>{}, 1, WR - 1, WR - 1);
  read_a(std::integral_constant<int, 0>{}, 0);
  read_words(wd[0], 0, 0);
  read_words(wd[1], 0, 1);
  op[0] = operand(std::integral_constant<int, 0>{}, wd[0]);
  for (int st = 0; st < NS; ++st) {
    const uint32_t abuf = (st & 1) * ABUF;
    static_for<8>([&](auto O) {
      constexpr int o = decltype(O)::value;
      if constexpr (o % 2 == 0 && o < 6)
        read_a(std::integral_constant<int, o / 2 + 1>{}, abuf);
      if constexpr (o == 6) {
        stage_end();
        slot = slot == WR - 1 ? 0 : slot + 1;
        read_a(std::integral_constant<int, 0>{}, ABUF - abuf);
        read_words(wd[0], slot * (WI * 1024), 0);
      }
      // the loads of two stages on (words WR; with two word slots stage 1's
      // words came with the prologue, and so on: the slot before this one's)
      constexpr int pos = (o + 2) & 7;
      if constexpr (pos < 6) {
        const int base = o >= 6 ? st : st - 1;
        issue(std::integral_constant<int, pos>{}, base + 2, base + WR,
              slot == 0 ? WR - 1 : slot - 1);
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (o == 7) {
        op[0] = operand(std::integral_constant<int, 0>{}, wd[0]);
        read_words(wd[1], slot * (WI * 1024), 1);
      } else {
        op[(o + 1) & 1] = operand(std::integral_constant<int, (o + 1) & 3>{}, wd[(o + 1) >> 2]);
      }
#pragma unroll
      for (int i = 0; i < MR; ++i)
        acc[i][o & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(op[o & 1], af[(o >> 1) & 1][i],
                                                               acc[i][o & 1], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < MR; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);            // one MFMA
        __builtin_amdgcn_sched_group_barrier(0x002, 30 / MR, 0);  // the decode beside it
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  }
  // no load may still write this workgroup's LDS when it is used again
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// z of one wave's row block: v[j][4 t + i] (f32 sums) = row l % 32, column
// 16 t + 8 j + 4 h + i of its 64 columns.
//
// The finish's rotation on column bits 0-5 of f16(z), in that order (each
// lo + hi, lo - hi, as the reference's kernels compute it,
// sushi_ds41/src/sushi/exl3/expert_exl3_kernels.zig:902-970): bits 0, 1 are
// i, bit 2 the lane half, bit 3 j, bits 4, 5 t.
__device__ __forceinline__ void rd_rotate64(f16v_t (&v)[2], int h) {
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int e = 0; e < 16; ++e) v[j][e] = h2f(f2h(v[j][e]));
  auto fly = [](float &a, float &b) {
    const float lo = a, hi = b;
    a = lo + hi;
    b = lo - hi;
  };
#pragma unroll
  for (int m = 1; m < 4; m <<= 1)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e)
        if (!(e & m)) {
          float a = v[j][e], b = v[j][e + m];
          fly(a, b);
          v[j][e] = a;
          v[j][e + m] = b;
        }
  const float sg = h == 0 ? 1.0f : -1.0f;
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int e = 0; e < 16; ++e) v[j][e] = butterfly(sg, v[j][e], xor_lanes(v[j][e], 32));
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    float a = v[0][e], b = v[1][e];
    fly(a, b);
    v[0][e] = a;
    v[1][e] = b;
  }
#pragma unroll
  for (int m = 4; m < 16; m <<= 1)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e)
        if (!(e & m)) {
          float a = v[j][e], b = v[j][e + m];
          fly(a, b);
          v[j][e] = a;
          v[j][e + m] = b;
        }
}

// The wave's (rotated) block into the exchange fx [32][rd_fld(CW)].
template <int CW>
__device__ __forceinline__ void rd_put(float *fx, const f16v_t (&v)[2], int cw, int lane) {
  float *p = fx + (lane & 31) * rd_fld(CW) + 64 * cw + 4 * (lane >> 5);
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int t = 0; t < 4; ++t)
      *reinterpret_cast<f4_t *>(p + 16 * t + 8 * j) =
          f4_t{v[j][4 * t], v[j][4 * t + 1], v[j][4 * t + 2], v[j][4 * t + 3]};
}

// Four consecutive finished f16 values in the output dtype; wide: the output
// array is 16-byte aligned.
__device__ __forceinline__ void store_out4(void *p, size_t i, const uint16_t (&y)[4], int dt,
                                           bool wide) {
  if (!wide) {
#pragma unroll
    for (int e = 0; e < 4; ++e) store_out(p, i + e, y[e], dt);
  } else if (dt == OUT_F32) {
    *reinterpret_cast<f4_t *>((float *)p + i) = f4_t{h2f(y[0]), h2f(y[1]), h2f(y[2]), h2f(y[3])};
  } else {
    uint32_t a, b;
    if (dt == OUT_F16) {
      a = (uint32_t)y[0] | ((uint32_t)y[1] << 16);
      b = (uint32_t)y[2] | ((uint32_t)y[3] << 16);
    } else {
      a = (uint32_t)f2bf(h2f(y[0])) | ((uint32_t)f2bf(h2f(y[1])) << 16);
      b = (uint32_t)f2bf(h2f(y[2])) | ((uint32_t)f2bf(h2f(y[3])) << 16);
    }
    *reinterpret_cast<u2_t *>((uint16_t *)p + i) = u2_t{a, b};
  }
}

// The rest of the finish over fx: the stage on column bit 6, * 1/sqrt(128)
// * svh, the output dtype; or, y null, f16(z) as it is.  THREADS threads;
// rows: valid rows of the block, orow(m): output row of its row m, ncols: the
// block's columns (a multiple of 128) from column col0 of out.
template <int THREADS, int CW, typename R>
__device__ __forceinline__ void rd_store(const float *fx, int tid, int rows, R &&orow, size_t out,
                                         int col0, int ncols, const uint16_t *svh, void *y,
                                         int ydt, uint16_t *zout) {
  const bool wide = (((uintptr_t)(y != nullptr ? y : (void *)zout)) & 15) == 0;
  constexpr int RI = 8 * CW;  // items of a row: 16 a 128-column block
  for (int e = tid; e < 32 * RI; e += THREADS) {
    const int row = e / RI, blk = (e % RI) >> 4, cl = 4 * (e & 15);
    if (row >= rows || 128 * blk >= ncols) continue;
    const float *p = fx + row * rd_fld(CW) + 128 * blk + cl;
    const f4_t lo = *reinterpret_cast<const f4_t *>(p);
    const f4_t hi = *reinterpret_cast<const f4_t *>(p + 64);
    const size_t o = orow(row) * out + col0 + 128 * blk + cl;
    uint16_t a[4], b[4];
    if (y == nullptr) {
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = f2h(lo[i]), b[i] = f2h(hi[i]);
      store_out4(zout, o, a, OUT_F16, wide);
      store_out4(zout, o + 64, b, OUT_F16, wide);
    } else {
      const uint16_t *sv = svh + col0 + 128 * blk + cl;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        a[i] = f2h(((lo[i] + hi[i]) * HAD_SCALE) * h2f(sv[i]));
        b[i] = f2h(((lo[i] - hi[i]) * HAD_SCALE) * h2f(sv[64 + i]));
      }
      store_out4(y, o, a, ydt, wide);
      store_out4(y, o + 64, b, ydt, wide);
    }
  }
}

// The end of a tile: the k-parts' sums added (part 0 + part 1), then either
// into a split's plane or finished.  With two k-parts row blocks go in pairs,
// each part's waves owning one block of the pair.  rows: valid rows of the tile;
// plane: f32 [rows][out] of this split at the tile's first row (null: finish).
template <int MR, int CW, int KP, typename R>
__device__ __forceinline__ void rd_end(f16v_t (&acc)[MR][2], char *smem, int rows, R &&orow,
                                       size_t out, int col0, int ncols, float *plane,
                                       const uint16_t *svh, void *y, int ydt, uint16_t *zout) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int cw = wave % CW, kp = wave / CW, h = lane >> 5;
  constexpr int PB = rd_pass(MR, KP);  // row blocks a pass
  constexpr int FX = rd_fbytes(CW) / 4;
  float *fx = reinterpret_cast<float *>(smem);
  auto quad = [](const f16v_t (&v)[2], int q) {
    return f4_t{v[q >> 2][4 * (q & 3)], v[q >> 2][4 * (q & 3) + 1], v[q >> 2][4 * (q & 3) + 2],
                v[q >> 2][4 * (q & 3) + 3]};
  };
  // a finished-sum block of the wave into its plane, or rotated into fx
  auto emit = [&](f16v_t (&v)[2], int ib, int region) {
    if (plane != nullptr) {
      // (32-byte runs a row: a lane holds four consecutive columns)
      if (32 * ib + (lane & 31) < rows && 64 * cw < ncols) {
        float *p = plane + (size_t)(32 * ib + (lane & 31)) * out + col0 + 64 * cw + 4 * h;
#pragma unroll
        for (int q = 0; q < 8; ++q)
          *reinterpret_cast<f4_t *>(p + 16 * (q & 3) + 8 * (q >> 2)) = quad(v, q);
      }
    } else {
      if (y != nullptr) rd_rotate64(v, h);
      rd_put<CW>(fx + region * FX, v, cw, lane);
    }
  };
  static_for<(MR + PB - 1) / PB>([&](auto P) {
    constexpr int i0 = PB * decltype(P)::value;
    if (32 * i0 >= rows) return;
    if constexpr (KP == 2) {
      // the block a wave gives away (part 1: the first of the pair, part 0:
      // the second) into its owner's exchange region, lane-contiguous
      auto give = [&](auto B) {
        constexpr int b = decltype(B)::value;
        float *p = fx + b * FX + cw * 2048 + lane * 4;
#pragma unroll
        for (int q = 0; q < 8; ++q) *reinterpret_cast<f4_t *>(p + q * 256) = quad(acc[i0 + b], q);
      };
      auto take = [&](auto B, f16v_t (&v)[2]) {
        constexpr int b = decltype(B)::value;
        const float *p = fx + b * FX + cw * 2048 + lane * 4;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const f4_t o = *reinterpret_cast<const f4_t *>(p + q * 256);
#pragma unroll
          for (int i = 0; i < 4; ++i)
            v[q >> 2][4 * (q & 3) + i] = acc[i0 + b][q >> 2][4 * (q & 3) + i] + o[i];
        }
      };
      using B0 = std::integral_constant<int, 0>;
      using B1 = std::integral_constant<int, PB - 1>;
      if (kp == 1)
        give(B0{});
      else if constexpr (PB == 2)
        give(B1{});
      lds_barrier();
      f16v_t v[2];
      if (kp == 0)
        take(B0{}, v);
      else if constexpr (PB == 2)
        take(B1{}, v);
      lds_barrier();  // the exchange is read
      if (PB == 2 || kp == 0) emit(v, i0 + (PB == 2 ? kp : 0), PB == 2 ? kp : 0);
    } else {
      emit(acc[i0], i0, 0);
    }
    if (plane != nullptr) return;
    lds_barrier();
#pragma unroll
    for (int b = 0; b < PB; ++b)
      rd_store<64 * CW * KP, CW>(
          fx + b * FX, tid, rows - 32 * (i0 + b), [&](int m) { return orow(32 * (i0 + b) + m); },
          out, col0, ncols, svh, y, ydt, zout);
    lds_barrier();
  });
}

// The dense GEMM over up to four linears that share rows, rate and codebook
// (each with its own prepared rows), column tiles side by side in grid x, row
// tiles in y, k-splits in z.
constexpr int RD_MAXW = 4;
struct RdWeight {
  const uint32_t *tw;
  const uint16_t *xp;   // [M][in]
  const uint16_t *svh;
  void *y;              // finished output in ydt, or null: zout
  uint16_t *zout;       // f16(z)
  float *kpart;         // split k: planes [split][M][out]
  int out_tiles;
  int ct0;              // first column tile in the grid
};
struct RdArgs {
  RdWeight w[RD_MAXW];
  int nw, ydt, M, in_tiles;
  CbRow dec;
};

template <int K, int CB, bool MASKED, int MR, int CW, int KP, int FR>
__global__ __launch_bounds__(rd_threads(CW, KP), (rd_waves<K, FR, MR, CW, KP>())) void
gemm_rd_kernel(RdArgs a) {
  __shared__ __attribute__((aligned(16))) char smem[rd_lds_bytes<K, FR, MR, CW, KP>()];
  constexpr int COLS = 64 * CW, CT = 4 * CW;  // columns and tiles of a column tile
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int cw = wave % CW, kp = wave / CW;
  // Workgroup n runs on XCD n % 8 (the dispatcher's round robin); taking the
  // row tile as n % (row tiles) gives each XCD a few row tiles of the
  // activations to keep in its L2.  (Only the speed depends on this.)
  const int mtiles = gridDim.y;
  const int lin = blockIdx.x + gridDim.x * blockIdx.y;
  const int gx = lin / mtiles, mt = lin % mtiles;
  const int m0 = mt * (32 * MR);
  int wi = 0;
#pragma unroll
  for (int i = 1; i < RD_MAXW; ++i)
    if (i < a.nw && gx >= a.w[i].ct0) wi = i;
  const RdWeight &W = a.w[wi];
  const int ct = gx - W.ct0;
  const int M = a.M, in = a.in_tiles * 16;
  const int out_tiles = W.out_tiles;
  const int ncols = min(COLS, out_tiles * 16 - ct * COLS);
  // k range: whole 128-input blocks per split; with two k-parts the first
  // half of the split's stages to part 0, the rest to part 1
  const int S = gridDim.z, ks = blockIdx.z;
  const int P = a.in_tiles / 8;
  const int p0 = (int)((long)P * ks / S), p1 = (int)((long)P * (ks + 1) / S);
  const int stages = (p1 - p0) * 2 / KP;    // of each k-part
  const int st0 = 2 * p0 + kp * stages;     // the part's first stage

  constexpr int NA = 4 * MR / CW;
  uint32_t va[NA];
#pragma unroll
  for (int u = 0; u < NA; ++u) {
    const int R = 8 * (NA * cw + u) + (lane >> 3);
    const int q = (lane & 7) ^ ((R >> 1) & 7);
    va[u] = (uint32_t)(((size_t)min(m0 + R, M - 1) * in + 8 * q) * 2);
  }
  constexpr int NW = rd_nw<K, FR>();
  RdSrc src;
  src.x = (const char *)W.xp + (size_t)st0 * (RD_BK * 2);
  src.wrow = (uint32_t)out_tiles * (NW * 4);
  // (columns past the last: the tile's first half again, not stored)
  const int cwe = 64 * cw < ncols ? cw : cw & 1;
  src.tw = (const char *)W.tw + (size_t)st0 * 4 * src.wrow +
           (size_t)(ct * CT + cwe * 4) * (NW * 4);
  src.stages = stages;
  f16v_t acc[MR][2];
#pragma unroll
  for (int i = 0; i < MR; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
  rd_main<K, CB, MASKED, MR, CW, KP, FR>(acc, smem, src, va, a.dec);
  const int rows = min(32 * MR, M - m0);
  const size_t out = (size_t)out_tiles * 16;
  float *plane = S > 1 ? W.kpart + ((size_t)ks * M + m0) * out : nullptr;
  rd_end<MR, CW, KP>(acc, smem, rows, [&](int m) { return (size_t)(m0 + m); },
                     out, ct * COLS, ncols, plane, W.svh, W.y, a.ydt, W.zout);
}

// ------------------------------------------------------- grouped GEMM
//
constexpr int RDG_CW = 4, RDG_ROWS = 128;

// Routed work items: workgroup (column tile, item), the item up to RDG_ROWS
// slots of one expert (sorted[start ..]); activation rows gathered by slot (xp
// holds one prepared row per slot), expert e's words and svh, outputs
// scattered to the slots' rows.  One k-part, so four-wave workgroups.  Up to
// two weights (gate and up) side by side in the column tiles.  A launch's
// items hold up to 32 MRMAX slots (2: four workgroups a CU, 4: two).
//
// Against gemm_grouped_kernel's workgroup of 256 rows x 128 columns, whose eight
// decode waves fill LDS for eight MFMA waves, on 256 experts of 7168 x 2048 at
// K = 3 with 32 slots each (moe layer of 1024 tokens): gate + up 3380 -> 1220
// us, down 1990 -> 665 us, which is 2.3 and 2.1 TB/s of packed words; 16
// experts of 4096 x 2048 with 128 / 1024 slots each, the whole call, 273 ->
// 253 and 1478 -> 1373 us.
struct RdGroupWeight {
  const uint32_t *tw;
  const uint16_t *xp;   // [slots][in]
  const uint16_t *svh;  // [E][out]
  void *y;              // [slots][out] in ydt
  size_t expert_words;  // trellis dwords per expert
  int out_tiles;
  int ct0;
};
struct RdGroupArgs {
  RdGroupWeight w[2];
  int nw, ydt, in_tiles, ct;  // ct: column tiles of all weights
  CbRow dec;
  const uint32_t *sorted;
  const MoeItem *items;
  const uint32_t *n_items;
};

template <int K, int CB, bool MASKED, int MR>
__device__ __forceinline__ void rd_group_tile(const RdGroupArgs &a, const RdGroupWeight &W, int ct,
                                              const MoeItem &item, char *smem) {
  constexpr int CW = RDG_CW, COLS = 64 * CW, NA = 4 * MR / CW, NW = rd_nw<K, 0>();
  const int lane = threadIdx.x & 63;
  const int cw = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int M = (int)item.count, in = a.in_tiles * 16, out_tiles = W.out_tiles;
  const int ncols = min(COLS, out_tiles * 16 - ct * COLS);
  auto slot_of = [&](int r) -> uint32_t { return a.sorted[item.start + r]; };
  uint32_t va[NA];
#pragma unroll
  for (int u = 0; u < NA; ++u) {
    const int R = 8 * (NA * cw + u) + (lane >> 3);
    const int q = (lane & 7) ^ ((R >> 1) & 7);
    va[u] = (uint32_t)(((size_t)slot_of(min(R, M - 1)) * in + 8 * q) * 2);
  }
  RdSrc src;
  src.x = (const char *)W.xp;
  src.wrow = (uint32_t)out_tiles * (NW * 4);
  const int cwe = 64 * cw < ncols ? cw : cw & 1;
  src.tw = (const char *)(W.tw + (size_t)item.expert * W.expert_words) +
           (size_t)(ct * 4 * CW + cwe * 4) * (NW * 4);
  src.stages = a.in_tiles / 4;
  f16v_t acc[MR][2];
#pragma unroll
  for (int i = 0; i < MR; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
  rd_main<K, CB, MASKED, MR, CW, 1, 0>(acc, smem, src, va, a.dec);
  const size_t out = (size_t)out_tiles * 16;
  rd_end<MR, CW, 1>(acc, smem, M, [&](int m) { return (size_t)slot_of(m); }, out, ct * COLS, ncols,
                    nullptr, W.svh + (size_t)item.expert * out, W.y, a.ydt, nullptr);
}

template <int K, int CB, bool MASKED, int MRMAX>
__global__ __launch_bounds__(64 * RDG_CW, (rd_waves<K, 0, MRMAX, RDG_CW, 1>())) void
gemm_rd_grouped_kernel(RdGroupArgs a) {
  __shared__ __attribute__((aligned(16))) char smem[rd_lds_bytes<K, 0, MRMAX, RDG_CW, 1>()];
  // Workgroup n runs on XCD n % 8: an item's column tiles go to one XCD, whose
  // L2 then holds the item's activations.  (Only the speed depends on this;
  // the grid holds a multiple of 8 items, some past the last.)
  const int xcd = blockIdx.x & 7, idx = blockIdx.x >> 3;
  const int it = (idx / a.ct) * 8 + xcd, gx = idx % a.ct;
  if ((uint32_t)it >= *a.n_items) return;  // the whole workgroup, before any barrier
  const MoeItem item = a.items[it];
  const int wi = a.nw > 1 && gx >= a.w[1].ct0;
  const RdGroupWeight &W = a.w[wi];
  const int ct = gx - W.ct0;
  // the row blocks that hold the item (1, 2 or 4)
  if constexpr (MRMAX > 2) {
    if ((int)item.count > 64) {
      rd_group_tile<K, CB, MASKED, 4>(a, W, ct, item, smem);
      return;
    }
  }
  if ((int)item.count > 32)
    rd_group_tile<K, CB, MASKED, 2>(a, W, ct, item, smem);
  else
    rd_group_tile<K, CB, MASKED, 1>(a, W, ct, item, smem);
}

}  // namespace exl3
