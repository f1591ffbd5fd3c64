// Prefill GEMM tiles of 64 tokens x 64 weight rows a wave (pf_tile_kernel):
// the form of every grouped prefill GEMM and of the dense ones that it runs
// faster (pt_dense_tile in glq_prefill.hip; the smaller tiles of pf_gemm_kernel
// take the rest).
//
// What bounds this contraction is neither memory nor the matrix cores alone:
// a wave's decode and scaling are vector work (per 16 codes 17 operations,
// per result and group one fma) and its A operands come from LDS.  Vector
// work and MFMAs of one SIMD overlap: 16 independent MFMA chains with v
// vector operations after each v_mfma_f32_16x16x32_f16 ran at 2137 (v = 0),
// 2117 (2), 1882 (3), 1580 (4), 1193 (6) TF/s with two waves a SIMD, and with
// the same work per v_mfma_f32_32x32x16_f16 at 2455, 2267 (2), 2076 (3), 1666
// (4).  So a wave takes 64 x 64 results: every decoded operand feeds 64
// tokens, every A operand 64 rows (half the LDS reads of a 32-row wave, which
// needed the LDS's whole read rate), at 3.7 vector operations per 16 x 16 x
// 32 products, on the 32 x 32 x 16 instruction.
//
//  * A workgroup is 4 waves, WM along the tokens x WN along the rows; a wave
//    owns MT 32-token blocks, dealt out round robin over the WM waves so that
//    a short tile's blocks spread over them, and blocks past the tile's rows
//    cost nothing.
//  * Per 128-code group one LDS slot receives the tile's A rows (16-byte piece
//    c of row r at c ^ (r % 16)) and its codes ([32-row block][piece][row]) by
//    direct global->LDS loads; a ring of D slots, one barrier a group.
//  * Lane (row li = lane % 32, half h = lane / 32): of a group's codes h holds
//    the words of its half of K, k-step t (0..7) uses slice t of them, and the
//    A operand of step t is decode-order piece 8 h + t of a token's row.
//  * Scales and zero-points: lanes of half 0 load the scale, of half 1 the
//    zero-point, and one v_permlane32_swap gives both to both; two groups a
//    load where the rows' scales are whole aligned pairs (SZQ), else one.
//  * y += s (acc - zf c2) as in pf_gemm_kernel.
#pragma once

namespace glq {

typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ f32x16 mfma_32x32x16(f16x8 a, f16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// What B is made of (template argument BITS): 2 or 4, group-quantized codes;
// kPtTurbo, 2-bit indices of a codebook with a norm per row (no groups: the
// products of all K run into y, the codebook in fp16 hi + lo parts, an MFMA
// each, the norm at the end; A in the 4-bit decode order, turbo_decode's);
// kPtHalf, fp16 rows (n, K), both operands in natural order.
constexpr int kPtTurbo = 3, kPtHalf = 16;

// fp16 codebook in v_perm_b32 form (low bytes of C0..C3, high bytes): hi part,
// or the residual of it.
__device__ __forceinline__ void pt_lut(const float* c, bool residual, uint32_t& lb, uint32_t& hb) {
  lb = hb = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const __half hi = __float2half(c[i]);
    const __half v = residual ? __float2half(c[i] - __half2float(hi)) : hi;
    const uint32_t u = __half_as_ushort(v);
    lb |= (u & 0xffu) << (8 * i);
    hb |= (u >> 8) << (8 * i);
  }
}

template <int BITS, int WM, int WN, int MT>
struct PtSlot {
  static constexpr int TM = 32 * MT * WM;           // tokens of a tile
  static constexpr int NB = 2 * WN;                 // 32-row blocks of a tile
  static constexpr int CB = BITS == 4 ? 64 : BITS == kPtHalf ? 256 : 32;  // B bytes per row per group
  static constexpr int C = TM * 256;                // A rows, then the codes
  static constexpr int BYTES = C + NB * 32 * CB;
  static constexpr int NIA = TM / 16;               // A load instructions per wave
  static constexpr int NIC = NB * CB / 128;         // code load instructions per wave
  static constexpr int NI = NIA + NIC;
  // ring depth: as many slots as let two workgroups share a CU, at most 4
  // (fp16 rows: three for one workgroup)
  static constexpr int D = BITS == kPtHalf ? 3
                                           : 4 * BYTES <= 80 * 1024 ? 4 : (3 * BYTES <= 80 * 1024 ? 3 : 2);
};

// Weight row of row li of 32-row block b (may be >= N: clamp for loads).
template <int MODE>
__device__ __forceinline__ int pt_row(int n0, int b, int li) {
  return MODE == kPfGateUp ? n0 + (b >> 1) * 32 + li : n0 + b * 32 + li;
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t pt_rsrc(const void* p) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, 0xFFFFFFFFu, 0x00027000);
}

// Column n in the decode order of out_bits (0: natural).
__device__ __forceinline__ int pt_col(int out_bits, int n) {
  return out_bits ? (n & ~15) + perm_pos_rt(out_bits, n & 15) : n;
}

// Both halves' value of a pair loaded as (scale | zero-point) by lane half.
__device__ __forceinline__ void pt_halves(uint32_t v, uint32_t& lo, uint32_t& hi) {
  const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  lo = r[0];
  hi = r[1];
}
__device__ __forceinline__ __half pt_half(uint32_t v, int odd) {
  return __ushort_as_half((unsigned short)(odd ? v >> 16 : v));
}

// pf_consts for a zero-point that is an integer wherever ZF is false: the
// constants as packed fp16 sums (exact integers; 2 + 5 operations instead of
// a conversion each).
template <int BITS, bool SYM, bool ZF>
__device__ __forceinline__ PfK<BITS> pt_consts(__half sh, __half zh, float zoff) {
  if constexpr (ZF) {
    PfK<BITS> k;
    const float z = __half2float(zh) + zoff, zi = rintf(z);
    k.zf = z - zi;
    k.s = __half2float(sh);
    const _Float16 nz = (_Float16)(-zi);
    const f16x2 n2 = {nz, nz};
    constexpr _Float16 b2[5] = {1024, 256, 64, 16, 4}, b4[2] = {1024, 64};
#pragma unroll
    for (int i = 0; i < (BITS == 2 ? 5 : 2); ++i) {
      const _Float16 b = BITS == 2 ? b2[i] : b4[i];
      k.c[i] = n2 - f16x2{b, b};
    }
    return k;
  } else {
    PfK<BITS> k;
    const _Float16 nz = SYM ? (_Float16)(float)-(1 << (BITS - 1))
                            : (_Float16)(-(__half2float(zh) + zoff));
    k.zf = 0.f;
    k.s = __half2float(sh);
    const f16x2 n2 = {nz, nz};
    constexpr _Float16 b2[5] = {1024, 256, 64, 16, 4}, b4[2] = {1024, 64};
#pragma unroll
    for (int i = 0; i < (BITS == 2 ? 5 : 2); ++i) {
      const _Float16 b = BITS == 2 ? b2[i] : b4[i];
      k.c[i] = n2 - f16x2{b, b};
    }
    return k;
  }
}

template <int BITS, int WM, int WN, int MT, int MODE, bool SYM, bool ZF, bool SZQ>
__device__ __forceinline__ void pt_body(const PfArgs& g, unsigned char* smem, int bx, int by,
                                        int bz) {
  constexpr bool SCALED = BITS == 2 || BITS == 4;
  static_assert(WM * WN == 4 && (SCALED || BITS == kPtTurbo || BITS == kPtHalf), "4 waves");
  static_assert(BITS != kPtHalf || MODE == kPfDense, "one matrix");
  using SL = PtSlot<BITS, WM, WN, MT>;
  constexpr bool TWO = MODE == kPfGateUp;
  constexpr int D = SL::D;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 31, h = lane >> 5;
  const int wm = wave % WM, wn = wave / WM;
  const int ty = by;
  int e = 0, p0, rows;
  if (g.tiles) {
    if (ty >= *g.ntiles) return;  // uniform over the workgroup
    e = g.tiles[3 * ty];
    p0 = g.tiles[3 * ty + 1];
    rows = g.tiles[3 * ty + 2];
  } else {
    p0 = ty * SL::TM;
    rows = min(SL::TM, g.M - p0);
  }
  const int n0 = bx * (TWO ? 32 : 64) * WN;
  // K split z (DOWN: fp32 results of their own, summed by the combine; split 0
  // has the low-rank term)
  const int g0 = MODE == kPfDown ? bz * g.gps : 0;

  // ---- load addresses: element offsets from uniform bases ----
  // (buffer loads: one constant offset a lane, the group's in a scalar; they
  // are also the loads to LDS past which the compiler can count the scales')
  unsigned aoff[SL::NIA];
#pragma unroll
  for (int q = 0; q < SL::NIA; ++q) {
    const int r = (wave * SL::NIA + q) * 4 + (lane >> 4);
    const int p = p0 + min(r, rows - 1);
    const unsigned ar = g.arow ? g.arow[p] : p;
    aoff[q] = 2u * (ar * (unsigned)g.K + (((lane & 15) ^ (r & 15)) << 3));
  }
  const auto arsrc = pt_rsrc(g.xp);
  __amdgpu_buffer_rsrc_t crsrc[SL::NIC];
  unsigned coff[SL::NIC];
#pragma unroll
  for (int q = 0; q < SL::NIC; ++q) {
    const int i = wave * SL::NIC + q;  // 1 KB of the slot's code region
    if constexpr (BITS == kPtHalf) {
      const int r = 4 * i + (lane >> 4);
      crsrc[q] = pt_rsrc(g.codes[0]);
      coff[q] = 2u * ((unsigned)min(pt_row<MODE>(n0, r >> 5, r & 31), g.N - 1) * (unsigned)g.K +
                      (((lane & 15) ^ (r & 15)) << 3));
    } else {
      const int b = BITS == 4 ? i >> 1 : i;
      const int piece = (BITS == 4 ? 2 * (i & 1) : 0) + h;
      crsrc[q] = pt_rsrc((TWO && (b & 1) ? g.codes[1] : g.codes[0]) + e * g.codes_es);
      coff[q] = 4u * ((unsigned)min(pt_row<MODE>(n0, b, li), g.N - 1) * g.kw + 4 * piece);
    }
  }
  // scale (half 0) or zero-point (half 1) of this lane's row in each of the
  // wave's two 32-row blocks
  const uint16_t* szp[2] = {};
  if constexpr (SCALED)
#pragma unroll
  for (int nt = 0; nt < 2; ++nt) {
    const int n = min(pt_row<MODE>(n0, 2 * wn + nt, li), g.N - 1);
    const int m = TWO ? nt : 0;
    const __half* base = (SYM || h == 0) ? g.scales[m] : g.zeros[m];
    szp[nt] = (const uint16_t*)base + e * g.sz_es + (int64_t)n * g.G + g0;
  }
  const int ng = MODE == kPfDown ? min(g.gps, g.G - g0) : g.G;
  auto issue = [&](int grp, unsigned char* slot) {
#pragma unroll
    for (int q = 0; q < SL::NIA; ++q)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          arsrc, (lds_void*)(slot + (wave * SL::NIA + q) * 1024), 16, aoff[q],
          (g0 + grp) * 256, 0, 0);
#pragma unroll
    for (int q = 0; q < SL::NIC; ++q) {
      const int i = wave * SL::NIC + q;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(crsrc[q], (lds_void*)(slot + SL::C + i * 1024), 16,
                                               coff[q], (g0 + grp) * SL::CB, 0, 0);
    }
  };

  f32x16 y[MT][2];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int j = 0; j < 16; ++j) y[i][nt][j] = 0.f;
  const DecodeConsts dk = DecodeConsts::make();
  // this wave's 32-token blocks with rows in them (block i: tokens from
  // 32 (i WM + wm))
  const int nact = max(0, min(MT, ((rows + 31) / 32 - wm + WM - 1) / WM));

  uint32_t lut[TWO ? 2 : 1][4] = {};  // codebook: hi's low and high bytes, lo's
  if constexpr (BITS == kPtTurbo)
#pragma unroll
    for (int m = 0; m < (TWO ? 2 : 1); ++m) {
      pt_lut(g.cent[m], false, lut[m][0], lut[m][1]);
      pt_lut(g.cent[m], true, lut[m][2], lut[m][3]);
    }

  // one group's products of NM token blocks
  auto group = [&](auto nm, int grp, const unsigned char* sl, const __half (&sh)[2],
                   const __half (&zh)[2], const auto& after_reads) {
    constexpr int NM = decltype(nm)::value;
    auto arow = [&](int i) { return sl + (32 * (i * WM + wm) + li) * 256; };
    auto piece = [&](int i, int p) { return *(const u32x4*)(arow(i) + ((p ^ (li & 15)) << 4)); };
    auto a_op = [&](int i, int t) { return __builtin_bit_cast(f16x8, piece(i, 8 * h + t)); };
    if constexpr (BITS == kPtHalf) {
      after_reads();
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        f16x8 bv[2];
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
          bv[nt] = *(const f16x8*)(sl + SL::C + ((2 * wn + nt) * 32 + li) * 256 +
                                   (((8 * h + t) ^ (li & 15)) << 4));
#pragma unroll
        for (int i = 0; i < NM; ++i) {
          const f16x8 av = a_op(i, t);
#pragma unroll
          for (int nt = 0; nt < 2; ++nt) y[i][nt] = mfma_32x32x16(av, bv[nt], y[i][nt]);
        }
      }
      return;
    } else if constexpr (BITS == kPtTurbo) {
      uint32_t tw[2][4];
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) {
        const u32x4 v = *(const u32x4*)(sl + SL::C + (2 * wn + nt) * 32 * SL::CB + li * 16 + h * 512);
        tw[nt][0] = v.x; tw[nt][1] = v.y; tw[nt][2] = v.z; tw[nt][3] = v.w;
      }
      f16x8 av[2][2][NM];  // [word parity][slice][block], a word ahead of its use
      auto load_a = [&](int i4) {
#pragma unroll
        for (int sl2 = 0; sl2 < 2; ++sl2)
#pragma unroll
          for (int i = 0; i < NM; ++i) av[i4 & 1][sl2][i] = a_op(i, 2 * i4 + sl2);
      };
      load_a(0);
      after_reads();
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        if (i4 < 3) load_a(i4 + 1);
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
          const int m = TWO ? nt : 0;
          uint32_t bh[2][4], bl[2][4];  // slices 0,4,1,5,.. and 8,12,9,13,.. of the word
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const uint32_t X = (tw[nt][i4] >> (2 * q)) & 0x03030303u, X4 = X | 0x04040404u;
            const uint32_t sa = __builtin_amdgcn_perm(X4, X, 0x05010400u);  // (q, q + 4)
            const uint32_t sb = __builtin_amdgcn_perm(X4, X, 0x07030602u);  // (q + 8, q + 12)
            bh[0][q] = __builtin_amdgcn_perm(lut[m][1], lut[m][0], sa);
            bh[1][q] = __builtin_amdgcn_perm(lut[m][1], lut[m][0], sb);
            bl[0][q] = __builtin_amdgcn_perm(lut[m][3], lut[m][2], sa);
            bl[1][q] = __builtin_amdgcn_perm(lut[m][3], lut[m][2], sb);
          }
#pragma unroll
          for (int sl2 = 0; sl2 < 2; ++sl2) {
            const f16x8 vh = __builtin_bit_cast(
                f16x8, u32x4{bh[sl2][0], bh[sl2][1], bh[sl2][2], bh[sl2][3]});
            const f16x8 vl = __builtin_bit_cast(
                f16x8, u32x4{bl[sl2][0], bl[sl2][1], bl[sl2][2], bl[sl2][3]});
#pragma unroll
            for (int i = 0; i < NM; ++i) {
              y[i][nt] = mfma_32x32x16(av[i4 & 1][sl2][i], vh, y[i][nt]);
              y[i][nt] = mfma_32x32x16(av[i4 & 1][sl2][i], vl, y[i][nt]);
            }
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      return;
    } else {
    uint32_t w[2][BITS == 2 ? 4 : 8];
    PfK<BITS> kc[2];
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      const unsigned char* cr = sl + SL::C + (2 * wn + nt) * 32 * SL::CB + li * 16;
      if constexpr (BITS == 2) {
        const u32x4 v = *(const u32x4*)(cr + h * 512);
        w[nt][0] = v.x; w[nt][1] = v.y; w[nt][2] = v.z; w[nt][3] = v.w;
      } else {
        const u32x4 v = *(const u32x4*)(cr + 2 * h * 512);
        const u32x4 u = *(const u32x4*)(cr + 2 * h * 512 + 512);
        w[nt][0] = v.x; w[nt][1] = v.y; w[nt][2] = v.z; w[nt][3] = v.w;
        w[nt][4] = u.x; w[nt][5] = u.y; w[nt][6] = u.z; w[nt][7] = u.w;
      }
      kc[nt] = pt_consts<BITS, SYM, ZF>(sh[nt], zh[nt], g.zoff);
    }
    // A operands two steps ahead of their use (an LDS read takes longer than
    // a step's four MFMAs), B operands one: a step's region holds its MFMAs
    // and the next step's decode, interleaved, so that a wave alone on its
    // SIMD keeps the matrix core busy
    f32x16 acc[NM][2];
    f16x8 av[3][NM], bv[2][2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < NM; ++i) av[t][i] = a_op(i, t);
    after_reads();
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) bv[0][nt] = pf_decode<BITS, SYM>(w[nt], kc[nt], 0, dk);
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      if (t + 2 < 8) {
#pragma unroll
        for (int i = 0; i < NM; ++i) av[(t + 2) % 3][i] = a_op(i, t + 2);
      }
      if (t < 7) {
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
          bv[(t + 1) & 1][nt] = pf_decode<BITS, SYM>(w[nt], kc[nt], t + 1, dk);
      }
#pragma unroll
      for (int i = 0; i < NM; ++i)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
          acc[i][nt] = mfma_32x32x16(av[t % 3][i], bv[t & 1][nt], t == 0 ? f32x16{} : acc[i][nt]);
#pragma unroll
      for (int q = 0; q < 2 * NM; ++q) {
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                 // LDS read
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                 // MFMA
        __builtin_amdgcn_sched_group_barrier(0x002, NM == 2 ? 5 : 10, 0);  // vector work
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (ZF) {
      // a fractional zero-point in the wave's rows: acc -= zf c2, c2 the
      // group's sum of x per token
      if (__builtin_amdgcn_ballot_w64(kc[0].zf != 0.f || kc[1].zf != 0.f) != 0) {  // uniform
#pragma unroll
        for (int i = 0; i < NM; ++i) {
          const float* cp = g.c2 + (int64_t)grp * g.c2_ld + p0 + 32 * (i * WM + wm) + 4 * h;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const float4 c2 = *(const float4*)(cp + 8 * q);
#pragma unroll
            for (int nt = 0; nt < 2; ++nt)
              if (kc[nt].zf != 0.f) {  // (c2 may be infinite)
                acc[i][nt][4 * q] -= kc[nt].zf * c2.x;
                acc[i][nt][4 * q + 1] -= kc[nt].zf * c2.y;
                acc[i][nt][4 * q + 2] -= kc[nt].zf * c2.z;
                acc[i][nt][4 * q + 3] -= kc[nt].zf * c2.w;
              }
          }
        }
      }
    }
#pragma unroll
    for (int i = 0; i < NM; ++i)
#pragma unroll
      for (int nt = 0; nt < 2; ++nt)
#pragma unroll
        for (int j = 0; j < 16; ++j) y[i][nt][j] = fmaf(kc[nt].s, acc[i][nt][j], y[i][nt][j]);
    }
  };

  // ---- main loop: U groups an iteration share one load of scales.  One loop
  // per count of token blocks (a branch in the loop costs copies of y) ----
  constexpr int U = SZQ ? 2 : 1;
  uint32_t sz[2];
  auto load_sz = [&](int grp) {
    if constexpr (!SCALED) return;
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      if constexpr (SZQ) sz[nt] = *(const uint32_t*)(szp[nt] + grp);
      else sz[nt] = szp[nt][grp];
    }
    asm volatile("" ::: "memory");  // before the ring's next loads
  };
  load_sz(0);
#pragma unroll
  for (int d = 0; d < D - 1; ++d) issue(min(d, ng - 1), smem + d * SL::BYTES);
  auto loop = [&](auto nm) {
    int in = D - 1, cur = 0;  // ring slots of the next issue and of the group
    for (int c = 0; c < ng; c += U) {
      uint32_t s2[2] = {}, z2[2] = {};  // [block]
      if constexpr (SCALED)
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) {
        // (moved to registers of their own, so that the next load goes to
        // sz's and not through a copy that waits for it at the loop's end)
        uint32_t v;
        asm volatile("v_mov_b32 %0, %1" : "=v"(v) : "v"(sz[nt]));
        pt_halves(v, s2[nt], z2[nt]);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        // this thread's loads of group c + u are in and its reads of the slot
        // before are done, then everyone's: the oldest slot is free
        wait_vmcnt<SL::NI * (D - 2)>();
        wait_lgkm0();
        asm volatile("s_barrier" ::: "memory");
        if (u == 0) load_sz(min(c + U, ng - U));
        unsigned char* const next = smem + in * SL::BYTES;
        const unsigned char* sl = smem + cur * SL::BYTES;
        in = in + 1 == D ? 0 : in + 1;
        cur = cur + 1 == D ? 0 : cur + 1;
        const auto load_next = [&] { issue(min(c + u + D - 1, ng - 1), next); };
        if constexpr (decltype(nm)::value == 0) load_next();
        else {
          __half sh[2], zh[2];
#pragma unroll
          for (int nt = 0; nt < 2; ++nt) {
            sh[nt] = pt_half(s2[nt], u);
            zh[nt] = pt_half(z2[nt], u);
          }
          group(nm, c + u, sl, sh, zh, load_next);  // (the loads after its first LDS reads)
        }
      }
    }
  };
  if (nact == MT) loop(std::integral_constant<int, MT>{});
  else if (MT == 2 && nact == 1) loop(std::integral_constant<int, 1>{});
  else loop(std::integral_constant<int, 0>{});
  wait_vmcnt<0>();  // the tail's loads land before the workgroup's LDS goes away

  if constexpr (BITS == kPtTurbo) {  // the rows' norms
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      const int n = min(pt_row<MODE>(n0, 2 * wn + nt, li), g.N - 1);
      const float nr = g.norms[TWO ? nt : 0][e * g.n_es + n];
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < 16; ++j) y[i][nt][j] *= nr;
    }
  }

  // ---- low-rank term: y += a SV^T (a: token rows, SV: weight rows) ----
  if (g.a != nullptr && g.rank > 0 && g0 == 0) {
    for (int j0 = 0; j0 < g.rank; j0 += 16) {
      const int jk = j0 + 8 * h;
      const bool jv = jk < g.rank;
      f16x8 bv[2];
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) {
        const int n = min(pt_row<MODE>(n0, 2 * wn + nt, li), g.N - 1);
        bv[nt] = jv ? *(const f16x8*)(g.sv[TWO ? nt : 0] + e * g.sv_es + (int64_t)n * g.rank + jk)
                    : f16x8{};
      }
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const __half* ap = g.a + (int64_t)(p0 + min(32 * (i * WM + wm) + li, rows - 1)) * g.a_ld + jk;
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
          f16x8 av = f16x8{};
          if (jv) {
            const __half* am = ap + (TWO ? nt * g.rank : 0);
            av = *(const f16x8*)am;
          }
          y[i][nt] = mfma_32x32x16(av, bv[nt], y[i][nt]);
        }
      }
    }
  }

  // ---- stores: lane holds tokens 8 (j / 4) + 4 h + j % 4 of weight row li ----
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int t0 = 32 * (i * WM + wm) + 4 * h;
    if constexpr (MODE == kPfGateUp) {
      const int n = pt_row<MODE>(n0, 2 * wn, li);
      if (n >= g.N) continue;
      const int col = pt_col(g.out_bits, n);
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const int r = t0 + 8 * (j >> 2) + (j & 3);
        if (r < rows)
          g.y[(int64_t)(p0 + r) * g.y_ld + col] = swiglu_fp16(y[i][0][j], y[i][1][j]);
      }
    } else {
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) {
        const int n = pt_row<MODE>(n0, 2 * wn + nt, li);
        if (n >= g.N) continue;
        const float bn = (MODE == kPfDense && g.bias) ? __half2float(g.bias[n]) : 0.f;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const int r = t0 + 8 * (j >> 2) + (j & 3);
          if (r >= rows) continue;
          if constexpr (MODE == kPfDense)
            g.y[(int64_t)(p0 + r) * g.y_ld + pt_col(g.out_bits, n)] =
                __float2half(y[i][nt][j] + bn);
          else
            g.yf[bz * g.yf_ss + (int64_t)(p0 + r) * g.yf_ld + n] = y[i][nt][j];
        }
      }
    }
  }
}

template <int BITS, int WM, int WN, int MT, int MODE, bool SYM, bool ZF, bool SZQ>
__global__ __launch_bounds__(kPfThreads, 2) void pf_tile_kernel(PfArgs g) {
#ifdef __HIP_DEVICE_COMPILE__  // (the host pass refuses pt_body's device types)
  extern __shared__ __align__(16) unsigned char smem[];
  pt_body<BITS, WM, WN, MT, MODE, SYM, ZF, SZQ>(g, smem, blockIdx.x, blockIdx.y, blockIdx.z);
#endif
}

template <int BITS, int WM, int WN, int MT, int MODE, bool SYM, bool ZF, bool SZQ>
static int pt_launch_k(const PfArgs& g, hipStream_t s) {
  static size_t attr = 64 * 1024;
  using SL = PtSlot<BITS, WM, WN, MT>;
  const size_t lds = (size_t)SL::D * SL::BYTES;
  int rc = set_lds_limit(pf_tile_kernel<BITS, WM, WN, MT, MODE, SYM, ZF, SZQ>, lds, attr);
  if (rc) return rc;
  const dim3 grid((unsigned)g.ntn, (unsigned)g.max_tiles, (unsigned)(MODE == kPfDown ? g.ks : 1));
  pf_tile_kernel<BITS, WM, WN, MT, MODE, SYM, ZF, SZQ><<<grid, dim3(kPfThreads), lds, s>>>(g);
  GLQ_LAUNCH_CHECK("pf_tile_kernel");
  return GLQ_OK;
}

// Two launches of 32-token tiles as one: b's nb workgroups (4-bit, the shared
// expert), then a's (2-bit or TurboQuant, the routed experts).  Their tiles do
// not fill the chip in whole rounds, so b's cost little beside a's: 19.5 + 11.3
// us of the block's 155 at 32 tokens as launches of their own.
template <int BA, int MODE, bool SZQ>
__global__ __launch_bounds__(kPfThreads, 2) void pf_tile_pair_kernel(PfArgs a, PfArgs b, int nb) {
#ifdef __HIP_DEVICE_COMPILE__
  extern __shared__ __align__(16) unsigned char smem[];
  int i = blockIdx.x;
  if (i < nb) {
    const int x = i % b.ntn, r = i / b.ntn;
    pt_body<4, 1, 4, 1, MODE, false, false, SZQ>(b, smem, x, r % b.max_tiles, r / b.max_tiles);
  } else {
    i -= nb;
    const int x = i % a.ntn, r = i / a.ntn;
    pt_body<BA, 1, 4, 1, MODE, false, false, BA == kPtTurbo ? false : SZQ>(
        a, smem, x, r % a.max_tiles, r / a.max_tiles);
  }
#endif
}

template <int BA, int MODE, bool SZQ>
static int pt_launch_pair_k(const PfArgs& a, const PfArgs& b, hipStream_t s) {
  static size_t attr = 64 * 1024;
  using SA = PtSlot<BA, 1, 4, 1>;
  using SB = PtSlot<4, 1, 4, 1>;
  const size_t lds = std::max((size_t)SA::D * SA::BYTES, (size_t)SB::D * SB::BYTES);
  int rc = set_lds_limit(pf_tile_pair_kernel<BA, MODE, SZQ>, lds, attr);
  if (rc) return rc;
  const int64_t nb = (int64_t)b.ntn * b.max_tiles * (MODE == kPfDown ? b.ks : 1);
  const int64_t na = (int64_t)a.ntn * a.max_tiles * (MODE == kPfDown ? a.ks : 1);
  GLQ_CHECK(na + nb < (1ll << 31), "too many workgroups");
  pf_tile_pair_kernel<BA, MODE, SZQ><<<dim3((unsigned)(na + nb)), dim3(kPfThreads), lds, s>>>(
      a, b, (int)nb);
  GLQ_LAUNCH_CHECK("pf_tile_pair_kernel");
  return GLQ_OK;
}

// Scales and zero-points whose rows are whole 4-byte aligned pairs.
static bool pt_pairs(const PfArgs& g, bool sym, int nmat) {
  uintptr_t m = 0;
  for (int i = 0; i < nmat; ++i)
    m |= (uintptr_t)g.scales[i] | (sym ? 0 : (uintptr_t)g.zeros[i]);
  return g.G % 2 == 0 && m % 4 == 0;
}

template <int WM, int WN, int MT, int MODE, bool SYM, bool ZF>
static int pt_launch(const PfArgs& g, int bits, hipStream_t s) {
  // (with the fractional zero-points' branch two groups an iteration would
  // spill registers)
  if constexpr (!ZF)
    if (pt_pairs(g, SYM, MODE == kPfGateUp ? 2 : 1))
      return bits == 2 ? pt_launch_k<2, WM, WN, MT, MODE, SYM, ZF, true>(g, s)
                       : pt_launch_k<4, WM, WN, MT, MODE, SYM, ZF, true>(g, s);
  return bits == 2 ? pt_launch_k<2, WM, WN, MT, MODE, SYM, ZF, false>(g, s)
                   : pt_launch_k<4, WM, WN, MT, MODE, SYM, ZF, false>(g, s);
}

template <int BA, int MODE>
static int pt_launch_pair(const PfArgs& a, const PfArgs& b, hipStream_t s) {
  const int nmat = MODE == kPfGateUp ? 2 : 1;
  if ((BA == kPtTurbo || pt_pairs(a, false, nmat)) && pt_pairs(b, false, nmat))
    return pt_launch_pair_k<BA, MODE, true>(a, b, s);
  return pt_launch_pair_k<BA, MODE, false>(a, b, s);
}
}  // namespace glq
