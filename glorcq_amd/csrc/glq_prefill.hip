// Prefill (many tokens): grouped dequant-to-fp16 MFMA GEMM with the low-rank
// correction, for one projection (glq_gemm_lora; the reference's
// gptq_dequant_gemm_kernel, inference/kernels/gptq_matmul.cu:111-213, taken
// for B > 4, plus the LoRA tail of GLoRCQLinear.forward,
// inference/quantized_linear.py:338-349) and for the routed experts of a MoE
// block over a prompt (glq_moe_prefill; the reference's _forward_sparse,
// inference/moe_block.py:704-740: each active expert's projections on its
// gathered tokens).
//
// The MoE block's projections, and dense ones where it is the faster form
// (pt_dense_tile), run in the tile form of glq_pf_tile.h.
// pf_gemm_kernel<BITS, TM, RT, SYM, ZF, DEEP> takes the other dense ones: a
// workgroup of 4 waves owns TM token rows x (4 * 16 RT) weight rows and a range
// of K.
//  * Per 128-code group one LDS slot receives, by direct global->LDS loads,
//    the TM rows of A (16-byte piece c of slot row r at c ^ (r % 16), so 16
//    lanes reading one piece of 16 rows hit 16 distinct bank groups), each
//    wave's codes, and its rows' scales and zero-points.  A ring of D slots
//    keeps D - 1 groups in flight; each thread waits for its own loads of a
//    group (vmcnt), one barrier makes them everyone's and frees the oldest
//    slot for the next issue.  DEEP rings give half the CU's LDS to one
//    workgroup (for small launches); others take 2 or 3 slots.
//  * A: the caller's x in natural order; each MFMA operand is built in the
//    decode's order with v_perm (pf_nat_a).
//  * B: codes decode into exact fp16 MFMA operands q - zi (zi the
//    zero-point's nearest integer): one v_and_or per code pair lands q under
//    an exponent chosen per bit position (exactly 2^e + q), one packed fp16
//    add removes 2^e + zi.  Each group's fp32 MFMA sum is scaled once,
//    y += s (acc - zf c2), zf = z - zi and c2 the group's sum of x (only for
//    non-integer zero-points: an MFMA of A against ones),
//    so W = s (q - z) enters exactly, as in the reference's fp32 kernel.
//    Lane group kb of a wave holds code words 2kb, 2kb+1 (2-bit) or
//    4kb..4kb+3 (4-bit) of a group; k-step t uses slice t of them.
//  * v_mfma_f32_16x16x32_f16 with A = 16 token rows, B = 16 weight rows: each
//    A operand feeds RT MFMAs and each decoded B operand TM/16.
//  * Split K (ks > 1; no plan takes it by itself, GLQ_PF_KS asks for it): each
//    (tile, split) workgroup writes an fp32 partial tile; the last of a tile's
//    splits to arrive (a per-tile counter, left zero again) sums the partials
//    in split order and runs the epilogue, so the result does not depend on
//    arrival order.
//  * Epilogue: y = fp16(acc + a SV^T + bias).
//
// pf_lowrank_body: a = x U for the low-rank term (fp32 accumulation, one fp16
// rounding), 64 rows per workgroup with U staged transposed in LDS: the MoE
// prompts' launches (pf_lowrank_kernel) and the dense tile form's
// (pf_prep_kernel).
#include <unistd.h>

#include <algorithm>
#include <cstdio>
#include <cstring>

#include "glq_handoff.h"
#include "glq_moe_route.h"
#include "glq_stream.h"

namespace glq {

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

enum PfMode { kPfDense = 0, kPfGateUp = 1, kPfDown = 2 };

constexpr int kPfThreads = 256;  // 4 waves

struct PfArgs {
  const __half* xp;          // A rows, K halves each: in decode order (tile form) or natural
  const int32_t* arow;       // tile form: A row of sorted row p (null: p)
  const uint32_t* codes[2];  // matrix m: (E, N, kw) words
  const __half* scales[2];   // (E, N, G)
  const __half* zeros[2];    // (E, N, G) (unused with SYM)
  int64_t codes_es, sz_es;   // expert strides (elements)
  const float* norms[2];     // TurboQuant codes: (E, N) row norms,
  int64_t n_es;
  const float* cent[2];      // and the 4-entry codebook
  const __half* a;           // low-rank a (rows, a_ld) fp16: matrix m at column m*rank, or null
  int a_ld;
  const __half* sv[2];       // (E, N, rank)
  int64_t sv_es;
  const __half* bias;        // (N,) or null (dense)
  __half* y;                 // DENSE: (M, N); GATE/UP: inter (rows, N) in decode order
  int64_t y_ld;
  float* yf;                 // DOWN: (rows, N) fp32
  int64_t yf_ld, yf_ss;      // and elements between its K splits (tile form)
  const float* c2;           // tile form, ZF: per (group, row) sum of x, (G, c2_ld) fp32
  int64_t c2_ld;
  float* part;               // pf_gemm_kernel: split-K partial tiles (ks, tiles, TM, ntn*WGR) fp32
  unsigned* cnt;             // split-K arrival counters (tiles * ntn), zero between launches
  const int32_t* tiles;      // tile form: (max_tiles, 3): expert, first sorted row, rows; null: dense
  const int32_t* ntiles;     // device count of valid tiles
  int M, K, N, G, kw, rank;
  int ntn;                   // weight-row tiles of a workgroup along N
  int ks, gps;               // K splits, groups per split
  int out_bits;              // tile form: decode order of y's consumer (2, 4, or 0: natural)
  int max_tiles;             // token tiles in the grid (y dimension)
  float zoff;                // added to every zero-point (signed codes stored offset by 2^(b-1))
  // a = x U formed in the same launch (dense form, no K split; pf_xu_job):
  // row-block jobs fill the first xu_rows rows of the grid, and the epilogue
  // waits for its token rows' blocks (a read coherently).  xu_rows == 0: a
  // is given (or absent).
  int xu_rows, xu_nrb, xu_ns, xu_rpad;
  const __half* xu_u;        // U (K, rank)
  float* xu_part;            // (nrb, ns, 16, rpad) fp32 slice partials
  unsigned* xu_cnt;          // (nrb) words: arrivals | ready bit | readers << 16; zero between launches
  uint64_t xu_spin;          // the epilogue's wait bound (100 MHz real-time counter ticks)
};

// The x U jobs of the fused dense launch (see PfArgs).  A row block's word:
// low bits the slices that arrived, kXuReady once its last slice has
// written a, then 1 << 16 per GEMM workgroup that has read it; whichever
// event completes the final word sets it back to zero.
constexpr unsigned kXuReady = 0x8000u;
constexpr size_t kXuJobLds = (4 * 4 * 64) * 4 + 16 * kLowrankRows * 2 +
                             64 * kLowrankUtStride * 2 + 16 * 128 * 4;

__device__ __forceinline__ unsigned pf_xu_final(const PfArgs& g) {
  return ((unsigned)g.ntn << 16) | kXuReady | (unsigned)g.xu_ns;
}

// Job (row block rb, K slice sp): lowrank_partial<4> over the slice, handed
// over; the block's last slice sums the slices in slice order and writes
// a = fp16 (agent-scope stores), then marks the block ready.
__device__ void pf_xu_job(const PfArgs& g, int job, unsigned char* smem, int* flag) {
  const int rb = job / g.xu_ns, sp = job - rb * g.xu_ns, tid = threadIdx.x;
  const int r0 = 16 * rb, rows = min(16, g.M - r0), rank = g.rank, rpad = g.xu_rpad;
  float* red = (float*)smem;
  __half* xl = (__half*)(red + 4 * 4 * 64);
  __half* ut = xl + 16 * kLowrankRows;
  const __half* xb = g.xp + (int64_t)r0 * g.K;
  auto xrow = [&](int m) { return xb + (int64_t)m * g.K; };
  float* slices = g.xu_part + (int64_t)rb * g.xu_ns * 16 * rpad;
  lowrank_partial<4, decltype(xrow), true>(xrow, rows, g.K, rank, rpad, g.xu_u, sp,
                                           slices + (int64_t)sp * 16 * rpad, red, xl, tid, ut);
  if (!handoff_arrive(g.xu_cnt + rb, (unsigned)g.xu_ns, flag)) return;
  for (int i = tid; i < rows * rank; i += kPfThreads) {
    const int m = i / rank, j = i - m * rank;
    const __half v = __float2half(sum_strided_coh(slices + m * rpad + j, 16 * rpad, g.xu_ns));
    handoff_put((uint16_t*)g.a + (int64_t)(r0 + m) * g.a_ld + j, __half_as_ushort(v));
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid == 0) {
    const unsigned old = __hip_atomic_fetch_add(g.xu_cnt + rb, kXuReady, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_AGENT);
    if (old + kXuReady == pf_xu_final(g)) handoff_reset(g.xu_cnt + rb);
  }
}

// The epilogue's wait for the row blocks of token rows [p0, p0 + rows): a
// block not ready within xu_spin is formed here, slice by slice in the
// jobs' order (the same bits), and written as the jobs write it.  Every
// thread calls it; smem is free (the ring has drained).
__device__ void pf_xu_wait(const PfArgs& g, int p0, int rows, unsigned char* smem, int* flag) {
  const int rb0 = p0 / 16, rb1 = (p0 + rows - 1) / 16, tid = threadIdx.x;
  if (tid == 0) {
    int missing = 0;
    for (int rb = rb0; rb <= rb1; ++rb) {
      const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
      while (!(handoff_get(g.xu_cnt + rb) & kXuReady)) {
        if (__builtin_amdgcn_s_memrealtime() - t0 > g.xu_spin) {
          missing |= 1 << (rb - rb0);
          break;
        }
        __builtin_amdgcn_s_sleep(2);
      }
    }
    *flag = missing;
  }
  __syncthreads();
  const int missing = *flag;
  __syncthreads();
  for (int rb = rb0; rb <= rb1; ++rb) {
    if (!(missing & (1 << (rb - rb0)))) continue;  // uniform
    const int r0 = 16 * rb, brows = min(16, g.M - r0), rank = g.rank, rpad = g.xu_rpad;
    float* red = (float*)smem;
    __half* xl = (__half*)(red + 4 * 4 * 64);
    __half* ut = xl + 16 * kLowrankRows;
    float* out = (float*)(ut + 64 * kLowrankUtStride);  // 16 x rpad
    const __half* xb = g.xp + (int64_t)r0 * g.K;
    auto xrow = [&](int m) { return xb + (int64_t)m * g.K; };
    float acc[4] = {0.f, 0.f, 0.f, 0.f};  // elements tid + 256 q of the block
    for (int sp = 0; sp < g.xu_ns; ++sp) {
      lowrank_partial<4>(xrow, brows, g.K, rank, rpad, g.xu_u, sp, out, red, xl, tid, ut);
      __syncthreads();
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int i = tid + kPfThreads * q, m = i / rpad, j = i - m * rpad;
        if (m < brows && j < rank) acc[q] += out[m * rpad + j];
      }
      __syncthreads();
    }
    const int pad = (8 - g.xu_ns % 8) % 8;  // sum_strided's zeros after the last batch
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      for (int z = 0; z < pad; ++z) acc[q] += 0.f;
      const int i = tid + kPfThreads * q, m = i / rpad, j = i - m * rpad;
      if (m < brows && j < rank)
        handoff_put((uint16_t*)g.a + (int64_t)(r0 + m) * g.a_ld + j,
                    __half_as_ushort(__float2half(acc[q])));
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  }
}

// 8 halves of a written inside this launch (agent-scope loads).
__device__ __forceinline__ f16x8 pf_load8_coh(const __half* p) {
  const unsigned long long lo = handoff_get((const unsigned long long*)p);
  const unsigned long long hi = handoff_get((const unsigned long long*)p + 1);
  return __builtin_bit_cast(f16x8, u32x4{(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi,
                                         (uint32_t)(hi >> 32)});
}

// Position of natural column c inside its 16-code block in decode order
// (inverse of perm_src).
template <int BITS>
__device__ __forceinline__ int perm_pos(int c) {
  if constexpr (BITS == 2) return c < 8 ? 2 * c : 2 * (c - 8) + 1;
  else {
    const int h = c & 8, q = c & 7;
    return h + (q < 4 ? 2 * q : 2 * (q - 4) + 1);
  }
}
__device__ __forceinline__ int perm_pos_rt(int bits, int c) {
  return bits == 2 ? perm_pos<2>(c) : perm_pos<4>(c);
}

// Per (row tile, group): packed constants -(2^e + zi) for the exponent biases
// of the decode (2-bit: 1024, 256, 64, 16, 4; 4-bit: 1024, 64), the scale, and
// the fractional part zf = z - zi of the zero-point (zi = the nearest integer).
template <int BITS>
struct PfK {
  f16x2 c[BITS == 2 ? 5 : 2];
  float s, zf;
};

template <int BITS, bool SYM>
__device__ __forceinline__ PfK<BITS> pf_consts(__half sh, __half zh, float zoff) {
  PfK<BITS> k;
  const float z = SYM ? (float)(1 << (BITS - 1)) : __half2float(zh) + zoff;
  const float zi = rintf(z);
  k.zf = z - zi;
  k.s = __half2float(sh);
  constexpr float b2[5] = {1024.f, 256.f, 64.f, 16.f, 4.f};
  constexpr float b4[2] = {1024.f, 64.f};
#pragma unroll
  for (int i = 0; i < (BITS == 2 ? 5 : 2); ++i) {
    const _Float16 v = (_Float16)(-((BITS == 2 ? b2[i] : b4[i]) + zi));  // exact integer
    k.c[i] = f16x2{v, v};
  }
  return k;
}

__device__ __forceinline__ uint32_t pf_sub(uint32_t h, f16x2 c) {
  return __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, h) + c);  // exact
}

// B operand of k-step t (0..3) of a group: q - zi as fp16 (exact small integers).
template <int BITS, bool SYM>
__device__ __forceinline__ f16x8 pf_decode(const uint32_t* w, const PfK<BITS>& k, int t,
                                           const DecodeConsts& dk) {
  constexpr uint32_t xm = SYM ? (BITS == 2 ? 0xAAAAAAAAu : 0x88888888u) : 0u;
  u32x4 o;
  if constexpr (BITS == 2) {
    const uint32_t wd = w[t >> 1] ^ xm;
    if ((t & 1) == 0) {
      o.x = pf_sub((wd & 0x00030003u) | dk.e25, k.c[0]);
      o.y = pf_sub((wd & 0x000C000Cu) | dk.e23, k.c[1]);
      o.z = pf_sub((wd & 0x00300030u) | dk.e21, k.c[2]);
      o.w = pf_sub((wd & 0x00C000C0u) | dk.e19, k.c[3]);
    } else {
      const uint32_t v = wd >> 10;
      o.x = pf_sub((wd & 0x03000300u) | dk.e17, k.c[4]);
      o.y = pf_sub((v & 0x00030003u) | dk.e25, k.c[0]);
      o.z = pf_sub((v & 0x000C000Cu) | dk.e23, k.c[1]);
      o.w = pf_sub((v & 0x00300030u) | dk.e21, k.c[2]);
    }
  } else {
    const uint32_t wd = w[t] ^ xm, v = wd >> 8;
    o.x = pf_sub((wd & 0x000F000Fu) | dk.e25, k.c[0]);
    o.y = pf_sub((wd & 0x00F000F0u) | dk.e21, k.c[1]);
    o.z = pf_sub((v & 0x000F000Fu) | dk.e25, k.c[0]);
    o.w = pf_sub((v & 0x00F000F0u) | dk.e21, k.c[1]);
  }
  return __builtin_bit_cast(f16x8, o);
}

// A operand of k-step t (0..3) from an LDS row holding x in NATURAL order
// (16-byte piece P at position P ^ li): the decode's order is made with
// v_perm.  2-bit step t pairs codes (j, j + 8) of word 2kb + t / 2, i.e.
// halves j of natural pieces 4kb + 2 (t / 2) and + 1 (j = 0..3 for even t,
// 4..7 for odd); 4-bit step t pairs codes (j, j + 4) of word 4kb + t, halves
// j and j + 4 of natural piece 4kb + t.
template <int BITS>
__device__ __forceinline__ f16x8 pf_nat_a(const unsigned char* row, int kb, int t, int li) {
  u32x4 o;
  if constexpr (BITS == 2) {
    const int p0 = 4 * kb + 2 * (t >> 1);
    const u32x4 lo = *(const u32x4*)(row + ((p0 ^ li) << 4));
    const u32x4 hi = *(const u32x4*)(row + (((p0 + 1) ^ li) << 4));
    const uint32_t a0 = (t & 1) ? lo.z : lo.x, a1 = (t & 1) ? lo.w : lo.y;
    const uint32_t b0 = (t & 1) ? hi.z : hi.x, b1 = (t & 1) ? hi.w : hi.y;
    o.x = __builtin_amdgcn_perm(b0, a0, 0x05040100u);
    o.y = __builtin_amdgcn_perm(b0, a0, 0x07060302u);
    o.z = __builtin_amdgcn_perm(b1, a1, 0x05040100u);
    o.w = __builtin_amdgcn_perm(b1, a1, 0x07060302u);
  } else {
    const u32x4 v = *(const u32x4*)(row + (((4 * kb + t) ^ li) << 4));
    o.x = __builtin_amdgcn_perm(v.z, v.x, 0x05040100u);
    o.y = __builtin_amdgcn_perm(v.z, v.x, 0x07060302u);
    o.z = __builtin_amdgcn_perm(v.w, v.y, 0x05040100u);
    o.w = __builtin_amdgcn_perm(v.w, v.y, 0x07060302u);
  }
  return __builtin_bit_cast(f16x8, o);
}

// Weight row of row tile rt of a wave (see the file comment); may be >= N
// (clamp for loads).
template <int RT>
__device__ __forceinline__ int pf_row(int n0, int wave, int rt, int li) {
  return n0 + wave * (16 * RT) + rt * 16 + li;
}

// LDS slot of one group: A (TM token rows x 256 B, swizzled pieces), then per
// wave its RT row tiles' codes (16 rows x CB bytes each, padded to whole
// 1 KB load instructions), scales and zero-points (one fp16 per (row tile,
// row) at a 4-byte stride, as the 2-byte direct-to-LDS load places them).
// Ring depth D: DEEP rings take half the CU's 160 KB (two workgroups per
// CU, as many groups in flight as fit); otherwise 3 slots when two
// workgroups fit a CU, else 2.
template <int BITS, int TM, int RT, bool DEEP = false>
struct PfSlot {
  static constexpr int CB = BITS == 2 ? 32 : 64;        // code bytes per row per group
  static constexpr int CW = RT * 16 * CB;                // code bytes per wave
  static constexpr int CR = CW < 1024 ? 1024 : CW;       // LDS bytes per wave (whole loads)
  static constexpr int A = 0;
  static constexpr int C = TM * 256;
  static constexpr int S = C + 4 * CR;
  static constexpr int Z = S + 4 * 256;
  static constexpr int BYTES = Z + 4 * 256;
  static constexpr int NC = CR / 1024;                   // code load instructions per wave
  static constexpr int NI = TM / 16 + NC + 2;            // loads per lane per group (max)
  static constexpr int DMAX = 2 + 63 / NI;               // the vmcnt field is 6 bits
  static constexpr int DFIT = (80 * 1024 - 64) / BYTES;  // two workgroups per CU
  static constexpr int D = DEEP ? (DFIT < DMAX ? (DFIT < 16 ? DFIT : 16) : (DMAX < 16 ? DMAX : 16))
                                : (2 * 3 * BYTES <= 160 * 1024 ? 3 : 2);
};

template <int BITS, int TM, int RT, bool SYM, bool ZF, bool DEEP>
__global__ __launch_bounds__(kPfThreads, 2) void pf_gemm_kernel(PfArgs g) {
  extern __shared__ __align__(16) unsigned char smem[];
  using SL = PfSlot<BITS, TM, RT, DEEP>;
  constexpr int TT = TM / 16;
  constexpr int XI = TM / 16;  // A load instructions per wave per group (4 rows each)
  constexpr int WGR = 4 * 16 * RT;
  constexpr int D = SL::D;
  constexpr int NI = XI + SL::NC + 1 + (SYM ? 0 : 1);  // loads per lane per group
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, kb = lane >> 4;
  __shared__ int xflag;
  if (g.xu_rows && (int)blockIdx.y < g.xu_rows) {  // an x U job (uniform)
    const int job = blockIdx.y * gridDim.x + blockIdx.x;
    if (job < g.xu_nrb * g.xu_ns) pf_xu_job(g, job, smem, &xflag);
    return;
  }
  const int ty = blockIdx.y - g.xu_rows;
  const int p0 = ty * TM, rows = min(TM, g.M - p0);
  const int tn = blockIdx.x % g.ntn, sp = blockIdx.x / g.ntn;
  const int n0 = tn * WGR;
  const int g0 = sp * g.gps, g1 = min(g0 + g.gps, g.G);

  // ---- per-lane load addresses: offsets in elements from uniform bases (the
  // workgroup's first weight row: weights of 4 GB and more come here) ----
  // A: this lane's XI slot rows
  int aoff[XI];
#pragma unroll
  for (int q = 0; q < XI; ++q) {
    const int r = (wave * XI + q) * 4 + (lane >> 4);
    aoff[q] = (p0 + min(r, rows - 1)) * g.K + (((lane & 15) ^ (r & 15)) << 3);
  }
  const uint32_t* cb = g.codes[0] + (int64_t)n0 * g.kw;
  const __half* sb = g.scales[0] + (int64_t)n0 * g.G;
  const __half* zb = SYM ? sb : g.zeros[0] + (int64_t)n0 * g.G;
  // codes: instruction q covers bytes q*1024 + 16*lane of the wave's region
  // (lanes past the wave's code bytes re-load its first ones into the padding)
  int coff[SL::NC];
#pragma unroll
  for (int q = 0; q < SL::NC; ++q) {
    const int o = (q * 1024 + 16 * lane) % SL::CW;
    const int rt = o / (16 * SL::CB), row = (o % (16 * SL::CB)) / SL::CB;
    const int piece = (o % SL::CB) / 16;
    const int n = min(pf_row<RT>(n0, wave, rt, row), g.N - 1);
    coff[q] = (n - n0) * g.kw + 4 * piece;
  }
  // scales / zero-points: lane -> (row tile lane/16, row lane%16)
  const int soff =
      (min(pf_row<RT>(n0, wave, min(lane >> 4, RT - 1), lane & 15), g.N - 1) - n0) * g.G;
  auto issue = [&](int grp, unsigned char* slot) {
#pragma unroll
    for (int q = 0; q < XI; ++q)
      __builtin_amdgcn_global_load_lds((const void*)(g.xp + aoff[q] + grp * 128),
                                       (lds_void*)(slot + SL::A + (wave * XI + q) * 1024), 16, 0, 0);
#pragma unroll
    for (int q = 0; q < SL::NC; ++q)
      __builtin_amdgcn_global_load_lds((const void*)(cb + coff[q] + grp * (SL::CB / 4)),
                                       (lds_void*)(slot + SL::C + wave * SL::CR + q * 1024),
                                       16, 0, 0);
    __builtin_amdgcn_global_load_lds((const void*)(sb + soff + grp),
                                     (lds_void*)(slot + SL::S + wave * 256), 2, 0, 0);
    if constexpr (!SYM)
      __builtin_amdgcn_global_load_lds((const void*)(zb + soff + grp),
                                       (lds_void*)(slot + SL::Z + wave * 256), 2, 0, 0);
  };

  f32x4 y[TT][RT];
#pragma unroll
  for (int i = 0; i < TT; ++i)
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) y[i][rt] = f32x4{0.f, 0.f, 0.f, 0.f};
  const DecodeConsts dk = DecodeConsts::make();
  const int ng = g1 - g0;
  // every group issues the same loads (past the split's end they re-read its
  // last group into a slot never consumed), so the explicit waits count exactly
#pragma unroll
  for (int d = 0; d < D - 1; ++d) issue(g0 + min(d, ng - 1), smem + d * SL::BYTES);
  for (int it = 0; it < ng; ++it) {
    const int grp = g0 + it;
    wait_vmcnt<NI * (D - 2)>();               // this thread's loads of grp are in
    asm volatile("s_barrier" ::: "memory");   // everyone's are; the slot of grp - 1 is free
    issue(g0 + min(it + D - 1, ng - 1), smem + ((it + D - 1) % D) * SL::BYTES);
    const unsigned char* sl = smem + (it % D) * SL::BYTES;
    // this lane's codes, scale and zero-point per row tile
    uint32_t w[RT][BITS == 2 ? 2 : 4];
    PfK<BITS> kc[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const unsigned char* cr = sl + SL::C + wave * SL::CR + (rt * 16 + li) * SL::CB;
      if constexpr (BITS == 2) {
        const u32x2 v = *(const u32x2*)(cr + 8 * kb);
        w[rt][0] = v.x;
        w[rt][1] = v.y;
      } else {
        const u32x4 v = *(const u32x4*)(cr + 16 * kb);
        w[rt][0] = v.x;
        w[rt][1] = v.y;
        w[rt][2] = v.z;
        w[rt][3] = v.w;
      }
      const __half sh = *(const __half*)(sl + SL::S + wave * 256 + (rt * 16 + li) * 4);
      const __half zh = SYM ? sh : *(const __half*)(sl + SL::Z + wave * 256 + (rt * 16 + li) * 4);
      kc[rt] = pf_consts<BITS, SYM>(sh, zh, g.zoff);
    }
    // the group's sum of x (q - zi), fp32
    auto a_op = [&](int i, int t) {
      return pf_nat_a<BITS>(sl + SL::A + (16 * i + li) * 256, kb, t, li);
    };
    f32x4 acc[TT][RT];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      f16x8 bf[RT];
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) bf[rt] = pf_decode<BITS, SYM>(w[rt], kc[rt], t, dk);
#pragma unroll
      for (int i = 0; i < TT; ++i) {
        const f16x8 av = a_op(i, t);
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
          acc[i][rt] = mfma_16x16x32(av, bf[rt], t == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[i][rt]);
      }
    }
    // y += s (acc - zf c2): c2 = the group's sum of x per token, needed only
    // for non-integer zero-points (zf != 0): an MFMA against ones when any row
    // of the wave has one
    f32x4 c2v[TT];
    if constexpr (ZF) {
      bool any = false;
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) any |= kc[rt].zf != 0.f;
      if (__builtin_amdgcn_ballot_w64(any) != 0) {  // uniform over the wave
        const f16x8 ones = __builtin_bit_cast(f16x8, u32x4{0x3C003C00u, 0x3C003C00u, 0x3C003C00u,
                                                           0x3C003C00u});
#pragma unroll
        for (int i = 0; i < TT; ++i) {
          c2v[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int t = 0; t < 4; ++t) c2v[i] = mfma_16x16x32(a_op(i, t), ones, c2v[i]);
        }
      }
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const float s = kc[rt].s;
      if (ZF && kc[rt].zf != 0.f) {
        const float zf = kc[rt].zf;
#pragma unroll
        for (int i = 0; i < TT; ++i) {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            y[i][rt][j] = fmaf(s, acc[i][rt][j] - zf * c2v[i][j], y[i][rt][j]);
        }
      } else {
#pragma unroll
        for (int i = 0; i < TT; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) y[i][rt][j] = fmaf(s, acc[i][rt][j], y[i][rt][j]);
      }
    }
  }
  wait_vmcnt<0>();  // the tail's loads land before the workgroup's LDS goes away

  // ---- split K: partial tiles, the last split of a tile reduces ----
  if (g.ks > 1) {
    // partial tile columns: (tn, wave, rt, li), 64 RT per workgroup
    const int ncol = g.ntn * 64 * RT;
    const int cbase = tn * 64 * RT + wave * 16 * RT + li;
    float* mine = g.part + (((int64_t)sp * g.max_tiles + ty) * TM) * ncol;
#pragma unroll
    for (int i = 0; i < TT; ++i)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        const int c = cbase + rt * 16;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          handoff_put(mine + (int64_t)(16 * i + 4 * kb + j) * ncol + c, y[i][rt][j]);
      }
    // arrival (glq_handoff.h); the last split reduces and leaves the counter
    // at zero for the next launch
    __shared__ int last;
    unsigned* cnt = g.cnt + (int64_t)ty * g.ntn + tn;
    if (!handoff_arrive(cnt, (unsigned)g.ks, &last)) return;
    if (tid == 0) handoff_reset(cnt);
#pragma unroll
    for (int i = 0; i < TT; ++i)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) y[i][rt] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < g.ks; ++s) {
      const float* ps = g.part + (((int64_t)s * g.max_tiles + ty) * TM) * ncol;
#pragma unroll
      for (int i = 0; i < TT; ++i)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
          const int c = cbase + rt * 16;
#pragma unroll
          for (int j = 0; j < 4; ++j)
            y[i][rt][j] += handoff_get(ps + (int64_t)(16 * i + 4 * kb + j) * ncol + c);
        }
    }
  }

  // ---- low-rank term: y += a SV^T (a: token rows, SV: weight rows) ----
  if (g.xu_rows && g.rank > 0) pf_xu_wait(g, p0, rows, smem, &xflag);
  if (g.a != nullptr && g.rank > 0) {
    for (int j0 = 0; j0 < g.rank; j0 += 32) {
      const int jk = j0 + 8 * kb;
      const bool jv = jk < g.rank;
      f16x8 bv[RT];
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        const int n = min(pf_row<RT>(n0, wave, rt, li), g.N - 1);
        bv[rt] = jv ? *(const f16x8*)(g.sv[0] + (int64_t)n * g.rank + jk) : f16x8{};
      }
#pragma unroll
      for (int i = 0; i < TT; ++i) {
        const int p = p0 + min(16 * i + li, rows - 1);
        f16x8 av = f16x8{};
        if (jv) {
          const __half* ap = g.a + (int64_t)p * g.a_ld + jk;
          av = g.xu_rows ? pf_load8_coh(ap) : *(const f16x8*)ap;
        }
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) y[i][rt] = mfma_16x16x32(av, bv[rt], y[i][rt]);
      }
    }
  }

  // ---- stores: lane holds tokens 16i + 4kb + j of weight row li ----
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const int n = pf_row<RT>(n0, wave, rt, li);
    if (n >= g.N) continue;
    const float bn = g.bias ? __half2float(g.bias[n]) : 0.f;
#pragma unroll
    for (int i = 0; i < TT; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int r = 16 * i + 4 * kb + j;
        if (r < rows) g.y[(int64_t)(p0 + r) * g.y_ld + n] = __float2half(y[i][rt][j] + bn);
      }
  }
  if (g.xu_rows && g.rank > 0) {  // the workgroup has read a of its rows' blocks
    __syncthreads();
    if (tid == 0)
      for (int rb = p0 / 16; rb <= (p0 + rows - 1) / 16; ++rb) {
        const unsigned old = __hip_atomic_fetch_add(g.xu_cnt + rb, 1u << 16, __ATOMIC_RELAXED,
                                                    __HIP_MEMORY_SCOPE_AGENT);
        if (old + (1u << 16) == pf_xu_final(g)) handoff_reset(g.xu_cnt + rb);
      }
  }
}

}  // namespace glq

#include "glq_pf_tile.h"

namespace glq {

// 16 halves of a code block in the decode order of bits (perm_src): pairs
// (c, c + 8) at 2 bits, (c, c + 4) of each 8 at 4.
__device__ __forceinline__ void pf_permute16(int bits, u32x4 lo, u32x4 hi, u32x4& o0, u32x4& o1) {
  const uint32_t l[4] = {lo.x, lo.y, lo.z, lo.w}, g[4] = {hi.x, hi.y, hi.z, hi.w};
  uint32_t o[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const uint32_t sel = i & 1 ? 0x07060302u : 0x05040100u;
    if (bits == 2) o[i] = __builtin_amdgcn_perm(g[i >> 1], l[i >> 1], sel);
    else o[i] = i < 4 ? __builtin_amdgcn_perm(l[2 + (i >> 1)], l[i >> 1], sel)
                      : __builtin_amdgcn_perm(g[2 + ((i - 4) >> 1)], g[(i - 4) >> 1], sel);
  }
  o0 = u32x4{o[0], o[1], o[2], o[3]};
  o1 = u32x4{o[4], o[5], o[6], o[7]};
}

// ---------------------------------------------------------------------------
// Low-rank a = x U over a tile list (one expert's rows a tile) or all rows.
// Workgroup (64-row block, K slice, block of four 32-column tiles of the
// matrices' a): per 128 codes, the rows of x come to LDS by buffer loads (two
// slots, 16-byte piece c of row r at c ^ (r % 16)) and U's rows through
// registers (the next chunk's are loaded while this one's are multiplied),
// written transposed and in A's code order as pairs (two rows' halves of a
// column in one word), so both MFMA operands are one 16-byte LDS read.  Row
// col of the transposed U is 16 pieces of 8 codes, piece c at c ^ pf_ut_sw(col):
// the reads' 16 columns and the writes' 8 columns x 8 pairs fall on distinct
// banks.  The four waves take the column tiles, and the block's two 32-row
// halves where there are fewer.
//
// A 16-row block with U in its natural layout (two-byte LDS reads of every B
// operand, U read again for every 16 rows) took 100 us a launch for 12000
// rows x (2048 -> 2 x 64) and 43 us for 1024 rows x (4096 -> 2 x 64).
// ---------------------------------------------------------------------------
struct PfLowrank {
  const __half* x;         // A rows, K halves each
  const int32_t* arow;     // A row of sorted row p (null: p)
  int aperm;               // 0: A natural; 2 or 4: A in that decode order
  const __half* U[2];      // (C, K, rank) per matrix
  int64_t u_cs;            // elements between clusters
  const int32_t* cluster[2];  // (E,) cluster of expert e per matrix (null: 0)
  const int32_t* uslot[2];    // cluster -> row of U[m] (a cross-layer pool), or null
  int ncl[2], urows[2];       // clusters of matrix m, rows of U[m]: ids are clamped (0: not)
  const int32_t* tiles;    // tile list of the GEMM (null: dense)
  const int32_t* ntiles;
  int tile_rows;           // rows per tile of the list
  int nmat, rows_total, K, rank, ks, kps;
  float* part;             // (ks, rows_total, nmat * rank) fp32 partial sums of a (ks > 1)
  __half* a_out;           // (rows_total, nmat * rank) a = fp16(x U) (ks == 1, or finalized)
  unsigned* zero_cnt;      // counters the following GEMM launch expects zero, or null
  int n_cnt;
  // arrival counters (row block x column block), zero before and after: the
  // splits' partials are summed by the last to arrive (null: by a launch)
  unsigned* cnt;
};

constexpr int kLrRows = 64;  // rows per low-rank workgroup
constexpr int kLrLds = 128 * 256 + 2 * kLrRows * 256;

__device__ __forceinline__ int pf_ut_sw(int col) { return (col ^ (col >> 3)) & 15; }

__device__ __forceinline__ void pf_lowrank_body(const PfLowrank& L, int job, int sp, int cb,
                                               unsigned char* smem) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 31, h = lane >> 5;
  int e = 0, p0, rows;
  if (L.tiles) {
    const int sub = (L.tile_rows + kLrRows - 1) / kLrRows;  // row blocks per tile
    const int ti = job / sub, part = job % sub;
    if (ti >= *L.ntiles) return;  // uniform over the workgroup
    e = L.tiles[3 * ti];
    p0 = L.tiles[3 * ti + 1] + part * kLrRows;
    rows = min(kLrRows, L.tiles[3 * ti + 2] - part * kLrRows);
  } else {
    p0 = job * kLrRows;
    rows = min(kLrRows, L.rows_total - p0);
  }
  if (rows <= 0) return;
  const int k0 = sp * L.kps, k1 = min(L.K, k0 + L.kps);
  const int r = L.rank, ctm = (r + 31) / 32;        // column tiles per matrix
  const int nct = min(4, L.nmat * ctm - 4 * cb);    // this block's
  const int wct = nct <= 2 ? nct : 4, ct = wave % wct, mg = wave / wct, mw = 4 / wct;
  unsigned char* ut = smem;
  unsigned char* as = smem + 128 * 256;
  const __half* U[2];
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    int c = (m < L.nmat && L.cluster[m]) ? L.cluster[m][e] : 0;
    if (L.ncl[m] > 0) c = min(max(c, 0), L.ncl[m] - 1);
    if (m < L.nmat && L.uslot[m]) c = L.uslot[m][c];
    if (L.urows[m] > 0) c = min(max(c, 0), L.urows[m] - 1);
    U[m] = m < L.nmat ? L.U[m] + (int64_t)c * L.u_cs : nullptr;
  }
  // A: instruction q of the wave loads rows 4 (4 wave + q) .. + 3
  unsigned aoff[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int ar = (4 * wave + q) * 4 + (lane >> 4);
    const int p = p0 + min(ar, rows - 1);
    const unsigned src = L.arow ? L.arow[p] : p;
    aoff[q] = 2u * (src * (unsigned)L.K + 8 * ((lane & 15) ^ (ar & 15)));
  }
  const auto ars = pt_rsrc(L.x);
  auto issue_a = [&](int kc, unsigned char* slot) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ars, (lds_void*)(slot + (4 * wave + q) * 1024), 16,
                                               aoff[q], kc * 2, 0, 0);
  };
  // U: item q of the thread is the pair of rows at A positions (2 pk, 2 pk + 1)
  // of the chunk x 8 columns
  const __half* us[4];
  int dk[4], wpos[4], wcol[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int idx = tid + kPfThreads * q;
    const int c8 = (idx & 7) + 8 * (idx >> 9), pk = (idx >> 3) & 63;
    const int gt = 4 * cb + (c8 >> 2);
    const int m = gt >= ctm ? 1 : 0, j0 = (gt - m * ctm) * 32 + (c8 & 3) * 8;
    int k;  // natural code of position 2 pk; position 2 pk + 1 is dk further
    if (L.aperm == 2) { k = 16 * (pk >> 3) + (pk & 7); dk[q] = 8; }
    else if (L.aperm == 4) { k = 8 * (pk >> 2) + (pk & 3); dk[q] = 4; }
    else { k = 2 * pk; dk[q] = 1; }
    us[q] = c8 < 4 * nct && j0 < r ? (m ? U[1] : U[0]) + (int64_t)k * r + j0 : nullptr;
    wcol[q] = c8 < 4 * nct ? 8 * c8 : -1;
    wpos[q] = pk;
  }
  u32x4 ua[4], ub[4];
  auto load_u = [&](int kc) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      ua[q] = ub[q] = u32x4{0u, 0u, 0u, 0u};
      if (us[q]) {
        ua[q] = *(const u32x4*)(us[q] + (int64_t)kc * r);
        ub[q] = *(const u32x4*)(us[q] + (int64_t)(kc + dk[q]) * r);
      }
    }
  };
  f32x16 acc[2] = {};
  issue_a(k0, as);
  load_u(k0);
  int s = 0;
  for (int kc = k0; kc < k1; kc += 128) {
    __syncthreads();  // the chunk before has been read
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (wcol[q] < 0) continue;
      const uint32_t a[4] = {ua[q].x, ua[q].y, ua[q].z, ua[q].w};
      const uint32_t b[4] = {ub[q].x, ub[q].y, ub[q].z, ub[q].w};
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const int col = wcol[q] + c;
        const uint32_t v = __builtin_amdgcn_perm(b[c >> 1], a[c >> 1],
                                                 c & 1 ? 0x07060302u : 0x05040100u);
        *(uint32_t*)(ut + col * 256 + (((wpos[q] >> 2) ^ pf_ut_sw(col)) << 4) +
                     4 * (wpos[q] & 3)) = v;
      }
    }
    wait_vmcnt<0>();  // this chunk's A
    __syncthreads();
    if (kc + 128 < k1) {  // uniform
      issue_a(kc + 128, as + (s ^ 1) * kLrRows * 256);
      load_u(kc + 128);
    }
    const unsigned char* sl = as + s * kLrRows * 256;
    const int col = ct * 32 + li;
    if (ct < nct) {  // uniform over the wave
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        const f16x8 bv = *(const f16x8*)(ut + col * 256 + (((8 * h + t) ^ pf_ut_sw(col)) << 4));
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int mb = mg + i * mw;  // 32-row half
          if (mb < 2) {                // uniform over the wave
            const int row = 32 * mb + li;
            const f16x8 av = *(const f16x8*)(sl + row * 256 + (((8 * h + t) ^ (row & 15)) << 4));
            acc[i] = mfma_32x32x16(av, bv, acc[i]);
          }
        }
      }
    }
    s ^= 1;
  }
  // acc[i][q]: row 8 (q / 4) + 4 h + q % 4 of 32-row half mg + i mw, column li
  const int gt = 4 * cb + ct, m = gt >= ctm ? 1 : 0, j = (gt - m * ctm) * 32 + li;
  const int ld = L.nmat * r;
  float* out = L.part + (int64_t)sp * L.rows_total * ld;
  if (ct < nct && j < r) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int mb = mg + i * mw;
      if (mb >= 2) continue;
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        const int rr = 32 * mb + 8 * (q >> 2) + 4 * h + (q & 3);
        if (rr < rows) {
          const int64_t o = (int64_t)(p0 + rr) * ld + m * r + j;
          if (L.ks == 1) L.a_out[o] = __float2half(acc[i][q]);
          else if (L.cnt) handoff_put(out + o, acc[i][q]);
          else out[o] = acc[i][q];
        }
      }
    }
  }
  if (L.cnt == nullptr || L.ks == 1) return;
  // the block's last split sums them in split order: its tiles' columns are
  // [c0, c0 + 2 nc2) of a row (whole pairs), two a load
  int* flag = (int*)smem;
  __syncthreads();  // every wave is done with smem
  const int nblk = (L.nmat * ctm + 3) / 4;
  if (!handoff_arrive(L.cnt + job * nblk + cb, (unsigned)L.ks, flag)) return;
  auto col0 = [&](int g) { return g >= L.nmat * ctm ? L.nmat * r : g / ctm * r + g % ctm * 32; };
  const int c0 = col0(4 * cb), nc2 = (col0(4 * cb + 4) - c0) / 2, n2 = rows * nc2;
  for (int i0 = tid; i0 < n2; i0 += 4 * kPfThreads) {
    float s0[4] = {0.f, 0.f, 0.f, 0.f}, s1[4] = {0.f, 0.f, 0.f, 0.f};
    int64_t o[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = min(i0 + kPfThreads * u, n2 - 1);
      o[u] = (int64_t)(p0 + i / nc2) * ld + c0 + 2 * (i % nc2);
    }
    for (int q0 = 0; q0 < L.ks; q0 += 4) {
      unsigned long long v[4][4];
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int u = 0; u < 4; ++u)
          v[q][u] = handoff_get((const unsigned long long*)(L.part + o[u] +
                                (int64_t)min(q0 + q, L.ks - 1) * L.rows_total * ld));
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (q0 + q < L.ks) {
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            s0[u] += __uint_as_float((uint32_t)v[q][u]);
            s1[u] += __uint_as_float((uint32_t)(v[q][u] >> 32));
          }
        }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (i0 + kPfThreads * u < n2)
        *(uint32_t*)(L.a_out + o[u]) = __half_as_ushort(__float2half(s0[u])) |
                                       (uint32_t)__half_as_ushort(__float2half(s1[u])) << 16;
  }
  if (tid == 0) handoff_reset(L.cnt + job * nblk + cb);
}

// a = fp16(x U) of the dense prefill in one launch: workgroup (row block
// rb, K slice sp) forms the fp32 partial of 16 token rows over a slice of
// kLowrankRows codes (lowrank_partial<4>: v_mfma_f32_16x16x32_f16 tiles
// with U staged transposed in LDS), hands it over and counts itself in on
// the row block's counter (glq_handoff.h); the last of the block's slices
// sums them in slice order, rounds once and leaves the counter at zero.
__global__ __launch_bounds__(256) void pf_xu_kernel(const __half* __restrict__ x, int M, int K,
                                                    const __half* __restrict__ U, int rank,
                                                    int rpad, int ns, float* part,
                                                    unsigned* cnt, __half* __restrict__ a_out) {
  __shared__ float red[4 * 4 * 64];
  __shared__ __align__(16) __half xl[16 * kLowrankRows];
  __shared__ __align__(16) __half ut[64 * kLowrankUtStride];
  __shared__ int last;
  const int rb = blockIdx.x / ns, sp = blockIdx.x - rb * ns, tid = threadIdx.x;
  const int r0 = rb * 16, rows = min(16, M - r0);
  const __half* xb = x + (int64_t)r0 * K;
  auto xrow = [&](int m) { return xb + (int64_t)m * K; };
  float* slices = part + (int64_t)rb * ns * 16 * rpad;  // [slice][row][rpad]
  lowrank_partial<4, decltype(xrow), true>(xrow, rows, K, rank, rpad, U, sp,
                                           slices + (int64_t)sp * 16 * rpad, red, xl, tid, ut);
  if (!handoff_arrive(cnt + rb, (unsigned)ns, &last)) return;
  for (int i = tid; i < rows * rank; i += 256) {
    const int m = i / rank, j = i - m * rank;
    a_out[(int64_t)(r0 + m) * rank + j] =
        __float2half(sum_strided_coh(slices + m * rpad + j, 16 * rpad, ns));
  }
  if (tid == 0) handoff_reset(cnt + rb);
}

// Grid: (row blocks, K splits, column blocks).
__global__ __launch_bounds__(kPfThreads) void pf_lowrank_kernel(PfLowrank L) {
  extern __shared__ __align__(16) unsigned char smem[];
  if (L.zero_cnt && blockIdx.x + blockIdx.y + blockIdx.z == 0)
    for (int i = threadIdx.x; i < L.n_cnt; i += kPfThreads) L.zero_cnt[i] = 0u;
  if (L.nmat == 0) return;  // the counters were all there was to do
  pf_lowrank_body(L, blockIdx.x, blockIdx.y, blockIdx.z, smem);
}

// The launch before a dense GEMM in tile form: its first n_lr workgroups are
// the jobs of a = x U (row blocks x K splits x column blocks); each of the
// others puts kPrepGroups (row, 128-code group) units of x in decode order and
// forms their sums c2 (group, row) for fractional zero-points (c2 may be
// null), 8 threads a unit.
struct PfPrep {
  PfLowrank L;
  int n_lr, ncb;
  const __half* x;
  __half* xp;
  float* c2;
  int64_t c2_ld;
  int bits, G;
  int64_t units;  // rows x groups
};
constexpr int kPrepGroups = 128;

__global__ __launch_bounds__(kPfThreads) void pf_prep_kernel(PfPrep p) {
  extern __shared__ __align__(16) unsigned char smem[];
  if ((int)blockIdx.x < p.n_lr) {
    const int cb = blockIdx.x % p.ncb, rest = blockIdx.x / p.ncb;
    pf_lowrank_body(p.L, rest / p.L.ks, rest % p.L.ks, cb, smem);
    return;
  }
  const int64_t u0 = (int64_t)(blockIdx.x - p.n_lr) * kPrepGroups;
  const int l8 = threadIdx.x & 7;
  u32x4 v[4][2];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int64_t u = min(u0 + 32 * q + (threadIdx.x >> 3), p.units - 1);
    const u32x4* s = (const u32x4*)(p.x + u * 128 + 16 * l8);
    v[q][0] = s[0];
    v[q][1] = s[1];
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int64_t u = u0 + 32 * q + (threadIdx.x >> 3);
    const bool in = u < p.units;
    if (in) {
      u32x4 o0, o1;
      pf_permute16(p.bits, v[q][0], v[q][1], o0, o1);
      u32x4* d = (u32x4*)(p.xp + u * 128 + 16 * l8);
      d[0] = o0;
      d[1] = o1;
    }
    if (p.c2) {  // uniform
      float c = 0.f;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const f16x8 hv = __builtin_bit_cast(f16x8, v[q][i]);
#pragma unroll
        for (int e = 0; e < 8; ++e) c += (float)hv[e];
      }
      c += __shfl_xor(c, 1);
      c += __shfl_xor(c, 2);
      c += __shfl_xor(c, 4);
      if (in && l8 == 0) {
        const int64_t row = u / p.G;
        p.c2[(u - row * p.G) * p.c2_ld + row] = c;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Host side shared by the dense GEMM and the MoE prefill
// ---------------------------------------------------------------------------

template <int BITS, int TM, int RT, bool SYM, bool ZF, bool DEEP = false>
static int pf_launch_k(const PfArgs& g, hipStream_t s) {
  static size_t attr = 64 * 1024;
  using SL = PfSlot<BITS, TM, RT, DEEP>;
  size_t lds = (size_t)SL::D * SL::BYTES;
  if (g.xu_rows) lds = std::max(lds, kXuJobLds);  // the x U jobs and the epilogue's local form
  int rc = set_lds_limit(pf_gemm_kernel<BITS, TM, RT, SYM, ZF, DEEP>, lds, attr);
  if (rc) return rc;
  const dim3 grid((unsigned)(g.ntn * g.ks), (unsigned)(g.max_tiles + g.xu_rows));
  pf_gemm_kernel<BITS, TM, RT, SYM, ZF, DEEP><<<grid, dim3(kPfThreads), lds, s>>>(g);
  GLQ_LAUNCH_CHECK("pf_gemm_kernel");
  return GLQ_OK;
}

// Tile of a dense launch: TM token rows x 64 RT weight rows, ring depth.
struct PfTile {
  int tm, rt;
  bool deep;
};

template <int BITS, bool SYM, bool ZF>
static int pf_launch_dense_bits(const PfArgs& g, PfTile t, hipStream_t s) {
  if (t.deep) {
    if (t.tm == 16) {
      if (t.rt == 1) return pf_launch_k<BITS, 16, 1, SYM, ZF, true>(g, s);
      return pf_launch_k<BITS, 16, 2, SYM, ZF, true>(g, s);
    }
    if (t.tm == 32) {
      if (t.rt == 1) return pf_launch_k<BITS, 32, 1, SYM, ZF, true>(g, s);
      return pf_launch_k<BITS, 32, 2, SYM, ZF, true>(g, s);
    }
    return pf_launch_k<BITS, 64, 2, SYM, ZF, true>(g, s);
  }
  if (t.tm == 128) return pf_launch_k<BITS, 128, 2, SYM, ZF>(g, s);
  if (t.tm == 64) return pf_launch_k<BITS, 64, 2, SYM, ZF>(g, s);
  return pf_launch_k<BITS, 32, 4, SYM, ZF>(g, s);
}

static int pf_launch_dense(const PfArgs& g, int bits, PfTile t, bool sym, hipStream_t s) {
  if (bits == 2) {
    return sym ? pf_launch_dense_bits<2, true, false>(g, t, s)
               : pf_launch_dense_bits<2, false, true>(g, t, s);
  }
  return sym ? pf_launch_dense_bits<4, true, false>(g, t, s)
             : pf_launch_dense_bits<4, false, true>(g, t, s);
}

// Weight rows of a workgroup of the tile form (glq_pf_tile.h) of tm = 32, 64
// (x 256 rows) or 128 (x 128 rows) tokens; a gate/up tile holds half as many
// rows of each matrix.
static int pt_wg_rows(int mode, int tm) {
  const int r = tm == 128 ? 128 : 256;
  return mode == kPfGateUp ? r / 2 : r;
}
static int pt_tiles_n(int64_t N, int mode, int tm) {
  const int r = pt_wg_rows(mode, tm);
  return (int)((N + r - 1) / r);
}

// K splits of a DOWN launch of `wgs` workgroups over G groups: towards two
// workgroups a CU, at least four groups each, at most 8 (whole pairs of groups
// where the rows' scales are).  Splits cost a fp32 pass over the results, so a
// launch of 256 workgroups or more has none.  (256 tokens x 5632 -> 2048: 32
// workgroups of 44 groups, 56 us unsplit.)
static int pt_down_split(int64_t wgs, int G, int& gps) {
  int ks = wgs >= 256 ? 1 : (int)std::min<int64_t>({8, 512 / wgs, std::max(1, G / 4)});
  ks = std::max(ks, 1);
  gps = (G + ks - 1) / ks;
  if (G % 2 == 0) gps = (gps + 1) / 2 * 2;
  return (G + gps - 1) / gps;
}

// fp32 elements pf_shared_launch may write to sy.
static int64_t pf_shared_sy_elems(int64_t T, int64_t H, int64_t SI, int tm) {
  int gps;
  const int64_t wgs = (int64_t)pt_tiles_n(H, kPfDown, tm) * ((T + tm - 1) / tm);
  return (int64_t)pt_down_split(wgs, (int)(SI / 128), gps) * T * H;
}

// K splits of the routed down of Pn pairs: its workgroups estimated from full
// tiles and one ragged tile an expert.  (Mixtral-shaped layer, 32 tokens: 128
// workgroups of 112 groups, 98 us unsplit.)
static int pt_routed_split(int64_t Pn, int64_t E, int64_t H, int tm, int G, int& gps) {
  return pt_down_split(pt_tiles_n(H, kPfDown, tm) * (Pn / tm + std::min(E, Pn)), G, gps);
}

// Arrival counters of the low-rank launches over a tile list (at most two
// column blocks: two matrices of rank 128).
static int pf_lrcnt(int max_tiles, int tm) { return max_tiles * ((tm + 63) / 64) * 2; }

template <int MODE, bool SYM, bool ZF>
static int pt_launch_tm(const PfArgs& g, int bits, int tm, hipStream_t s) {
  if constexpr (MODE != kPfDense)
    if (tm == 128) return pt_launch<2, 2, 2, MODE, SYM, ZF>(g, bits, s);
  if (tm == 64) return pt_launch<1, 4, 2, MODE, SYM, ZF>(g, bits, s);
  return pt_launch<1, 4, 1, MODE, SYM, ZF>(g, bits, s);
}

// a = fp16(sum of the K-split partials in split order): four elements a thread
// (n is a multiple of 8).
__global__ __launch_bounds__(256) void pf_lowrank_finalize_kernel(const float* part, int ks,
                                                                  int64_t n, __half* a) {
  const int64_t i = 4 * ((int64_t)blockIdx.x * 256 + threadIdx.x);
  if (i >= n) return;
  float s[4] = {0.f, 0.f, 0.f, 0.f};
  for (int q0 = 0; q0 < ks; q0 += 4) {
    float4 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = *(const float4*)(part + min(q0 + u, ks - 1) * n + i);
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (q0 + u < ks) {
        s[0] += v[u].x;
        s[1] += v[u].y;
        s[2] += v[u].z;
        s[3] += v[u].w;
      }
  }
  uint16_t o[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) o[u] = __half_as_ushort(__float2half(s[u]));
  *(u32x2*)(a + i) = u32x2{o[0] | (uint32_t)o[1] << 16, o[2] | (uint32_t)o[3] << 16};
}

// n_jobs: 64-row blocks; with no matrix, one workgroup still clears L.zero_cnt.
static int pf_lowrank_launch(const PfLowrank& L, int n_jobs, hipStream_t s) {
  if (L.nmat == 0) n_jobs = L.zero_cnt ? 1 : 0;
  if (n_jobs == 0) return GLQ_OK;
  const int ctm = (L.rank + 31) / 32;
  const dim3 grid((unsigned)n_jobs, (unsigned)(L.nmat ? L.ks : 1),
                  (unsigned)(L.nmat ? (L.nmat * ctm + 3) / 4 : 1));
  static size_t attr = 64 * 1024;
  int rc = set_lds_limit(pf_lowrank_kernel, (size_t)kLrLds, attr);
  if (rc) return rc;
  pf_lowrank_kernel<<<grid, dim3(kPfThreads), kLrLds, s>>>(L);
  GLQ_LAUNCH_CHECK("pf_lowrank_kernel");
  if (L.nmat > 0 && L.ks > 1 && !L.cnt) {
    const int64_t n = (int64_t)L.rows_total * L.nmat * L.rank;
    pf_lowrank_finalize_kernel<<<dim3((unsigned)((n / 4 + 255) / 256)), dim3(256), 0, s>>>(
        L.part, L.ks, n, L.a_out);
    GLQ_LAUNCH_CHECK("pf_lowrank_finalize_kernel");
  }
  return GLQ_OK;
}

// K split of a = x U for `blocks` workgroups a split: enough splits for about
// 512 workgroups (two on each CU), at most 16, each of at least 256 codes.
static void pf_lowrank_split(int64_t K, int64_t blocks, int& ks, int& kps) {
  int64_t n = std::max<int64_t>(1, std::min<int64_t>(16, 512 / std::max<int64_t>(blocks, 1)));
  n = std::max<int64_t>(1, std::min<int64_t>(n, K / 256));
  const int64_t per = ((K + n - 1) / n + 127) / 128 * 128;
  kps = (int)per;
  ks = (int)((K + per - 1) / per);
}

// ---------------------------------------------------------------------------
// Dense plan: token tile, K splits and workspace of one projection.
// ---------------------------------------------------------------------------
struct PfDensePlan {
  int pt;            // token tile of the tile form (glq_pf_tile.h), or 0
  int64_t xp_bytes, c2_bytes, c2_ld;
  int tm, rt, ntn, ntm, ks, gps, lr_ks, lr_kps;
  bool deep;
  bool xu1;          // a = x U by pf_xu_kernel (one launch)
  int xu_ns;         // its K slices
  int64_t a_bytes, lp_bytes, part_bytes, cnt_bytes, total;
};

// The dense prefill workspace starts with kPfSyncBytes of counter words (the
// x U row blocks' arrivals), zero before the first call and after every
// call, so the one-launch x U takes at most kPfSyncBytes / 4 row blocks.
constexpr int64_t kPfSyncBytes = 4096;

// Token tile of the tile form (64 or 32, x 256 rows) for a dense launch, or 0
// where pf_gemm_kernel's smaller tiles are the better form: estimates of the
// three in us, with x U formed in the call (xu) or none to form.  Each form's
// time is a start, then a cost a 128-code group for its first round of 256
// workgroups and one for every further round (a CU's workgroups share its
// rate, so a round begun costs nearly a whole one): 257 tiles take as long as
// 500.  The tile form's launch before costs 7 us with x U; pf_gemm_kernel
// forms x U in its own grid, where its epilogues wait for it.  The tile form is
// taken where it is 5 % ahead.  Over 22 shapes (K 512 to 14336, N 512 to
// 14336, both widths) x 20 row counts from 17 to 2048, the rule's choice is 0.6
// (xu) and 0.1 % (none) off the best of the three in the mean, and never 3 %
// slower than pf_gemm_kernel; over 360 further random calls 4 and 0.6 % off,
// six of them more than 5 % slower than pf_gemm_kernel (the worst 82 against
// 66 us: 4-bit, 8192, 1000, 336 rows).
//   (K, N, bits, M): tile form 32 / 64, pf_gemm_kernel (us)
//   with x U:                                        no x U:
//   2048, 4096, 4,  512: 35.4 / 41.6, 35.7            26.4 / 31.8, 23.1
//   2048, 4096, 4, 1024: 51.7 / 45.6, 63.6            41.7 / 36.1, 31.5
//   4096, 4096, 2,  256: 48.3 / 57.7, 41.5            37.3 / 45.1, 31.8
//   4096, 4096, 4,  640: 81.1 / 62.6, 75.6            68.2 / 50.3, 54.3
//   4096, 4096, 4, 2048: 150.7 / 112.2, 160.7         132.9 / 94.3, 111.2
//   768, 2048, 2,  2048: 33.3 / 33.8, 39.5            25.4 / 25.0, 16.6
static int pt_dense_tile(int64_t M, int64_t K, int64_t N, int bits, bool xu) {
  if (N * K * bits / 8 >= (1ll << 32)) return 0;  // its code offsets have 32 bits
  const auto up = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
  const double G = (double)(K / 128);
  // us of a launch of tm x wr tiles
  const auto us = [&](int tm, int wr, double start, double first, double more) {
    return start + G * (first + more * (double)(up(up(M, tm) * up(N, wr), 256) - 1));
  };
  double t64, t32, old;
  const bool big = up(M, 64) * up(N, 128) >= 256;  // pf_dense_plan's tiles
  if (xu) {
    t64 = us(64, 256, 20, 1.25, 0.87);
    t32 = us(32, 256, 18, 0.92, 0.91);
    old = big        ? us(64, 128, 11.7, 1.47, 0.98)
          : M >= 256 ? us(32, 128, 14.7, 1.04, 0.28)
                     : us(16, 64, 12.6, 0.58, 0.42);
  } else {
    t64 = us(64, 256, 13, 1.27, 0.87);
    t32 = us(32, 256, 11, 0.95, 0.92);
    old = big        ? us(64, 128, 5.6, 1.05, 0.74)
          : M >= 256 ? us(32, 128, 4.6, 0.76, 0.36)
                     : us(16, 64, 4.3, 0.52, 0.475);
  }
  if (std::min(t32, t64) >= 0.95 * old) return 0;
  return t64 <= t32 ? 64 : 32;
}

// The tests' GLQ_PF_* settings.  One pass over the environment a plan finds
// that there is none (a call makes five plans).
struct PfEnv {
  bool any = false;
  PfEnv() {
    for (char** e = environ; e && *e; ++e)
      if ((*e)[0] == 'G' && strncmp(*e, "GLQ_PF_", 7) == 0) any = true;
  }
  const char* get(const char* name) const { return any ? getenv(name) : nullptr; }
};

// tile: the tile form may be taken.
static PfDensePlan pf_dense_plan(int64_t M, int64_t K, int64_t N, int64_t rank, int bits,
                                 bool tile) {
  PfDensePlan P;
  const PfEnv env;
  // Big launches (a 64 x 128 tile per CU or more): 64-token tiles, shallow
  // rings, two workgroups per CU.  Smaller ones: 32-token tiles of
  // 128 rows from 256 tokens, else 16-token tiles of 64 rows, with deep rings
  // (the whole K range of a small tile nearly in flight).  No K split: the
  // tiles are sized to give the chip enough workgroups without one.
  const int64_t t64 = ((M + 63) / 64) * ((N + 127) / 128);
  if (t64 >= 256) {
    // (64-token tiles: the 128-token tile of asymmetric codes needs more
    // than 256 VGPRs and spills)
    P.tm = 64;
    P.rt = 2;
    P.deep = false;
  } else if (M >= 256) {
    P.tm = 32;
    P.rt = 2;
    P.deep = true;
  } else {
    P.tm = 16;
    P.rt = 1;
    P.deep = true;
  }
  if (const char* e = env.get("GLQ_PF_CFG")) {  // "tm,rt,deep": a supported tile
    int tm = 0, rt = 0, deep = 0;
    if (sscanf(e, "%d,%d,%d", &tm, &rt, &deep) == 3) {
      const bool ok = deep ? ((tm == 16 || tm == 32) && (rt == 1 || rt == 2)) || (tm == 64 && rt == 2)
                           : (tm == 32 && rt == 4) || ((tm == 64 || tm == 128) && rt == 2);
      if (ok) {
        P.tm = tm;
        P.rt = rt;
        P.deep = deep != 0;
      }
    }
  }
  const int wgr = 64 * P.rt;
  P.ntn = (int)((N + wgr - 1) / wgr);
  P.ntm = (int)((M + P.tm - 1) / P.tm);
  const int G = (int)(K / 128);
  int ks = 1;
  if (const char* e = env.get("GLQ_PF_KS")) ks = std::max(1, std::min(G, atoi(e)));
  P.gps = (G + ks - 1) / ks;
  P.ks = (G + P.gps - 1) / P.gps;
  P.pt = 0;
  P.xp_bytes = P.c2_bytes = P.c2_ld = 0;
  if (tile && ks == 1 && !env.get("GLQ_PF_CFG")) {
    P.pt = pt_dense_tile(M, K, N, bits, rank > 0);
    if (const char* e = env.get("GLQ_PF_TILE")) {  // the tile form (0: not) of 32 or 64 tokens
      const int v = atoi(e);
      if (v == 0 || ((v == 32 || v == 64) && N * K * bits / 8 < (1ll << 32))) P.pt = v;
    }
  }
  pf_lowrank_split(K, (M + kLrRows - 1) / kLrRows, P.lr_ks, P.lr_kps);
  if (P.pt) {
    // x in decode order, its group sums (whole tiles of rows), a and its
    // partials, summed in their launch (a counter word per 64-row block)
    P.ntn = pt_tiles_n(N, kPfDense, P.pt);
    P.ntm = (int)((M + P.pt - 1) / P.pt);
    P.ks = 1;
    P.gps = G;
    if ((M + kLrRows - 1) / kLrRows > kPfSyncBytes / 4) {
      P.lr_ks = 1;
      P.lr_kps = (int)K;
    }
    P.xu1 = false;
    P.xp_bytes = align_up(M * K * 2, 256);
    P.c2_ld = align_up(M, 128);
    P.c2_bytes = align_up((int64_t)G * P.c2_ld * 4, 256);
    P.a_bytes = rank > 0 ? align_up(M * rank * 2, 256) : 0;
    P.lp_bytes = rank > 0 && P.lr_ks > 1 ? align_up((int64_t)P.lr_ks * M * rank * 4, 256) : 0;
    P.part_bytes = P.cnt_bytes = 0;
    P.total = kPfSyncBytes + P.xp_bytes + P.c2_bytes + P.a_bytes + P.lp_bytes;
    return P;
  }
  P.a_bytes = rank > 0 ? align_up(M * rank * 2, 256) : 0;
  // a = x U in one launch (16-row blocks x K slices, last arrivers sum) when
  // the GEMM needs no split-K counters (those are cleared by the two-launch
  // form's first launch)
  const int64_t nrb = (M + 15) / 16;
  P.xu_ns = (int)((K + kLowrankRows - 1) / kLowrankRows);
  P.xu1 = rank > 0 && rank <= 128 && P.ks == 1 && nrb <= kPfSyncBytes / 4 &&
          !env.get("GLQ_PF_XU2");
  if (P.xu1) {
    const int64_t rpad = align_up(rank, 32);
    P.lp_bytes = align_up(nrb * P.xu_ns * 16 * rpad * 4, 256);
  } else {
    P.lp_bytes = rank > 0 && P.lr_ks > 1 ? align_up((int64_t)P.lr_ks * M * rank * 4, 256) : 0;
  }
  P.part_bytes = P.ks > 1 ? align_up((int64_t)P.ks * P.ntm * P.tm * P.ntn * 64 * P.rt * 4, 256)
                          : 0;
  P.cnt_bytes = P.ks > 1 ? align_up((int64_t)P.ntm * P.ntn * 4, 256) : 0;
  // the counter words come first in every workspace this path uses, so no
  // call's tables overwrite another's counters
  const int64_t body = P.a_bytes + P.lp_bytes + P.part_bytes + P.cnt_bytes;
  P.total = body ? kPfSyncBytes + body : 0;
  return P;
}

// Workspace of the prefill path of glq_gemm_lora: kPfSyncBytes of counter
// words (zero before the first call, left zero by every call), then a, its
// partials, the split-K tiles (whose arrival counters the two-launch form's
// first launch clears); none at all when the call needs no tables.
// With the tile form allowed, or (tile false) what the call takes at least.
int64_t pf_gemm_prefill_workspace_bytes(int64_t M, int64_t K, int64_t N, int64_t rank,
                                        int bits, bool tile) {
  if (M <= 0 || K <= 0 || N <= 0) return 0;
  if (rank < 0) return -1;
  return pf_dense_plan(M, K, N, rank, bits, tile).total;
}

// The dense GEMM in tile form: x in decode order, a = x U, then the tiles.
static int pt_dense_gemm(const PfDensePlan& P, const void* x, int64_t M, int64_t K, int64_t N,
                         const int32_t* codes, int bits, const void* scales, const void* zeros,
                         int sym, const void* U, const void* SV, int64_t rank, const void* xU,
                         const void* bias, void* y, void* workspace, hipStream_t s) {
  char* w = (char*)workspace + kPfSyncBytes;
  PfPrep q = {};
  q.x = (const __half*)x;
  q.xp = (__half*)w;
  q.c2 = sym == 1 ? nullptr : (float*)(w + P.xp_bytes);
  q.c2_ld = P.c2_ld;
  q.bits = bits;
  q.G = (int)(K / 128);
  q.units = M * q.G;
  const bool lora = SV != nullptr && rank > 0;
  __half* abuf = (__half*)(w + P.xp_bytes + P.c2_bytes);
  q.ncb = 1;
  if (lora && xU == nullptr) {
    PfLowrank& L = q.L;
    L.x = q.x;
    L.nmat = 1;
    L.U[0] = (const __half*)U;
    L.rows_total = (int)M;
    L.K = (int)K;
    L.rank = (int)rank;
    L.ks = P.lr_ks;
    L.kps = P.lr_kps;
    L.part = (float*)((char*)abuf + P.a_bytes);
    L.a_out = abuf;
    L.cnt = P.lr_ks > 1 ? (unsigned*)workspace : nullptr;
    q.n_lr = (int)((M + kLrRows - 1) / kLrRows) * P.lr_ks;
  }
  const int64_t grid = q.n_lr + (q.units + kPrepGroups - 1) / kPrepGroups;
  GLQ_CHECK(grid < (1ll << 31), "too many workgroups");
  static size_t attr = 64 * 1024;
  const size_t lds = q.n_lr ? (size_t)kLrLds : 0;
  int rc = set_lds_limit(pf_prep_kernel, lds, attr);
  if (rc) return rc;
  pf_prep_kernel<<<dim3((unsigned)grid), dim3(kPfThreads), lds, s>>>(q);
  GLQ_LAUNCH_CHECK("pf_prep_kernel");
  PfArgs g = {};
  g.xp = q.xp;
  g.c2 = q.c2;
  g.c2_ld = q.c2_ld;
  g.codes[0] = (const uint32_t*)codes;
  g.scales[0] = (const __half*)scales;
  g.zeros[0] = (const __half*)zeros;
  g.a = lora ? (xU ? (const __half*)xU : abuf) : nullptr;
  g.a_ld = (int)rank;
  g.sv[0] = lora ? (const __half*)SV : nullptr;
  g.bias = (const __half*)bias;
  g.y = (__half*)y;
  g.y_ld = N;
  g.M = (int)M;
  g.K = (int)K;
  g.N = (int)N;
  g.G = q.G;
  g.kw = (int)(K * bits / 32);
  g.rank = lora ? (int)rank : 0;
  g.ntn = P.ntn;
  g.max_tiles = P.ntm;
  g.zoff = sym == 2 ? (float)(1 << (bits - 1)) : 0.f;
  return sym == 1 ? pt_launch_tm<kPfDense, true, false>(g, bits, P.pt, s)
                  : pt_launch_tm<kPfDense, false, true>(g, bits, P.pt, s);
}

// The prefill GEMM of glq_gemm_lora (called after its argument checks).
int pf_dense_gemm(const void* x, int64_t M, int64_t K, int64_t N, const int32_t* codes,
                  int bits, const void* scales, const void* zeros, int sym, const void* U,
                  const void* SV, int64_t rank, const void* xU, const void* bias, void* y,
                  void* workspace, int64_t workspace_bytes, hipStream_t s) {
  const bool lora = SV != nullptr && rank > 0;
  // a = x U needs room only when it is formed here
  const int64_t xr = lora && xU == nullptr ? rank : 0;
  PfDensePlan P = pf_dense_plan(M, K, N, xr, bits, true);
  // a workspace too small for the tile form takes the other one
  if (P.pt && workspace_bytes < P.total) P = pf_dense_plan(M, K, N, xr, bits, false);
  GLQ_CHECK(P.total == 0 || (workspace != nullptr && workspace_bytes >= P.total),
            "workspace of %lld bytes needed (got %lld)", (long long)P.total,
            (long long)workspace_bytes);
  GLQ_CHECK(M * K < (1ll << 31), "M*K too large for the prefill path");
  if (P.pt)
    return pt_dense_gemm(P, x, M, K, N, codes, bits, scales, zeros, sym, U, SV, rank, xU, bias, y,
                         workspace, s);
  unsigned* xcnt = (unsigned*)workspace;  // zero between calls
  char* w = (char*)workspace + (P.total ? kPfSyncBytes : 0);
  __half* abuf = P.a_bytes ? (__half*)w : nullptr;
  float* lpart = P.lp_bytes ? (float*)(w + P.a_bytes) : nullptr;
  char* w3 = w + P.a_bytes + P.lp_bytes;
  float* part = P.ks > 1 ? (float*)w3 : nullptr;
  unsigned* cnt = P.ks > 1 ? (unsigned*)(w3 + P.part_bytes) : nullptr;
  const PfEnv env;
  const bool fused = P.xu1 && xU == nullptr && !env.get("GLQ_PF_XU1");
  if (fused) {
    // a = x U in the GEMM's launch (its first grid rows)
  } else if (P.xu1 && xU == nullptr) {
    // launch 1: a = x U in one launch (its row blocks count on the
    // workspace's first words)
    const int nrb = (int)((M + 15) / 16);
    pf_xu_kernel<<<dim3((unsigned)(nrb * P.xu_ns)), dim3(256), 0, s>>>(
        (const __half*)x, (int)M, (int)K, (const __half*)U, (int)rank,
        (int)align_up(rank, 32), P.xu_ns, lpart, xcnt, abuf);
    GLQ_LAUNCH_CHECK("pf_xu_kernel");
  } else if (P.a_bytes || cnt) {
    // launch 1 (when U is given, or split-K counters need clearing): the split
    // partials of a = x U, summed by a finalize launch
    PfLowrank L = {};
    L.x = (const __half*)x;
    L.aperm = 0;
    L.nmat = P.a_bytes ? 1 : 0;
    L.U[0] = (const __half*)U;
    L.u_cs = 0;
    L.tile_rows = kLrRows;
    L.rows_total = (int)M;
    L.K = (int)K;
    L.rank = L.nmat ? (int)rank : 8;
    L.ks = P.lr_ks;
    L.kps = P.lr_kps;
    L.part = lpart;
    L.a_out = abuf;
    L.zero_cnt = cnt;  // the GEMM's split-K counters start at zero
    L.n_cnt = P.ntm * P.ntn;
    int rc = pf_lowrank_launch(L, (int)((M + kLrRows - 1) / kLrRows), s);
    if (rc) return rc;
  }
  // launch 2: the GEMM, A = x in natural order
  PfArgs g = {};
  g.xp = (const __half*)x;
  g.codes[0] = (const uint32_t*)codes;
  g.scales[0] = (const __half*)scales;
  g.zeros[0] = (const __half*)zeros;
  g.a = lora ? (xU ? (const __half*)xU : abuf) : nullptr;
  g.a_ld = (int)rank;
  g.sv[0] = lora ? (const __half*)SV : nullptr;
  g.bias = (const __half*)bias;
  g.y = (__half*)y;
  g.y_ld = N;
  g.part = part;
  g.cnt = cnt;
  g.M = (int)M;
  g.K = (int)K;
  g.N = (int)N;
  g.G = (int)(K / 128);
  g.kw = (int)(K * bits / 32);
  g.rank = lora ? (int)rank : 0;
  g.ntn = P.ntn;
  g.ks = P.ks;
  g.gps = P.gps;
  g.max_tiles = P.ntm;
  g.zoff = sym == 2 ? (float)(1 << (bits - 1)) : 0.f;
  if (fused) {
    g.xu_nrb = (int)((M + 15) / 16);
    g.xu_ns = P.xu_ns;
    g.xu_rows = (int)((g.xu_nrb * g.xu_ns + g.ntn * g.ks - 1) / (g.ntn * g.ks));
    g.xu_rpad = (int)align_up(rank, 32);
    g.xu_u = (const __half*)U;
    g.xu_part = lpart;
    g.xu_cnt = xcnt;
    // GLQ_PF_SPIN_TICKS: the epilogue's wait bound (tests set 0 to take the
    // local form)
    const char* e = env.get("GLQ_PF_SPIN_TICKS");
    g.xu_spin = e ? (uint64_t)strtoull(e, nullptr, 10) : 100000;  // 1 ms
  }
  return pf_launch_dense(g, bits, PfTile{P.tm, P.rt, P.deep}, sym == 1, s);
}
}  // namespace glq

namespace glq {

// ===========================================================================
// MoE block over many tokens (glq_moe_prefill): the reference's
// _forward_sparse (inference/moe_block.py:704-740) semantics -- route every
// token, gather each active expert's tokens, run its SwiGLU projections on
// them, weight and sum -- with the decode step's routing and combine
// arithmetic (glq_moe.hip), so a prompt and a decode step of the same tokens
// agree.
//   1. pf_moe_route_kernel     logits (MFMA, fp32 sums rounded once), softmax,
//                              top-k, weights, the shared-expert gate, and x in
//                              the decode order(s) of the GEMMs
//   2. pf_moe_dispatch_kernel  per-expert counts and positions: the pairs
//                              (token, pick) sorted by expert, and the list of
//                              TM-row tiles (expert, first row, rows)
//   3. pf_lowrank_kernel       a = x U_c(e) for gate and up per pair
//   4. tile form GATE/UP       inter = SwiGLU per pair (down's decode order)
//   5. pf_lowrank_kernel       a = inter U_down,c(e) per pair
//   6. tile form DOWN          y per pair (fp32, in K splits)
//   7. shared expert (GATE/UP, DOWN over all tokens), when present: riding in 4
//      and 6 as a pair launch, or two launches of its own
//   8. pf_moe_combine_kernel   out = fp16(sum_k w_k y_k + sg fp16(shared))
//                              (+ residual)
// Rows within an expert come in the order of an atomic counter, but every
// row's results depend on that row alone, so the output is the same on
// every run.
// ===========================================================================
struct PfMoe {
  int T, H, E, I, topk, norm, SI, bits, sbits, tm, max_tiles;
  const __half* h;
  const __half* router_w;  // (E, H)
  const __half* sgw;       // (H,) or null
  __half* logits_out;      // (T, E) or null
  __half* xp;              // (T, H) in the routed experts' decode order
  __half* xps;             // (T, H) in the shared expert's decode order (may alias xp)
  int32_t* sel;            // (T * topk) expert of each pick
  __half* wts;             // (T * topk)
  __half* sg;              // (T,) sigmoid(shared gate logit)
  int32_t* pos;            // (T * topk) sorted row of each pick
  int32_t* stok;           // (T * topk) token of each sorted row
  int32_t* tiles;          // (max_tiles, 3)
  int32_t* ntiles;
  unsigned* lrcnt;         // the low-rank launches' arrival counters (zeroed here)
  int n_lrcnt;
  const float* ybuf;       // (yks, T * topk, H) routed outputs per sorted row in K splits
  int yks;
  const float* sy;         // (sks, T, H) shared expert output in K splits, or null
  int sks;
  const __half* syh;       // or it as fp16
  const __half* xsrc;      // rows that xp holds in decode order (null: h)
  const __half* res;       // (T, H) residual or null
  __half* out;             // (T, H)
};

// Largest of the wave's 64 unsigned values, on every lane.
__device__ __forceinline__ uint32_t pf_wave_max(uint32_t v) {
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xF, 0xF, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xF, 0xF, false));
  const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  v = max(r[0], r[1]);
  const auto q = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return max(q[0], q[1]);
}

// Rows t0 .. t0 + 15 of x in the routed experts' decode order (and in the
// shared expert's when it differs), by 512 threads, four blocks in flight.
__device__ __forceinline__ void pf_permute_rows(const PfMoe& a, int t0, int tid) {
  const int nb = a.H / 16, n = min(16, a.T - t0) * nb;  // 16-half blocks
  for (int which = 0; which < 2; ++which) {
    __half* dst = which ? a.xps : a.xp;
    if (dst == nullptr || (which && dst == a.xp)) continue;
    const __half* src = (which == 0 && a.xsrc ? a.xsrc : a.h) + (int64_t)t0 * a.H;
    const int bits = which ? a.sbits : a.bits;
    dst += (int64_t)t0 * a.H;
    for (int i0 = tid; i0 < n; i0 += 4 * 512) {
      u32x4 v[4][2];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const __half* p = src + 16 * (int64_t)min(i0 + 512 * u, n - 1);
        v[u][0] = *(const u32x4*)p;
        v[u][1] = *(const u32x4*)(p + 8);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int i = i0 + 512 * u;
        if (i >= n) continue;
        u32x4 o0, o1;
        pf_permute16(bits, v[u][0], v[u][1], o0, o1);
        *(u32x4*)(dst + 16 * (int64_t)i) = o0;
        *(u32x4*)(dst + 16 * (int64_t)i + 8) = o1;
      }
    }
  }
}

// n rows of 16-half blocks in the 4-bit decode order: two blocks a thread.
__global__ __launch_bounds__(256) void pf_permute_kernel(const __half* src, int64_t blocks,
                                                         __half* dst) {
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int64_t i = ((int64_t)blockIdx.x * 2 + u) * 256 + threadIdx.x;
    if (i >= blocks) continue;
    u32x4 o0, o1;
    pf_permute16(4, *(const u32x4*)(src + 16 * i), *(const u32x4*)(src + 16 * i + 8), o0, o1);
    *(u32x4*)(dst + 16 * i) = o0;
    *(u32x4*)(dst + 16 * i + 8) = o1;
  }
}

// One workgroup per 16 tokens: logits of every router row (MFMA tiles of 16
// rows, K split over four of the eight waves, partial tiles summed in LDS in
// wave order), then per token (one wave) softmax, top-k with ties to the
// lower index and weights.  A second workgroup a block writes the rows of x
// in decode order meanwhile.
//
// It is a chain of memory round trips and of cross-lane steps: each wave
// holds every other router tile (NT of them) and loads two to eight K steps
// of them and of x at once, and an argmax is one key (moe_key) through DPP and
// permlane steps.  A tile at a time, a K step at a time and value and index
// through LDS shuffles, it took 107 us at 1500 tokens x 128 experts, 51 us at
// 512 x 8 over 4096 columns.
template <int NT>
__global__ __launch_bounds__(512) void pf_moe_route_kernel(PfMoe a) {
  __shared__ float red[2][4][16][17];  // per wave partial logits of one 16-row tile
  __shared__ float lg[16][257];        // fp16-rounded logits (as float) of the 16 tokens
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, kb = lane >> 4;
  const int kw = wave & 3, par = wave >> 2;  // K quarter, tile parity
  const int t0 = blockIdx.x * 16;
  if (blockIdx.y) {  // uniform: the rows of x in decode order
    pf_permute_rows(a, t0, tid);
    return;
  }
  const int nrow = a.E + (a.sgw ? 1 : 0);
  const int ta = min(t0 + li, a.T - 1);
  const int nks = a.H / 32;
  {
    const __half* xr = a.h + (int64_t)ta * a.H + 8 * kb;
    const __half* wr[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int row = (2 * i + par) * 16 + li;
      wr[i] = row < a.E ? a.router_w + (int64_t)row * a.H + 8 * kb
                        : (row == a.E && a.sgw ? a.sgw + 8 * kb : nullptr);
    }
    f32x4 acc[NT] = {};
    constexpr int U = NT <= 2 ? 8 : NT <= 4 ? 4 : 2;  // K steps loaded at once
    for (int k0 = kw; k0 < nks; k0 += 4 * U) {
      f16x8 av[U], bv[U][NT];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int ks = 32 * min(k0 + 4 * u, nks - 1);
        av[u] = *(const f16x8*)(xr + ks);
#pragma unroll
        for (int i = 0; i < NT; ++i) bv[u][i] = wr[i] ? *(const f16x8*)(wr[i] + ks) : f16x8{};
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (k0 + 4 * u < nks) {  // uniform over the wave
#pragma unroll
          for (int i = 0; i < NT; ++i) acc[i] = mfma_16x16x32(av[u], bv[u][i], acc[i]);
        }
    }
    // acc[i][j]: token 4kb + j, router row li of tile 2 i + par
#pragma unroll
    for (int i = 0; i < NT; ++i) {
#pragma unroll
      for (int j = 0; j < 4; ++j) red[par][kw][4 * kb + j][li] = acc[i][j];
      __syncthreads();
      {
        const int pr = tid >> 8, t = (tid >> 4) & 15, c = tid & 15;
        const float s = red[pr][0][t][c] + red[pr][1][t][c] + red[pr][2][t][c] + red[pr][3][t][c];
        const int row = (2 * i + pr) * 16 + c;
        if (row < nrow) lg[t][row] = __half2float(__float2half(s));
      }
      __syncthreads();
    }
  }
  // routing, one wave per token
  for (int t = wave; t < 16; t += 8) {
    const int tok = t0 + t;
    if (tok >= a.T) continue;
    if (a.logits_out)
      for (int e = lane; e < a.E; e += 64)
        a.logits_out[(int64_t)tok * a.E + e] = __float2half(lg[t][e]);
    if (lane == 0)
      a.sg[tok] = __float2half(a.sgw ? 1.f / (1.f + expf(-lg[t][a.E])) : 1.f);
    // top-k: k rounds of the largest key (logit, then lower index) not yet
    // taken; key 0 is no expert
    uint32_t key[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int e = lane + 64 * q;
      key[q] = e < a.E ? moe_key(__half_as_ushort(__float2half(lg[t][e])), e) : 0u;
    }
    float mx = 0.f, wsel = 0.f;
    int esel = 0;
    for (int j = 0; j < a.topk; ++j) {
      const uint32_t best = pf_wave_max(max(max(key[0], key[1]), max(key[2], key[3])));
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (key[q] == best) key[q] = 0u;
      const float bv = moe_key_logit(best);
      if (j == 0) mx = bv;
      if (lane == j) { esel = 0xFFFF - (int)(best & 0xFFFFu); wsel = bv; }
    }
    float sum = 0.f;
    for (int e = lane; e < a.E; e += 64) sum += expf(lg[t][e] - mx);
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) sum += __shfl_xor(sum, o);
    const float w = lane < a.topk ? expf(wsel - mx) / sum : 0.f;
    float ws = 0.f;
    if (a.norm)
      for (int j = 0; j < a.topk; ++j) ws += __shfl(w, j);
    if (lane < a.topk) {
      a.sel[(int64_t)tok * a.topk + lane] = esel;
      a.wts[(int64_t)tok * a.topk + lane] = __float2half(a.norm ? w / ws : w);
    }
  }
}

// One workgroup: per-expert counts, offsets, each pick's sorted row, the token
// of each sorted row, and the tile list.  A chain of memory round trips, so
// eight picks a thread are loaded at once and the offsets are one wave's scan
// (one load a pick and a serial walk over the experts took 18.7 us for 12000
// picks of 128 experts).
__global__ __launch_bounds__(1024) void pf_moe_dispatch_kernel(PfMoe a) {
  __shared__ int cnt[256], off[256], cur[256], tb[256];
  const int tid = threadIdx.x, P = a.T * a.topk;
  if (tid < 256) cnt[tid] = 0;
  for (int i = tid; i < a.n_lrcnt; i += 1024) a.lrcnt[i] = 0u;
  __syncthreads();
  constexpr int U = 8;
  for (int p0 = 0; p0 < P; p0 += 1024 * U) {
    int e[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int p = p0 + 1024 * u + tid;
      e[u] = p < P ? a.sel[p] : -1;
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (e[u] >= 0) atomicAdd(&cnt[e[u]], 1);
  }
  __syncthreads();
  if (tid < 64) {  // lane l: experts 4 l .. 4 l + 3
    int c[4], rs = 0, ts = 0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      c[u] = cnt[4 * tid + u];
      rs += c[u];
      ts += (c[u] + a.tm - 1) / a.tm;
    }
    int ri = rs, ti = ts;  // inclusive sums over the lanes
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int rv = __shfl_up(ri, o), tv = __shfl_up(ti, o);
      if (tid >= o) {
        ri += rv;
        ti += tv;
      }
    }
    if (tid == 63) *a.ntiles = ti;
    int ro = ri - rs, to = ti - ts;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      off[4 * tid + u] = cur[4 * tid + u] = ro;
      tb[4 * tid + u] = to;
      ro += c[u];
      to += (c[u] + a.tm - 1) / a.tm;
    }
  }
  __syncthreads();
  for (int p0 = 0; p0 < P; p0 += 1024 * U) {
    int e[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int p = p0 + 1024 * u + tid;
      e[u] = p < P ? a.sel[p] : -1;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (e[u] < 0) continue;
      const int p = p0 + 1024 * u + tid, r = atomicAdd(&cur[e[u]], 1);
      a.pos[p] = r;
      a.stok[r] = p / a.topk;
    }
  }
  for (int e = tid; e < a.E; e += 1024) {
    const int n = (cnt[e] + a.tm - 1) / a.tm;
    for (int i = 0; i < n; ++i) {
      int32_t* tl = a.tiles + 3 * (tb[e] + i);
      tl[0] = e;
      tl[1] = off[e] + i * a.tm;
      tl[2] = min(a.tm, cnt[e] - i * a.tm);
    }
  }
}

// out[t][n] = fp16(sum_k w_k y[pos(t, k)][n] + sg[t] fp16(shared[t][n])),
// then fp16(residual + out): the decode step's combine (glq_moe.hip).  Four
// columns a thread, the picks' rows loaded four at a time.  (top_k fp32 rows
// read a token: 98 MB for 1500 tokens x 8 picks x 2048, 36.5 us at one column
// a thread.)
__global__ __launch_bounds__(256) void pf_moe_combine_kernel(PfMoe a) {
  const int64_t i = 4 * ((int64_t)blockIdx.x * 256 + threadIdx.x);
  if (i >= (int64_t)a.T * a.H) return;
  const int t = (int)(i / a.H), n = (int)(i - (int64_t)t * a.H);
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  const int64_t ss = (int64_t)a.T * a.topk * a.H;
  for (int k0 = 0; k0 < a.topk; k0 += 4) {
    float4 v[4];
    float w[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int p = t * a.topk + min(k0 + u, a.topk - 1);
      const float* yp = a.ybuf + (int64_t)a.pos[p] * a.H + n;
      v[u] = *(const float4*)yp;
      w[u] = __half2float(a.wts[p]);
      for (int q = 1; q < a.yks; ++q) {
        const float4 m = *(const float4*)(yp + q * ss);
        v[u].x += m.x;
        v[u].y += m.y;
        v[u].z += m.z;
        v[u].w += m.w;
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (k0 + u < a.topk) {
        acc[0] = fmaf(w[u], v[u].x, acc[0]);
        acc[1] = fmaf(w[u], v[u].y, acc[1]);
        acc[2] = fmaf(w[u], v[u].z, acc[2]);
        acc[3] = fmaf(w[u], v[u].w, acc[3]);
      }
  }
  const float sg = a.sy || a.syh ? __half2float(a.sg[t]) : 0.f;
  float sh[4] = {0.f, 0.f, 0.f, 0.f};
  if (a.sy)
    for (int q0 = 0; q0 < a.sks; q0 += 4) {
      float4 v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u)
        v[u] = *(const float4*)(a.sy + (int64_t)min(q0 + u, a.sks - 1) * a.T * a.H + i);
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (q0 + u < a.sks) {
          sh[0] += v[u].x;
          sh[1] += v[u].y;
          sh[2] += v[u].z;
          sh[3] += v[u].w;
        }
    }
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    if (a.syh) acc[c] = fmaf(sg, __half2float(a.syh[i + c]), acc[c]);
    else if (a.sy) acc[c] = fmaf(sg, __half2float(__float2half(sh[c])), acc[c]);
    float o = __half2float(__float2half(acc[c]));
    if (a.res) o += __half2float(a.res[i + c]);
    a.out[i + c] = __float2half(o);
  }
}

// ---------------------------------------------------------------------------
// Host plan of glq_moe_prefill
// ---------------------------------------------------------------------------
struct PfMoePlan {
  int yks, ygps;  // K splits of the routed down
  int64_t off_lrcnt;
  int tm, max_tiles, ks_gu, kps_gu, ks_d, kps_d, stm;
  int64_t off_xp, off_xps, off_sel, off_wts, off_sg, off_pos, off_stok, off_tiles, off_lp,
      off_agu, off_ad, off_inter, off_y, off_sinter, off_sy, total;
};

static PfMoePlan pf_moe_plan(int64_t T, int64_t H, int64_t E, int64_t I, int64_t k,
                             int64_t rank, int64_t SI, int bits, int sbits) {
  PfMoePlan P;
  const int64_t Pn = T * k;
  const int64_t avg = Pn / std::max<int64_t>(E, 1);
  // Token tile by the mean tokens an expert gets: 128 tokens where most experts
  // fill one such tile and overflow a 64-token one, 64 above, 32 where most
  // of a 64-token tile would be empty.  Whole blocks at 32 / 64 / 128: 19
  // tokens an expert 293 / 336 / 458 us, 47: 382 / 363 / 421.  128 against 64
  // over five blocks (experts, top-k: 60, 4; 128, 8; 8, 2; 32, 4; 64, 6): at 80
  // tokens 0.978 to 0.995 of the time, 88 0.97 to 1.01, 96 0.984 to 1.003;
  // 100 0.97 to 1.04, 104 0.99 to 1.02, 112 1.00 to 1.03, 128 0.99 to 1.08.
  P.tm = avg < 46 ? 32 : (avg >= 80 && avg < 98 ? 128 : 64);
  if (const char* e = getenv("GLQ_PF_MOE_TM")) {
    const int v = atoi(e);
    P.tm = v >= 128 ? 128 : (v >= 64 ? 64 : 32);
  }
  P.max_tiles = (int)((Pn + P.tm - 1) / P.tm + E);
  // (about as many row blocks as experts' full blocks and one ragged each)
  const int64_t lrb = (Pn + kLrRows - 1) / kLrRows + std::min<int64_t>(E, Pn) / 2;
  pf_lowrank_split(H, lrb, P.ks_gu, P.kps_gu);
  pf_lowrank_split(I, lrb, P.ks_d, P.kps_d);
  P.stm = T > 32 && P.tm != 32 ? 64 : 32;
  P.yks = pt_routed_split(Pn, E, H, P.tm, (int)(I / 128), P.ygps);
  int64_t o = 0;
  auto take = [&](int64_t bytes) {
    const int64_t at = o;
    o = align_up(o + bytes, 256);
    return at;
  };
  P.off_xp = take(T * H * 2);
  P.off_xps = (SI > 0 && sbits != bits) ? take(T * H * 2) : P.off_xp;
  P.off_sel = take(Pn * 4);
  P.off_wts = take(Pn * 2);
  P.off_sg = take(T * 2);
  P.off_pos = take(Pn * 4);
  P.off_stok = take(Pn * 4);
  P.off_tiles = take((int64_t)P.max_tiles * 12 + 4);
  P.off_lrcnt = take(4 * (int64_t)pf_lrcnt(P.max_tiles, P.tm));
  const int64_t lp = rank > 0 ? std::max<int64_t>(P.ks_gu > 1 ? P.ks_gu * Pn * 2 * rank * 4 : 0,
                                                  P.ks_d > 1 ? P.ks_d * Pn * rank * 4 : 0)
                              : 0;
  P.off_lp = take(lp);
  P.off_agu = take(rank > 0 ? Pn * 2 * rank * 2 : 0);
  P.off_ad = take(rank > 0 ? Pn * rank * 2 : 0);
  P.off_inter = take(Pn * I * 2);
  P.off_y = take(P.yks * Pn * H * 4);
  P.off_sinter = take(SI > 0 ? T * SI * 2 : 0);
  P.off_sy = take(SI > 0 ? pf_shared_sy_elems(T, H, SI, P.stm) * 4 : 0);
  P.total = o;
  return P;
}

// Launches 1-2 of a prompt: routing (and x in decode order), dispatch.
static int pf_route_launch(const PfMoe& a, hipStream_t s) {
  const int nt = (a.E + (a.sgw ? 1 : 0) + 31) / 32;  // pairs of 16-row router tiles
  const auto kern = nt <= 1   ? pf_moe_route_kernel<1>
                    : nt <= 2 ? pf_moe_route_kernel<2>
                    : nt <= 4 ? pf_moe_route_kernel<4>
                              : pf_moe_route_kernel<9>;
  kern<<<dim3((unsigned)((a.T + 15) / 16), 2), dim3(512), 0, s>>>(a);
  GLQ_LAUNCH_CHECK("pf_moe_route_kernel");
  pf_moe_dispatch_kernel<<<dim3(1), dim3(1024), 0, s>>>(a);
  GLQ_LAUNCH_CHECK("pf_moe_dispatch_kernel");
  return GLQ_OK;
}

// The shared expert over every token, two GEMMs in the tile form of tm tokens:
// xps (T, H) in its decode order -> sinter (T, SI) -> sy (sks, T, H) fp32 in K
// splits.  pair: 32-token tiles of 4-bit codes ride in the routed launches.
struct PfShared {
  PfArgs gu, down;
  int bits, tm;
  bool pair;
};

static PfShared pf_shared(int64_t T, int64_t H, int64_t SI, int bits, int tm, bool pair,
                          const __half* xps, const int32_t* const codes[3],
                          const void* const scales[3], const void* const zeros[3],
                          __half* sinter, float* sy) {
  PfShared S = {};
  S.bits = bits;
  S.tm = tm;
  S.pair = pair && bits == 4 && tm == 32;
  const int ntm = (int)((T + tm - 1) / tm);
  PfArgs& g = S.gu;
  g.xp = xps;
  for (int m = 0; m < 2; ++m) {
    g.codes[m] = (const uint32_t*)codes[m];
    g.scales[m] = (const __half*)scales[m];
    g.zeros[m] = (const __half*)zeros[m];
  }
  g.y = sinter;
  g.y_ld = SI;
  g.M = (int)T; g.K = (int)H; g.N = (int)SI; g.G = (int)(H / 128);
  g.kw = (int)(H * bits / 32);
  g.ntn = pt_tiles_n(SI, kPfGateUp, tm);
  g.out_bits = bits;
  g.max_tiles = ntm;
  PfArgs& d = S.down;
  d.xp = sinter;
  d.codes[0] = (const uint32_t*)codes[2];
  d.scales[0] = (const __half*)scales[2];
  d.zeros[0] = (const __half*)zeros[2];
  d.yf = sy;
  d.yf_ld = H;
  d.M = (int)T; d.K = (int)SI; d.N = (int)H; d.G = (int)(SI / 128);
  d.kw = (int)(SI * bits / 32);
  d.ntn = pt_tiles_n(H, kPfDown, tm);
  d.max_tiles = ntm;
  d.ks = pt_down_split((int64_t)d.ntn * ntm, d.G, d.gps);
  d.yf_ss = T * H;
  return S;
}

// A routed launch, with the shared expert's of the same step where it rides.
template <int BA, int MODE>
static int pf_routed_launch(const PfArgs& g, int tm, const PfShared* S, hipStream_t s) {
  if (S && S->pair && tm == 32)
    return pt_launch_pair<BA, MODE>(g, MODE == kPfGateUp ? S->gu : S->down, s);
  if constexpr (BA == kPtTurbo)
    return tm == 64 ? pt_launch_k<kPtTurbo, 1, 4, 2, MODE, false, false, false>(g, s)
                    : pt_launch_k<kPtTurbo, 1, 4, 1, MODE, false, false, false>(g, s);
  else
    return pt_launch_tm<MODE, false, false>(g, BA, tm, s);
}

// The shared expert's launches, where they do not ride in the routed ones.
static int pf_shared_launch(const PfShared* S, int routed_tm, hipStream_t s) {
  if (!S || (S->pair && routed_tm == 32)) return GLQ_OK;
  const int rc = pt_launch_tm<kPfGateUp, false, false>(S->gu, S->bits, S->tm, s);
  return rc ? rc : pt_launch_tm<kPfDown, false, false>(S->down, S->bits, S->tm, s);
}

static int pf_moe_check(const glq_moe_params* p) {
  GLQ_CHECK(p != nullptr, "null params");
  const int64_t T = p->tokens, H = p->hidden, E = p->experts, I = p->inter, k = p->top_k;
  GLQ_CHECK(T >= 1 && T <= (1 << 20), "tokens=%lld must be in 1..%d", (long long)T, 1 << 20);
  GLQ_CHECK(E >= 1 && E <= 256, "experts=%lld must be in 1..256", (long long)E);
  GLQ_CHECK(k >= 1 && k <= 16 && k <= E && k <= 64, "top_k=%lld out of range", (long long)k);
  GLQ_CHECK(p->group == 128, "group must be 128 (got %d)", p->group);
  GLQ_CHECK(p->bits == 2 || p->bits == 4, "bits must be 2 or 4");
  GLQ_CHECK(H >= 128 && H % 128 == 0 && H <= (1 << 16), "hidden=%lld must be a multiple of 128",
            (long long)H);
  GLQ_CHECK(I >= 128 && I % 128 == 0 && I <= (1 << 17), "inter=%lld must be a multiple of 128",
            (long long)I);
  GLQ_CHECK(T * H < (1ll << 31) && T * k * std::max(I, H) < (1ll << 31), "tokens x width too large");
  const int64_t SI = p->shared_inter;
  GLQ_CHECK(SI >= 0 && SI % 128 == 0 && SI <= (1 << 17), "shared_inter=%lld must be a multiple of 128",
            (long long)SI);
  GLQ_CHECK(T * SI < (1ll << 31), "tokens x shared_inter too large");  // 32-bit row offsets
  if (SI > 0) GLQ_CHECK(p->shared_bits == 2 || p->shared_bits == 4, "shared_bits must be 2 or 4");
  const int64_t r = p->rank;
  const bool lora = r > 0 && p->SV[0] != nullptr;
  if (lora) {
    GLQ_CHECK(r % 8 == 0 && r <= 128, "rank=%lld must be a multiple of 8, <= 128", (long long)r);
    for (int s = 0; s < 3; ++s) {
      GLQ_CHECK(p->U[s] && p->cluster_of[s] && p->SV[s], "U, cluster_of and SV are needed with a rank");
      GLQ_CHECK(p->u_rows[s] >= 0 && p->u_rows[s] < (1ll << 24) && p->n_clusters < (1ll << 24),
                "u_rows or n_clusters out of range");
    }
  }
  GLQ_CHECK(p->h && p->router_w && p->out, "null h, router_w or out");
  for (int s = 0; s < 3; ++s) {
    GLQ_CHECK(p->codes[s] && p->scales[s] && p->zeros[s], "null routed weights (proj %d)", s);
    if (SI > 0)
      GLQ_CHECK(p->shared_codes[s] && p->shared_scales[s] && p->shared_zeros[s],
                "null shared-expert weights (proj %d)", s);
  }
  auto al16 = [](const void* q) { return ((uintptr_t)q & 15) == 0; };
  GLQ_CHECK(al16(p->h) && al16(p->router_w) && (!p->shared_gate_w || al16(p->shared_gate_w)),
            "h, router_w and shared_gate_w must be 16-byte aligned");
  for (int s = 0; s < 3; ++s)
    GLQ_CHECK(al16(p->codes[s]) && (!lora || (al16(p->U[s]) && al16(p->SV[s]))),
              "codes, U and SV must be 16-byte aligned");
  return GLQ_OK;
}

}  // namespace glq

extern "C" int64_t glq_moe_prefill_workspace_bytes(const glq_moe_params* p) {
  using namespace glq;
  clear_error();
  if (pf_moe_check(p) != GLQ_OK) return -1;
  const bool lora = p->rank > 0 && p->SV[0] != nullptr;
  return pf_moe_plan(p->tokens, p->hidden, p->experts, p->inter, p->top_k, lora ? p->rank : 0,
                     p->shared_inter, p->bits, p->shared_bits)
      .total;
}

extern "C" int glq_moe_prefill(const glq_moe_params* p, void* workspace, int64_t workspace_bytes,
                               void* stream) {
  using namespace glq;
  clear_error();
  int rc = pf_moe_check(p);
  if (rc) return rc;
  const int64_t T = p->tokens, H = p->hidden, E = p->experts, I = p->inter, k = p->top_k;
  const int64_t SI = p->shared_inter, Pn = T * k;
  const bool lora = p->rank > 0 && p->SV[0] != nullptr;
  const int r = lora ? (int)p->rank : 0;
  const PfMoePlan P = pf_moe_plan(T, H, E, I, k, r, SI, p->bits, p->shared_bits);
  GLQ_CHECK(workspace != nullptr && workspace_bytes >= P.total && ((uintptr_t)workspace & 255) == 0,
            "a 256-byte aligned workspace of %lld bytes is needed (got %lld)", (long long)P.total,
            (long long)workspace_bytes);
  hipStream_t s = (hipStream_t)stream;
  char* w = (char*)workspace;
  PfMoe a = {};
  a.T = (int)T; a.H = (int)H; a.E = (int)E; a.I = (int)I; a.topk = (int)k;
  a.norm = p->norm_topk_prob ? 1 : 0;
  a.SI = (int)SI; a.bits = p->bits; a.sbits = SI > 0 ? p->shared_bits : p->bits;
  a.tm = P.tm; a.max_tiles = P.max_tiles;
  a.h = (const __half*)p->h;
  a.router_w = (const __half*)p->router_w;
  a.sgw = (const __half*)p->shared_gate_w;
  a.logits_out = (__half*)p->router_logits;
  a.xp = (__half*)(w + P.off_xp);
  a.xps = (__half*)(w + P.off_xps);
  a.sel = (int32_t*)(w + P.off_sel);
  a.wts = (__half*)(w + P.off_wts);
  a.sg = (__half*)(w + P.off_sg);
  a.pos = (int32_t*)(w + P.off_pos);
  a.stok = (int32_t*)(w + P.off_stok);
  a.tiles = (int32_t*)(w + P.off_tiles);
  a.ntiles = a.tiles + 3 * P.max_tiles;
  a.lrcnt = (unsigned*)(w + P.off_lrcnt);
  a.n_lrcnt = pf_lrcnt(P.max_tiles, P.tm);
  a.yks = P.yks;
  a.ybuf = (const float*)(w + P.off_y);
  a.sy = SI > 0 ? (const float*)(w + P.off_sy) : nullptr;
  a.res = (const __half*)p->residual;
  a.out = (__half*)p->out;
  __half* inter = (__half*)(w + P.off_inter);
  float* ybuf = (float*)(w + P.off_y);
  __half* agu = (__half*)(w + P.off_agu);
  __half* ad = (__half*)(w + P.off_ad);
  float* lp = (float*)(w + P.off_lp);

  // 1-2. routing and dispatch
  rc = pf_route_launch(a, s);
  if (rc) return rc;

  PfShared sh;
  const PfShared* shared = nullptr;
  if (SI > 0) {
    sh = pf_shared(T, H, SI, p->shared_bits, P.stm, p->bits == 2, a.xps, p->shared_codes,
                   p->shared_scales, p->shared_zeros, (__half*)(w + P.off_sinter),
                   (float*)(w + P.off_sy));
    shared = &sh;
    a.sks = sh.down.ks;
  }
  // expert strides (elements)
  const int64_t kw_gu = H * p->bits / 32, kw_d = I * p->bits / 32;
  // 3. a = x U for gate and up per pair
  if (lora) {
    PfLowrank L = {};
    L.x = a.xp;
    L.arow = a.stok;
    L.aperm = p->bits;
    L.nmat = 2;
    for (int m = 0; m < 2; ++m) {
      L.U[m] = (const __half*)p->U[m];
      L.cluster[m] = p->cluster_of[m];
      L.uslot[m] = p->u_slot[m];
      L.ncl[m] = (int)p->n_clusters;
      L.urows[m] = (int)(p->u_rows[m] > 0 ? p->u_rows[m] : p->n_clusters);
    }
    L.u_cs = H * r;
    L.tiles = a.tiles;
    L.ntiles = a.ntiles;
    L.tile_rows = P.tm;
    L.rows_total = (int)Pn;
    L.K = (int)H;
    L.rank = r;
    L.ks = P.ks_gu;
    L.kps = P.kps_gu;
    L.part = lp;
    L.cnt = a.lrcnt;
    L.a_out = agu;
    rc = pf_lowrank_launch(L, P.max_tiles * ((P.tm + kLrRows - 1) / kLrRows), s);
    if (rc) return rc;
  }
  // 4. gate/up + SwiGLU -> inter (rows sorted by expert, down's decode order)
  {
    PfArgs g = {};
    g.xp = a.xp;
    g.arow = a.stok;
    for (int m = 0; m < 2; ++m) {
      g.codes[m] = (const uint32_t*)p->codes[m];
      g.scales[m] = (const __half*)p->scales[m];
      g.zeros[m] = (const __half*)p->zeros[m];
      g.sv[m] = lora ? (const __half*)p->SV[m] : nullptr;
    }
    g.codes_es = I * kw_gu;
    g.sz_es = I * (H / 128);
    g.a = lora ? agu : nullptr;
    g.a_ld = 2 * r;
    g.sv_es = I * r;
    g.y = inter;
    g.y_ld = I;
    g.tiles = a.tiles;
    g.ntiles = a.ntiles;
    g.M = (int)Pn; g.K = (int)H; g.N = (int)I; g.G = (int)(H / 128);
    g.kw = (int)kw_gu; g.rank = r;
    g.ntn = pt_tiles_n(I, kPfGateUp, P.tm);
    g.ks = 1; g.gps = g.G;
    g.out_bits = p->bits;
    g.max_tiles = P.max_tiles;
    rc = p->bits == 2 ? pf_routed_launch<2, kPfGateUp>(g, P.tm, shared, s)
                      : pt_launch_tm<kPfGateUp, false, false>(g, 4, P.tm, s);
    if (rc) return rc;
  }
  // 5. a = inter U_down per pair
  if (lora) {
    PfLowrank L = {};
    L.x = inter;
    L.aperm = p->bits;
    L.nmat = 1;
    L.U[0] = (const __half*)p->U[2];
    L.cluster[0] = p->cluster_of[2];
    L.urows[0] = (int)(p->u_rows[2] > 0 ? p->u_rows[2] : p->n_clusters);
    L.u_cs = I * r;
    L.tiles = a.tiles;
    L.ntiles = a.ntiles;
    L.tile_rows = P.tm;
    L.rows_total = (int)Pn;
    L.K = (int)I;
    L.rank = r;
    L.ks = P.ks_d;
    L.kps = P.kps_d;
    L.part = lp;
    L.cnt = a.lrcnt;
    L.a_out = ad;
    rc = pf_lowrank_launch(L, P.max_tiles * ((P.tm + kLrRows - 1) / kLrRows), s);
    if (rc) return rc;
  }
  // 6. down -> y per sorted row (fp32)
  {
    PfArgs g = {};
    g.xp = inter;
    g.codes[0] = (const uint32_t*)p->codes[2];
    g.scales[0] = (const __half*)p->scales[2];
    g.zeros[0] = (const __half*)p->zeros[2];
    g.sv[0] = lora ? (const __half*)p->SV[2] : nullptr;
    g.codes_es = H * kw_d;
    g.sz_es = H * (I / 128);
    g.a = lora ? ad : nullptr;
    g.a_ld = r;
    g.sv_es = H * r;
    g.yf = ybuf;
    g.yf_ld = H;
    g.tiles = a.tiles;
    g.ntiles = a.ntiles;
    g.M = (int)Pn; g.K = (int)I; g.N = (int)H; g.G = (int)(I / 128);
    g.kw = (int)kw_d; g.rank = r;
    g.ntn = pt_tiles_n(H, kPfDown, P.tm);
    g.ks = P.yks; g.gps = P.ygps;
    g.yf_ss = Pn * H;
    g.max_tiles = P.max_tiles;
    rc = p->bits == 2 ? pf_routed_launch<2, kPfDown>(g, P.tm, shared, s)
                      : pt_launch_tm<kPfDown, false, false>(g, 4, P.tm, s);
    if (rc) return rc;
  }
  // 7. shared expert over every token (2-bit or larger tiles)
  rc = pf_shared_launch(shared, p->bits == 2 ? P.tm : 0, s);
  if (rc) return rc;
  // 8. combine
  pf_moe_combine_kernel<<<dim3((unsigned)((T * H / 4 + 255) / 256)), dim3(256), 0, s>>>(a);
  GLQ_LAUNCH_CHECK("pf_moe_combine_kernel");
  return GLQ_OK;
}

namespace glq {
// ===========================================================================
// A TurboQuant block over a prompt (glq_turbo_moe_prefill): the steps of
// glq_moe_prefill with the experts' inputs rotated before their codebook
// GEMMs (the reference's _forward_sparse on TurboQuant layers,
// inference/moe_block.py:704-740, quantized_linear.py:315-349).  x U takes the
// unrotated inputs.  As consecutive 16-token decode steps each read the picked
// experts again: 256 tokens through the 60-expert block took 16 steps, 2.2 ms.
// ===========================================================================
struct TpPlan {
  int yks, ygps;  // K splits of the routed down
  int64_t off_lrcnt;
  int tm, max_tiles, stm, ks_gu, kps_gu, ks_d, kps_d;
  int64_t off_xr, off_xp, off_xps, off_sel, off_wts, off_sg, off_pos, off_stok, off_tiles, off_lp,
      off_agu, off_ad, off_inter, off_tmp, off_xd, off_y, off_sinter, off_sy, total;
};

static TpPlan tp_plan(const glq_turbo_prefill_params* p) {
  const int64_t T = p->tokens, H = p->hidden, E = p->experts, I = p->inter, k = p->top_k;
  const int64_t r = p->rank, SI = p->shared_inter, Pn = T * k;
  TpPlan P;
  P.tm = Pn / std::max<int64_t>(E, 1) < 46 ? 32 : 64;  // as pf_moe_plan's tiles
  P.max_tiles = (int)((Pn + P.tm - 1) / P.tm + E);
  P.stm = T > 32 && P.tm != 32 ? 64 : 32;
  P.yks = pt_routed_split(Pn, E, H, P.tm, (int)(I / 128), P.ygps);
  const int64_t lrb = (Pn + kLrRows - 1) / kLrRows + std::min<int64_t>(E, Pn) / 2;
  pf_lowrank_split(H, lrb, P.ks_gu, P.kps_gu);
  pf_lowrank_split(I, lrb, P.ks_d, P.kps_d);
  int64_t o = 0;
  auto take = [&](int64_t bytes) {
    const int64_t at = o;
    o = align_up(o + bytes, 256);
    return at;
  };
  P.off_xr = take(T * H * 2);
  P.off_xp = take(T * H * 2);
  P.off_xps = take(SI > 0 ? T * H * 2 : 0);
  P.off_sel = take(Pn * 4);
  P.off_wts = take(Pn * 2);
  P.off_sg = take(T * 2);
  P.off_pos = take(Pn * 4);
  P.off_stok = take(Pn * 4);
  P.off_tiles = take((int64_t)P.max_tiles * 12 + 4);
  P.off_lrcnt = take(4 * (int64_t)pf_lrcnt(P.max_tiles, P.tm));
  const int64_t lp = r > 0 ? std::max<int64_t>(P.ks_gu > 1 ? P.ks_gu * Pn * 2 * r * 4 : 0,
                                               P.ks_d > 1 ? P.ks_d * Pn * r * 4 : 0)
                           : 0;
  P.off_lp = take(lp);
  P.off_agu = take(Pn * 2 * r * 2);
  P.off_ad = take(Pn * r * 2);
  P.off_inter = take(Pn * I * 2);
  P.off_tmp = take(p->signs[1] ? Pn * I * 2 : 0);
  P.off_xd = take(Pn * I * 2);
  P.off_y = take(P.yks * Pn * H * 4);
  P.off_sinter = take(SI > 0 ? T * SI * 2 : 0);
  P.off_sy = take(SI > 0 ? pf_shared_sy_elems(T, H, SI, P.stm) * 4 : 0);
  P.total = o;
  return P;
}

static int tp_check(const glq_turbo_prefill_params* p) {
  GLQ_CHECK(p != nullptr, "null params");
  const int64_t T = p->tokens, H = p->hidden, E = p->experts, I = p->inter, k = p->top_k;
  GLQ_CHECK(T >= 1 && T <= (1 << 20), "tokens=%lld must be in 1..%d", (long long)T, 1 << 20);
  GLQ_CHECK(E >= 1 && E <= 256, "experts=%lld must be in 1..256", (long long)E);
  GLQ_CHECK(k >= 1 && k <= 16 && k <= E, "top_k=%lld out of range", (long long)k);
  GLQ_CHECK(H >= 128 && H % 128 == 0 && H <= (1 << 16), "hidden=%lld must be a multiple of 128",
            (long long)H);
  GLQ_CHECK(I >= 128 && I % 128 == 0 && I <= (1 << 16), "inter=%lld must be a multiple of 128",
            (long long)I);
  GLQ_CHECK(T * H < (1ll << 31) && T * k * std::max(I, H) < (1ll << 31), "tokens x width too large");
  GLQ_CHECK(p->rank >= 0 && p->rank % 8 == 0 && p->rank <= 128,
            "rank=%lld must be a multiple of 8, <= 128", (long long)p->rank);
  const int64_t SI = p->shared_inter;
  GLQ_CHECK(SI >= 0 && SI % 128 == 0 && SI <= (1 << 17) && T * std::max<int64_t>(SI, 1) < (1ll << 31),
            "shared_inter=%lld must be a multiple of 128", (long long)SI);
  GLQ_CHECK(SI == 0 || p->shared_bits == 2 || p->shared_bits == 4, "shared_bits must be 2 or 4");
  GLQ_CHECK(SI == 0 || p->shared_y == nullptr, "shared weights or a shared output, not both");
  GLQ_CHECK(p->h && p->router_w && p->out, "null h, router_w or out");
  auto al16 = [](const void* q) { return ((uintptr_t)q & 15) == 0; };
  GLQ_CHECK(al16(p->h) && al16(p->router_w) && (!p->shared_gate_w || al16(p->shared_gate_w)),
            "h, router_w and shared_gate_w must be 16-byte aligned");
  for (int i = 0; i < 3; ++i) {
    GLQ_CHECK(p->codes[i] && p->norms[i] && p->centroids[i] && al16(p->codes[i]),
              "codes (16-byte aligned), norms and centroids are needed (proj %d)", i);
    if (p->rank > 0)
      GLQ_CHECK(p->U[i] && p->cluster_of[i] && p->SV[i] && al16(p->U[i]) && al16(p->SV[i]),
                "U, cluster_of and SV (16-byte aligned) are needed with a rank");
    GLQ_CHECK(p->u_rows[i] >= 0 && p->u_rows[i] < (1ll << 24), "u_rows out of range (proj %d)", i);
    if (SI > 0)
      GLQ_CHECK(p->shared_codes[i] && p->shared_scales[i] && p->shared_zeros[i] &&
                    al16(p->shared_codes[i]),
                "null or misaligned shared-expert weights (proj %d)", i);
  }
  for (int i = 0; i < 2; ++i) {
    GLQ_CHECK((p->signs[i] != nullptr) != (p->Pi[i] != nullptr),
              "one rotation, signs or Pi, is needed for %s", i ? "down" : "gate and up");
    const int64_t d = i ? I : H;
    GLQ_CHECK(p->Pi[i] == nullptr || (al16(p->Pi[i]) && d <= 32768),
              "Pi must be 16-byte aligned, its width <= 32768 (got %lld)", (long long)d);
    GLQ_CHECK(p->signs[i] == nullptr || ((d & (d - 1)) == 0 && d <= 32768),
              "the Hadamard transform takes a power of two <= 32768 (got %lld)", (long long)d);
  }
  return GLQ_OK;
}

// out (rows, d) = fp16(x Pi^T) in the 4-bit decode order.
static int tp_rotate(const __half* x, int64_t rows, int64_t d, const void* Pi, __half* out,
                     hipStream_t s) {
  PfArgs g = {};
  g.xp = x;
  g.codes[0] = (const uint32_t*)Pi;
  g.y = out;
  g.y_ld = d;
  g.out_bits = 4;
  g.M = (int)rows; g.K = (int)d; g.N = (int)d; g.G = (int)(d / 128);
  g.ntn = (int)((d + 127) / 128);
  g.max_tiles = (int)((rows + 63) / 64);
  return pt_launch_k<kPtHalf, 2, 2, 1, kPfDense, false, false, false>(g, s);
}
}  // namespace glq

extern "C" int64_t glq_turbo_moe_prefill_workspace_bytes(const glq_turbo_prefill_params* p) {
  using namespace glq;
  clear_error();
  return tp_check(p) == GLQ_OK ? tp_plan(p).total : -1;
}

extern "C" int glq_turbo_moe_prefill(const glq_turbo_prefill_params* p, void* workspace,
                                     int64_t workspace_bytes, void* stream) {
  using namespace glq;
  clear_error();
  int rc = tp_check(p);
  if (rc) return rc;
  const int64_t T = p->tokens, H = p->hidden, E = p->experts, I = p->inter, k = p->top_k;
  const int64_t SI = p->shared_inter, Pn = T * k, r = p->rank;
  const TpPlan P = tp_plan(p);
  GLQ_CHECK(workspace != nullptr && workspace_bytes >= P.total && ((uintptr_t)workspace & 255) == 0,
            "a 256-byte aligned workspace of %lld bytes is needed (got %lld)", (long long)P.total,
            (long long)workspace_bytes);
  hipStream_t s = (hipStream_t)stream;
  char* w = (char*)workspace;
  auto hp = [&](int64_t off) { return (__half*)(w + off); };
  PfMoe a = {};
  a.T = (int)T; a.H = (int)H; a.E = (int)E; a.I = (int)I; a.topk = (int)k;
  a.norm = p->norm_topk_prob ? 1 : 0;
  a.SI = (int)SI; a.bits = 4; a.sbits = SI > 0 ? p->shared_bits : 4;
  a.tm = P.tm; a.max_tiles = P.max_tiles;
  a.h = (const __half*)p->h;
  a.router_w = (const __half*)p->router_w;
  a.sgw = (const __half*)p->shared_gate_w;
  a.logits_out = (__half*)p->router_logits;
  a.xps = SI > 0 ? hp(P.off_xps) : nullptr;
  a.sel = (int32_t*)(w + P.off_sel);
  a.wts = hp(P.off_wts);
  a.sg = hp(P.off_sg);
  a.pos = (int32_t*)(w + P.off_pos);
  a.stok = (int32_t*)(w + P.off_stok);
  a.tiles = (int32_t*)(w + P.off_tiles);
  a.ntiles = a.tiles + 3 * P.max_tiles;
  a.lrcnt = (unsigned*)(w + P.off_lrcnt);
  a.n_lrcnt = pf_lrcnt(P.max_tiles, P.tm);
  a.yks = P.yks;
  a.ybuf = (const float*)(w + P.off_y);
  a.sy = SI > 0 ? (const float*)(w + P.off_sy) : nullptr;
  a.syh = (const __half*)p->shared_y;
  a.res = (const __half*)p->residual;
  a.out = (__half*)p->out;
  // 1. gate/up's input: the transform of h (put in decode order by the routing
  // launch), or h Pi^T
  if (p->signs[0]) {
    rc = glq_rht(p->h, 0, T, H, p->signs[0], 0, hp(P.off_xr), 0, stream);
    a.xsrc = hp(P.off_xr);
    a.xp = hp(P.off_xp);
  } else {
    rc = tp_rotate(a.h, T, H, p->Pi[0], hp(P.off_xp), s);
  }
  if (rc) return rc;
  // 2-3. routing and dispatch
  rc = pf_route_launch(a, s);
  if (rc) return rc;
  PfShared sh;
  const PfShared* shared = nullptr;
  if (SI > 0) {
    sh = pf_shared(T, H, SI, p->shared_bits, P.stm, true, a.xps, p->shared_codes,
                   p->shared_scales, p->shared_zeros, hp(P.off_sinter),
                   (float*)(w + P.off_sy));
    shared = &sh;
    a.sks = sh.down.ks;
  }
  // 4. a = x U for gate and up per pair, 5. gate/up + SwiGLU -> inter
  auto lowrank = [&](const __half* x, const int32_t* arow, int m0, int nmat, int64_t K, int ks,
                     int kps, __half* out) {
    PfLowrank L = {};
    L.x = x;
    L.arow = arow;
    L.nmat = nmat;
    for (int m = 0; m < nmat; ++m) {
      L.U[m] = (const __half*)p->U[m0 + m];
      L.cluster[m] = p->cluster_of[m0 + m];
      L.urows[m] = (int)p->u_rows[m0 + m];
    }
    L.u_cs = K * r;
    L.tiles = a.tiles;
    L.ntiles = a.ntiles;
    L.tile_rows = P.tm;
    L.rows_total = (int)Pn;
    L.K = (int)K;
    L.rank = (int)r;
    L.ks = ks;
    L.kps = kps;
    L.part = (float*)(w + P.off_lp);
    L.cnt = a.lrcnt;
    L.a_out = out;
    return pf_lowrank_launch(L, P.max_tiles * ((P.tm + kLrRows - 1) / kLrRows), s);
  };
  if (r > 0) {
    rc = lowrank(a.h, a.stok, 0, 2, H, P.ks_gu, P.kps_gu, hp(P.off_agu));
    if (rc) return rc;
  }
  __half* inter = hp(P.off_inter);
  {
    PfArgs g = {};
    g.xp = hp(P.off_xp);
    g.arow = a.stok;
    for (int m = 0; m < 2; ++m) {
      g.codes[m] = (const uint32_t*)p->codes[m];
      g.norms[m] = p->norms[m];
      g.cent[m] = p->centroids[m];
      g.sv[m] = r > 0 ? (const __half*)p->SV[m] : nullptr;
    }
    g.kw = (int)(H / 16);
    g.codes_es = I * g.kw;
    g.n_es = I;
    g.a = r > 0 ? hp(P.off_agu) : nullptr;
    g.a_ld = (int)(2 * r);
    g.sv_es = I * r;
    g.y = inter;
    g.y_ld = I;
    g.tiles = a.tiles;
    g.ntiles = a.ntiles;
    g.M = (int)Pn; g.K = (int)H; g.N = (int)I; g.G = (int)(H / 128);
    g.rank = (int)r;
    g.ntn = pt_tiles_n(I, kPfGateUp, P.tm);
    g.max_tiles = P.max_tiles;
    rc = pf_routed_launch<kPtTurbo, kPfGateUp>(g, P.tm, shared, s);
    if (rc) return rc;
  }
  // 6. a = inter U_down per pair, 7. the down's input rotated, in decode order
  if (r > 0) {
    rc = lowrank(inter, nullptr, 2, 1, I, P.ks_d, P.kps_d, hp(P.off_ad));
    if (rc) return rc;
  }
  if (p->signs[1]) {
    rc = glq_rht(inter, 0, Pn, I, p->signs[1], 0, hp(P.off_tmp), 0, stream);
    if (rc) return rc;
    const int64_t blocks = Pn * I / 16;
    pf_permute_kernel<<<dim3((unsigned)((blocks + 511) / 512)), dim3(256), 0, s>>>(
        hp(P.off_tmp), blocks, hp(P.off_xd));
    GLQ_LAUNCH_CHECK("pf_permute_kernel");
  } else {
    rc = tp_rotate(inter, Pn, I, p->Pi[1], hp(P.off_xd), s);
    if (rc) return rc;
  }
  // 8. down -> y per sorted row (fp32)
  {
    PfArgs g = {};
    g.xp = hp(P.off_xd);
    g.codes[0] = (const uint32_t*)p->codes[2];
    g.norms[0] = p->norms[2];
    g.cent[0] = p->centroids[2];
    g.sv[0] = r > 0 ? (const __half*)p->SV[2] : nullptr;
    g.kw = (int)(I / 16);
    g.codes_es = H * g.kw;
    g.n_es = H;
    g.a = r > 0 ? hp(P.off_ad) : nullptr;
    g.a_ld = (int)r;
    g.sv_es = H * r;
    g.yf = (float*)(w + P.off_y);
    g.yf_ld = H;
    g.tiles = a.tiles;
    g.ntiles = a.ntiles;
    g.M = (int)Pn; g.K = (int)I; g.N = (int)H; g.G = (int)(I / 128);
    g.rank = (int)r;
    g.ntn = pt_tiles_n(H, kPfDown, P.tm);
    g.ks = P.yks; g.gps = P.ygps;
    g.yf_ss = Pn * H;
    g.max_tiles = P.max_tiles;
    rc = pf_routed_launch<kPtTurbo, kPfDown>(g, P.tm, shared, s);
    if (rc) return rc;
  }
  // 9. shared expert (2-bit or larger tiles), 10. combine
  rc = pf_shared_launch(shared, P.tm, s);
  if (rc) return rc;
  pf_moe_combine_kernel<<<dim3((unsigned)((T * H / 4 + 255) / 256)), dim3(256), 0, s>>>(a);
  GLQ_LAUNCH_CHECK("pf_moe_combine_kernel");
  return GLQ_OK;
}
