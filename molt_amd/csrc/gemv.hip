// Skinny-M (M <= 16) NF4 GEMV with the rank-r LoRA add-on (gfx950), HBM-bound.
//
// Y[m, n] = sum_b scale(n, b) * sum_{k in block b} X[m, k] * code[W(n, k)]
//           + sum_j T[m, j] * bf16(s * B[n, j])
//
// v_mfma_f32_16x16x32_bf16 with X as the 16-row operand (rows >= M repeat
// row 0 and are never stored) and the NF4 codes as the 16-column operand.
// Lane group g = lane/16 owns the contiguous 16 elements [64b + 16g, +16) of
// block b (8 packed bytes, one 8-byte load per row), split over two 32-deep
// MFMAs, so each MFMA pair sums exactly one block and the block scale is
// applied once to its 16x16 result instead of to every weight.
//
// A workgroup (8 waves) owns 16 rows of W and all of K; its waves take
// contiguous slices of K, keep a whole chunk of blocks in flight (8 blocks
// when the u8 codes of 4 blocks can be read as one 4-byte load and share an
// absmax2 entry, else 4), and are summed in wave order through LDS, so no
// cross-workgroup reduction (and no device-scope fence) is needed. Codes come
// from an LDS table of bf16 code pairs indexed by the packed byte, replicated
// 32 times with the copy chosen by lane % 32, so the data-dependent lookups of
// a half-wave hit 32 distinct banks. The LoRA term is one more MFMA step per
// 32 ranks; its B rows are copied into LDS by direct global->LDS loads and T
// is held in registers, both issued with the first weight chunk.
#include <algorithm>
#include <mutex>

#include "common.h"

#include <stdlib.h>

namespace molt {
namespace {

constexpr int GV_WAVES = 8;
constexpr int GV_NT = 64 * GV_WAVES;
constexpr int GV_TILES = 1;              // 16-row MFMA tiles per wave
constexpr int GV_ROWS = 16 * GV_TILES;   // weight rows per workgroup
// Blocks per wave chunk (all loads of a chunk are in flight together).
template <bool Q4> constexpr int gv_u() { return Q4 ? 8 : 4; }
constexpr int GV_RMAX = 128;             // largest LoRA rank
constexpr int GV_TABW = 32;              // table copies (one per lane of a half-wave)
constexpr int GV_LT = 16 * GV_RMAX / GV_NT;   // T elements per thread

typedef __bf16 bf16x8v __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(1))) const void* gptr_t;
typedef __attribute__((address_space(3))) void* lptr_t;

struct GemvParams {
  const uint16_t* x; int64_t ldx; int M;
  const uint8_t* packed; int64_t N; int K;
  const float* scales;                                   // resolved, or null when nested
  const uint8_t* q; const float* absmax2; const float* code2; float offset; int dq_shift;
  const float* code; int order;
  const uint16_t* t; int64_t ldt; const float* lb; int r; float s;
  uint16_t* y; int64_t ldy;
};

// One chunk of gv_u<Q4>() blocks. Q4 (nested statistics, 4-aligned blocks): the
// u8 codes of a row's four blocks are one 4-byte load and share one absmax2
// entry; otherwise one code (or resolved scale) load per block.
template <bool Q4>
struct GvChunk {
  static constexpr int U = gv_u<Q4>();
  u32x2_t w[U][GV_TILES];
  u32x4_t xa[U], xb[U];
  uint32_t q[Q4 ? U / 4 : U][GV_TILES];
  float s[Q4 ? U / 4 : U][GV_TILES];
};

// Loads of one chunk. Every address is clamped into its tensor (past-the-end
// blocks repeat the last one and are not consumed; rows past N or M feed only
// outputs that are never stored), so no load is predicated. Offsets are 32-bit
// (a weight holds < 2^31 bytes and blocks), added to the uniform base pointers.
template <bool Q4>
MOLT_DEV void gv_load(GvChunk<Q4>& c, const GemvParams& p, const uint32_t (&wofs)[GV_TILES],
                      const uint32_t (&blk0)[GV_TILES], uint32_t xofs, int b, int b1) {
#pragma unroll
  for (int u = 0; u < gv_u<Q4>(); ++u) {
    const uint32_t bb = (uint32_t)(b + u < b1 ? b + u : b1 - 1);
    c.xa[u] = *reinterpret_cast<const u32x4_t*>(p.x + (xofs + 64u * bb));
    c.xb[u] = *reinterpret_cast<const u32x4_t*>(p.x + (xofs + 64u * bb + 8u));
#pragma unroll
    for (int t = 0; t < GV_TILES; ++t) {
      c.w[u][t] = *reinterpret_cast<const u32x2_t*>(p.packed + (wofs[t] + 32u * bb));
      const uint32_t blk = blk0[t] + bb;
      if (Q4) {
        if (u % 4 == 0) {
          // Whole 4-block units: a unit past the end repeats the last one
          // (b1 - 4 is unit-aligned), so the 4-byte code load stays inside
          // the row's codes.
          const uint32_t qblk = blk0[t] + (uint32_t)(b + u < b1 ? b + u : b1 - 4);
          c.q[u / 4][t] = *reinterpret_cast<const uint32_t*>(p.q + qblk);
          c.s[u / 4][t] = p.absmax2[qblk >> p.dq_shift];
        }
      } else if (p.scales) {
        c.s[u][t] = p.scales[blk];
      } else {
        c.q[u][t] = p.q[blk];
        c.s[u][t] = p.absmax2[blk >> p.dq_shift];
      }
    }
  }
}

MOLT_DEV float gv_scale(const GemvParams& p, const float* code2s, uint32_t q, float s) {
#pragma clang fp contract(off)
  if (p.scales) return s;
  const float prod = code2s[q & 0xffu] * s;
  return prod + p.offset;
}

struct GvSmem {
  union {
    uint32_t tab[256 * GV_TABW];                          // bf16 code pair of byte b at [b * 32 + copy]
    f32x4_t red[GV_WAVES - 1][GV_TILES][64];
  };
  float code2s[256];
  float lb[GV_ROWS * GV_RMAX];                            // raw fp32 LoRA B rows n0.., row stride r
  uint16_t lt[16 * GV_RMAX];                              // T rows 0..15, row stride r
};

// With gridDim.y > 1 (narrow outputs: few 16-row groups) K is split over
// gridDim.y workgroups per group, contiguous ranges of whole units; each writes
// its fp32 partial to `part` (slice-major) and gm_reduce_kernel sums them in
// slice order. The LoRA term belongs to slice 0.
template <bool Q4>
__global__ __launch_bounds__(GV_NT) __attribute__((amdgpu_waves_per_eu(4)))
void nf4_gemv_kernel(const GemvParams p, float* part) {
  __shared__ GvSmem sm;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t n0 = (int64_t)blockIdx.x * GV_ROWS;
  const int col = lane & 15, g = lane >> 4;
  const int KB = p.K >> 6;
  // Waves take contiguous slices of whole units (4 blocks under Q4) of this
  // workgroup's K range.
  constexpr int unit = Q4 ? 4 : 1;
  const int all_units = KB / unit, ns = (int)gridDim.y, sl = (int)blockIdx.y;
  const int u0 = sl * all_units / ns, units = (sl + 1) * all_units / ns - u0;
  const int b0 = unit * (u0 + wave * units / GV_WAVES), b1 = unit * (u0 + (wave + 1) * units / GV_WAVES);
  const int mc = col < p.M ? col : p.M - 1;
  const uint32_t xofs = (uint32_t)(mc * p.ldx + 16 * g);
  uint32_t wofs[GV_TILES], blk0[GV_TILES];
#pragma unroll
  for (int t = 0; t < GV_TILES; ++t) {
    const int64_t n = n0 + 16 * t + col;
    const int64_t nc = n < p.N ? n : p.N - 1;
    wofs[t] = (uint32_t)(nc * (p.K >> 1) + 8 * g);
    blk0[t] = (uint32_t)(nc * KB);
  }

  // Issue order: the codebooks (tiny, L2-resident), the first weight chunk,
  // then the LoRA operands straight into LDS. Nothing waits until all of
  // them are in flight.
  // The codebook is read through the constant address space (scalar loads
  // into SGPRs: one copy per wave instead of per lane).
  typedef __attribute__((address_space(4))) const f32x4_t* cptr_t;
  const cptr_t cbp = (cptr_t)p.code;
  const f32x4_t cb0 = cbp[0], cb1 = cbp[1], cb2 = cbp[2], cb3 = cbp[3];
  const float c2 = (p.code2 ? p.code2 : p.code)[p.code2 ? (tid & 255) : 0];
  GvChunk<Q4> c;
  if (b0 < b1) gv_load<Q4>(c, p, wofs, blk0, xofs, b0, b1);
  const bool lora = p.r > 0 && sl == 0;
  if (lora) {
    // B rows n0 .. n0+63 are contiguous (row stride r): 4-byte copies.
    const int nb = GV_ROWS * p.r;
    const int64_t bmax = p.N * p.r - 1;
    for (int base = wave * 64; base < nb; base += GV_NT) {
      int64_t e = n0 * p.r + base + lane;
      e = e < bmax ? e : bmax;
      __builtin_amdgcn_global_load_lds((gptr_t)(p.lb + e), (lptr_t)(sm.lb + base), 4, 0, 0);
    }
  }
  // T rows 0 .. 15 (rows >= M repeat row 0) into registers; stored below.
  uint32_t traw[GV_LT];
#pragma unroll
  for (int k = 0; k < GV_LT; ++k) {
    traw[k] = 0;
    if (lora) {
      int i = tid + k * GV_NT;
      i = i < 16 * p.r ? i : 0;
      const int m = i / p.r, j = i - m * p.r;
      traw[k] = p.t[(int64_t)(m < p.M ? m : 0) * p.ldt + j];
    }
  }

  // Replicated code-pair table: this thread writes byte values b with low
  // nibble tid / 32 (copy tid % 32) for every high nibble.
  {
    const float cv[16] = {cb0[0], cb0[1], cb0[2], cb0[3], cb1[0], cb1[1], cb1[2], cb1[3],
                          cb2[0], cb2[1], cb2[2], cb2[3], cb3[0], cb3[1], cb3[2], cb3[3]};
    const int lo = tid >> 5, copy = tid & 31;
    float clo = cv[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) clo = lo == i ? cv[i] : clo;
#pragma unroll
    for (int hi = 0; hi < 16; ++hi) {
      const float first = p.order ? cv[hi] : clo, second = p.order ? clo : cv[hi];
      sm.tab[(hi * 16 + lo) * GV_TABW + copy] = pack_bf16x2(first, second);
    }
    if (tid < 256) sm.code2s[tid] = c2;
  }
  if (lora) {
#pragma unroll
    for (int k = 0; k < GV_LT; ++k) {
      const int i = tid + k * GV_NT;
      if (i < 16 * p.r) sm.lt[i] = (uint16_t)traw[k];
    }
  }
  __syncthreads();

  const uint32_t* tab = sm.tab + (lane & 31);
  f32x4_t acc[GV_TILES];
#pragma unroll
  for (int t = 0; t < GV_TILES; ++t) acc[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int b = b0; b < b1;) {
#pragma unroll
    for (int u = 0; u < gv_u<Q4>(); ++u) {
      if (b + u >= b1) break;
      const bf16x8v xa = __builtin_bit_cast(bf16x8v, c.xa[u]);
      const bf16x8v xb = __builtin_bit_cast(bf16x8v, c.xb[u]);
#pragma unroll
      for (int t = 0; t < GV_TILES; ++t) {
        u32x4_t w0, w1;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          w0[j] = tab[((c.w[u][t][0] >> (8 * j)) & 0xffu) * GV_TABW];
          w1[j] = tab[((c.w[u][t][1] >> (8 * j)) & 0xffu) * GV_TABW];
        }
        f32x4_t tmp = {0.f, 0.f, 0.f, 0.f};
        tmp = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa, __builtin_bit_cast(bf16x8v, w0), tmp, 0, 0, 0);
        tmp = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xb, __builtin_bit_cast(bf16x8v, w1), tmp, 0, 0, 0);
        const float sc = Q4 ? gv_scale(p, sm.code2s, c.q[u / 4][t] >> (8 * (u % 4)), c.s[u / 4][t])
                            : gv_scale(p, sm.code2s, c.q[u][t], c.s[u][t]);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[t][e] += sc * tmp[e];
      }
    }
    b += gv_u<Q4>();
    if (b < b1) gv_load<Q4>(c, p, wofs, blk0, xofs, b, b1);
  }

  __syncthreads();                       // the table area becomes the reduction area
  if (wave > 0) {
#pragma unroll
    for (int t = 0; t < GV_TILES; ++t) sm.red[wave - 1][t][lane] = acc[t];
  }
  __syncthreads();
  if (wave != 0) return;
#pragma unroll
  for (int w = 0; w < GV_WAVES - 1; ++w)
#pragma unroll
    for (int t = 0; t < GV_TILES; ++t) acc[t] += sm.red[w][t][lane];

  if (lora) {
    // acc += T . bf16(s B)^T, 32 ranks per MFMA step (ranks past r are zero).
    for (int j0 = 0; j0 < p.r; j0 += 32) {
      u32x4_t ta;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int j = j0 + 8 * g + 2 * e;
        const uint32_t lo = j < p.r ? sm.lt[col * p.r + j] : 0u;
        const uint32_t hi = j + 1 < p.r ? sm.lt[col * p.r + j + 1] : 0u;
        ta[e] = lo | (hi << 16);
      }
#pragma unroll
      for (int t = 0; t < GV_TILES; ++t) {
        const float* brow = sm.lb + (16 * t + col) * p.r;
        u32x4_t bw;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int j = j0 + 8 * g + 2 * e;
          const float lo = j < p.r ? round_bf16(p.s * brow[j]) : 0.0f;
          const float hi = j + 1 < p.r ? round_bf16(p.s * brow[j + 1]) : 0.0f;
          bw[e] = pack_bf16x2(lo, hi);
        }
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8v, ta),
                                                         __builtin_bit_cast(bf16x8v, bw), acc[t], 0, 0, 0);
      }
    }
  }

  // acc[t][e] is C[m][n] with m = 4 (lane / 16) + e, n = n0 + 16 t + lane % 16.
#pragma unroll
  for (int t = 0; t < GV_TILES; ++t) {
    const int64_t n = n0 + 16 * t + col;
    if (n >= p.N) continue;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int m = 4 * g + e;
      if (m >= p.M) continue;
      if (ns == 1) p.y[(int64_t)m * p.ldy + n] = bf16_bits(acc[t][e]);
      else part[((int64_t)sl * p.M + m) * p.N + n] = acc[t][e];
    }
  }
}


// ---------------------------------------------------------------------------
// Streaming dot-product variant for few tokens (decode; see dot_serves). Each wave walks rows of W
// in rounds: round j covers RW rows at j * (grid waves * RW) + (this wave's
// index) * RW, so every round of the grid reads a contiguous band of W. A
// lane reads 16 contiguous packed bytes (32 elements, half a block) of each
// 1 KB piece of a row, so each load instruction is 1 KB of one row. The loads
// of a round (weight pieces, block statistics, LoRA B entries) are issued two
// rounds ahead into three rotating register sets, so the dot-product work of
// round j overlaps the HBM stream of rounds j + 1 and j + 2. Codes come from
// the replicated LDS table of bf16 code pairs and meet X (staged once per
// workgroup in LDS) through v_dot2_f32_bf16; the block scale multiplies each
// lane's half-block sum, lane j < r adds T[j] bf16(s B[n, j]), and the 64
// lanes of a row are summed by DPP row reductions and scalar reads. MX rows of X (the tokens,
// M <= MX; rows past M repeat row M - 1 and are not stored) share each code
// lookup, one dot2 per token. K is any multiple of 64 up to 7 x 2048: the last
// piece of a row may be partial (its lanes past the row end are masked).
constexpr int GD_WAVES = 8;
constexpr int GD_NT = 64 * GD_WAVES;
constexpr int GD_XPAD = 8;                // bf16 elements of X row padding

// Code-pair table of the dot kernel: entry (byte b, copy c) at b * TS + c.
// With TS = 64 (256 bytes per entry, copies in the first 128) a lane's
// lookup address is one v_perm_b32 of the packed dword: the byte lands in
// bits 8-15 beside the lane's copy offset (lane % 32) * 4 in bits 0-7, where
// the 32-dword stride takes a bit-field extract and a shift-add per byte.
// It doubles the table's footprint (64 KB), so it is used where the LDS
// allows (see gd_perm).
template <int TS>
struct GdSmem {
  uint32_t tab[256 * TS];
  float code2s[256];
};
template <int IPR, int MX>
constexpr bool gd_perm() { return IPR == 2 ? MX == 1 : MX <= 2; }

typedef __bf16 bf16x2v __attribute__((ext_vector_type(2)));

template <int RW, int IPR>
struct GdRound {
  u32x4_t w[RW * IPR];
  uint32_t q[RW * IPR];
  float s[RW * IPR];
  float lb[RW][2];
};

// Pieces of a row that may be partial or idle: the last one, and the one before
// it where the pieces a row needs were rounded up to an instantiated IPR (4 runs
// as 5, 6 as 7).
template <int IPR, bool FULL>
constexpr int gd_tails() { return FULL ? 0 : IPR >= 5 ? 2 : 1; }

// Loads of one round (rows n0 .. n0 + RW - 1, clamped to the matrix). Every
// load is unconditional (statistics layout and LoRA presence are template
// parameters, out-of-range indices are clamped and their values masked), so
// each round issues the same fixed number of loads and the compiler's vmcnt
// wait before a round's arithmetic counts exactly the two later rounds as
// still in flight; a load under a run-time branch made it wait for those too.
// Rows past the matrix read row `fallback` instead (the wave's own first row,
// already on its way to the cache; one shared row would be a hot spot).
template <int RW, int IPR, bool NESTED, bool LORA, bool FULL>
MOLT_DEV void gd_load(GdRound<RW, IPR>& R, const GemvParams& p, int64_t n0, int lane, int KB, int64_t fallback) {
#pragma unroll
  for (int r = 0; r < RW; ++r) {
    const int64_t n = n0 + r < p.N ? n0 + r : fallback;
#pragma unroll
    for (int i = 0; i < IPR; ++i) {
      const int j = r * IPR + i;
      // a tail piece may end inside the row: its lanes past the end re-read
      // the row's last 16 bytes and block (their products are dropped)
      constexpr int whole = IPR - gd_tails<IPR, FULL>();
      const int wo = i < whole ? 1024 * i + 16 * lane : min(1024 * i + 16 * lane, (p.K >> 1) - 16);
      const int bo = i < whole ? 32 * i + (lane >> 1) : min(32 * i + (lane >> 1), KB - 1);
      R.w[j] = *reinterpret_cast<const u32x4_t*>(p.packed + (uint32_t)(n * (p.K >> 1) + wo));
      const uint32_t blk = (uint32_t)(n * KB + bo);
      if constexpr (NESTED) {
        R.q[j] = p.q[blk];
        R.s[j] = p.absmax2[blk >> p.dq_shift];
      } else {
        R.q[j] = 0;
        R.s[j] = p.scales[blk];
      }
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int jr = lane + 64 * q;
      if constexpr (LORA) {
        const float v = p.lb[n * p.r + (jr < p.r ? jr : p.r - 1)];
        R.lb[r][q] = jr < p.r ? v : 0.0f;
      } else {
        R.lb[r][q] = 0.0f;
      }
    }
  }
}

// Sum over the 64 lanes of a wave with no LDS traffic (a shuffle becomes an
// LDS permute whose wait also drains the round's outstanding table lookups):
// DPP within each row of 16 lanes (swap neighbours, swap pairs, half-row
// mirror, row mirror), then the four row sums read into scalars and added in
// row order. The result is wave-uniform.
MOLT_DEV float gd_wave_sum(float v) {
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, false));
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xF, 0xF, false));
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xF, 0xF, false));
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x140, 0xF, 0xF, false));
  const int iv = __builtin_bit_cast(int, v);
  return (__builtin_bit_cast(float, __builtin_amdgcn_readlane(iv, 0)) +
          __builtin_bit_cast(float, __builtin_amdgcn_readlane(iv, 16))) +
         (__builtin_bit_cast(float, __builtin_amdgcn_readlane(iv, 32)) +
          __builtin_bit_cast(float, __builtin_amdgcn_readlane(iv, 48)));
}

// Dot products of one round; returns the value lane r * MX + m stores (row r
// of token m, see gd_store). X row m sits at
// xs + m * xstride (elements); with XREG (one token) the lane's X chunks are
// xg[4 i + h] in registers instead.
template <int RW, int IPR, int MX, bool XREG, bool PERM, bool FULL>
MOLT_DEV float gd_compute(const GdRound<RW, IPR>& R, const GemvParams& p, const uint32_t* tab, const uint16_t* xs,
                         int xstride, const u32x4_t* xg, const float* code2s, const float (&lt)[MX][2], int64_t n0,
                         int lane) {
  const uint32_t lb = (uint32_t)(lane & 31) * 4;     // PERM: byte offset of the lane's copy
  float acc[RW][MX];
#pragma unroll
  for (int r = 0; r < RW; ++r)
#pragma unroll
    for (int m = 0; m < MX; ++m) acc[r][m] = 0.0f;
#pragma unroll
  for (int i = 0; i < IPR; ++i) {                                      // piece i of every row: X read once
    float bs[RW][MX];
#pragma unroll
    for (int r = 0; r < RW; ++r)
#pragma unroll
      for (int m = 0; m < MX; ++m) bs[r][m] = 0.0f;
#pragma unroll
    for (int h = 0; h < 4; ++h) {                                      // 4 bytes per dword, 8 elements
      u32x4_t xv[MX];
#pragma unroll
      for (int m = 0; m < MX; ++m)
        xv[m] = XREG ? xg[4 * i + h] : *reinterpret_cast<const u32x4_t*>(xs + m * xstride + 8 * (256 * i + 64 * h + lane));
#pragma unroll
      for (int b = 0; b < 4; ++b) {
#pragma unroll
        for (int r = 0; r < RW; ++r) {
          uint32_t pair;
          if constexpr (PERM) {
            // bits 15:8 = byte b of the dword, bits 7:0 = lb: selectors 4 + b (S0), 0 (S1), 12 (zero)
            const uint32_t off = __builtin_amdgcn_perm(R.w[r * IPR + i][h], lb, 0x0C0C0400u | ((uint32_t)b << 8));
            pair = *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(tab) + off);
          } else {
            pair = tab[((R.w[r * IPR + i][h] >> (8 * b)) & 0xffu) * GV_TABW];
          }
#pragma unroll
          for (int m = 0; m < MX; ++m) {
            // copy the element out first: __builtin_bit_cast of a vector-element
            // lvalue reads element 0 with this compiler
            const uint32_t xw = xv[m][b];
            bs[r][m] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2v, pair),
                                                       __builtin_bit_cast(bf16x2v, xw), bs[r][m], false);
          }
        }
      }
    }
    // lanes past the end of a row in a tail piece contribute nothing
    const bool live = i < IPR - gd_tails<IPR, FULL>() || 1024 * i + 16 * lane < (p.K >> 1);
#pragma unroll
    for (int r = 0; r < RW; ++r) {
      const float sc = gv_scale(p, code2s, R.q[r * IPR + i], R.s[r * IPR + i]);
#pragma unroll
      for (int m = 0; m < MX; ++m) {
        acc[r][m] += live ? sc * bs[r][m] : 0.0f;
        asm volatile("" : "+v"(acc[r][m]));                           // keeps each piece's lookups short-lived
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  // LoRA partials join the row sums; sum over the wave (gd_wave_sum); lane
  // r * MX + m stores row r of token m
#pragma unroll
  for (int r = 0; r < RW; ++r) {
    const float b0 = round_bf16(p.s * R.lb[r][0]), b1 = round_bf16(p.s * R.lb[r][1]);
#pragma unroll
    for (int m = 0; m < MX; ++m) acc[r][m] = gd_wave_sum(acc[r][m] + (lt[m][0] * b0 + lt[m][1] * b1));
  }
  float v = acc[0][0];
#pragma unroll
  for (int r = 0; r < RW; ++r)
#pragma unroll
    for (int m = 0; m < MX; ++m) v = lane == r * MX + m ? acc[r][m] : v;
  return v;
}

// Store of one round's results: lane r * MX + m holds row n0 + r of token m.
template <int RW, int MX>
MOLT_DEV void gd_store(const GemvParams& p, float v, int64_t n0, int lane) {
  if (lane < RW * MX) {
    const int rr = lane / MX, m = lane % MX;
    const int64_t n = n0 + rr;
    if (n < p.N && m < p.M) p.y[(int64_t)m * p.ldy + n] = bf16_bits(v);
  }
}

// At K = 4096 with up to two X rows the kernel is held to 128 registers, so two
// workgroups fit on a CU.
//
// MAXR > 0: at most MAXR rounds per wave, all issued up front in straight-line
// code (rounds past `rounds` load the clamped last row and are not computed),
// each round's arithmetic starting as soon as its own loads have landed, and
// every store after the last round: with no branch between a load and its use
// the compiler's waits count exactly the later loads still in flight. MAXR = 0:
// any number of rounds, loaded two ahead in three rotating register sets.
template <int RW, int IPR, int MX, bool NESTED, bool LORA, int MAXR, bool FULL>
__global__ __launch_bounds__(GD_NT) __attribute__((amdgpu_waves_per_eu(IPR <= 2 && MX <= 2 ? 4 : 1)))
void nf4_gemv_dot_kernel(const GemvParams p, int rounds) {
  constexpr bool PERM = gd_perm<IPR, MX>();
  constexpr int TS = PERM ? 64 : GV_TABW;
  __shared__ GdSmem<TS> sm;
  extern __shared__ __attribute__((aligned(16))) uint16_t gd_xs[];      // X, MX rows of K + GD_XPAD elements
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t stride = (int64_t)gridDim.x * GD_WAVES * RW;          // rows per round of the grid
  const int64_t nb = ((int64_t)blockIdx.x * GD_WAVES + wave) * RW;    // first row of round 0
  const int KB = p.K >> 6;

  typedef __attribute__((address_space(4))) const f32x4_t* cptr_t;
  const cptr_t cbp = (cptr_t)p.code;
  const f32x4_t cb0 = cbp[0], cb1 = cbp[1], cb2 = cbp[2], cb3 = cbp[3];

  // X first (16-byte chunks into registers), so that the wait before its LDS
  // stores, and the barrier after them, do not wait for the weight stream.
  // One token at K = 4096: the lane's 64 elements of X (16-byte chunks
  // 256 i + 4 lane + h, the elements its weight bytes multiply) stay in
  // registers, read straight from memory; otherwise X is staged in LDS. (At
  // K = 14336 with two rounds per wave the 112 registers fit, but the decode
  // measured slower: 11.3 -> 12.5 us at 4096 x 14336.)
  constexpr bool XREG = IPR == 2 && MX == 1;
  constexpr int XCH = IPR * 256, XIT = XREG ? 0 : (MX * XCH + GD_NT - 1) / GD_NT;   // 16-byte chunks of X
  // X rows in LDS take whole pieces (IPR x 2048 elements); chunks past the end
  // of a row (a partial last piece) re-read its last chunk, whose products
  // the compute drops
  const int xstride = IPR * 2048 + GD_XPAD;
  const int xlast = (p.K >> 3) - 1;                                   // last 16-byte chunk of a row
  u32x4_t xr[XIT > 0 ? XIT : 1];
  u32x4_t xg[XREG ? 4 * IPR : 1];
  if constexpr (XREG) {
#pragma unroll
    for (int c = 0; c < 4 * IPR; ++c)
      xg[c] = *reinterpret_cast<const u32x4_t*>(p.x + 8 * min(256 * (c >> 2) + 4 * lane + (c & 3), xlast));
  }
#pragma unroll
  for (int it = 0; it < XIT; ++it) {
    const int c = tid + it * GD_NT < MX * XCH ? tid + it * GD_NT : MX * XCH - 1;
    const int m = c / XCH < p.M ? c / XCH : p.M - 1;
    xr[it] = *reinterpret_cast<const u32x4_t*>(p.x + m * p.ldx + 8 * min(c % XCH, xlast));
  }
  // unconditional loads here too (clamped, then masked): see gd_load
  float c2 = 0.0f;
  if constexpr (NESTED) c2 = p.code2[tid & 255];
  float lt[MX][2];
#pragma unroll
  for (int m = 0; m < MX; ++m) {
    const int mm = m < p.M ? m : p.M - 1;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int jr = lane + 64 * q;
      lt[m][q] = 0.0f;
      if constexpr (LORA) {
        const float v = bf16_to_f32(p.t[mm * p.ldt + (jr < p.r ? jr : p.r - 1)]);
        lt[m][q] = jr < p.r ? v : 0.0f;
      }
    }
  }

  // The small loads above (X, the nested code table, T) are issued before any
  // weight load and must stay there: a wait for one of them placed after the
  // weight loads would wait for the whole weight stream too.
  __builtin_amdgcn_sched_barrier(0);
  constexpr int NB = MAXR > 0 ? MAXR : 3;
  const int64_t nf = nb < p.N ? nb : p.N - 1;
  GdRound<RW, IPR> b[NB];
  gd_load<RW, IPR, NESTED, LORA, FULL>(b[0], p, nb, lane, KB, nf);
#pragma unroll
  for (int j = 1; j < (MAXR > 0 ? MAXR : 2); ++j) gd_load<RW, IPR, NESTED, LORA, FULL>(b[j], p, nb + j * stride, lane, KB, nf);

  // X in LDS by (piece, dword, lane): 16-byte chunk c = 256 i + 4 l + h (elements
  // 2048 i + 32 l + 8 h ..) sits at 256 i + 64 h + l, so the reads of a piece's
  // dword h by the 64 lanes are 1 KB contiguous (bank-conflict free).
#pragma unroll
  for (int it = 0; it < XIT; ++it) {
    const int c = tid + it * GD_NT;
    const int m = c / XCH, cc = c % XCH;
    if (c < MX * XCH)
      *reinterpret_cast<u32x4_t*>(gd_xs + m * xstride + 8 * ((cc & ~255) | ((cc & 3) << 6) | ((cc >> 2) & 63))) =
          xr[it];
  }
  {
    const float cv[16] = {cb0[0], cb0[1], cb0[2], cb0[3], cb1[0], cb1[1], cb1[2], cb1[3],
                          cb2[0], cb2[1], cb2[2], cb2[3], cb3[0], cb3[1], cb3[2], cb3[3]};
    static_assert(GV_TABW == 32 && GD_NT % 512 == 0 && GD_NT <= 8192, "table build covers 256 x 32 entries");
    constexpr int HS = GD_NT / 512;                                    // high nibbles per pass
    const int lo = (tid >> 5) & 15, copy = tid & 31, h0 = tid >> 9;
    float clo = cv[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) clo = lo == i ? cv[i] : clo;
#pragma unroll
    for (int k = 0; k < 16 / HS; ++k) {
      const int hi = h0 + HS * k;
      float chi = cv[0];
#pragma unroll
      for (int i = 1; i < 16; ++i) chi = hi == i ? cv[i] : chi;
      const float first = p.order ? chi : clo, second = p.order ? clo : chi;
      sm.tab[(hi * 16 + lo) * TS + copy] = pack_bf16x2(first, second);
    }
    sm.code2s[tid & 255] = c2;                       // every thread: no branch around the load
  }
  __syncthreads();

  const uint32_t* tab = PERM ? sm.tab : sm.tab + (lane & 31);
  if constexpr (MAXR > 0) {
    float out[MAXR];
#pragma unroll
    for (int j = 0; j < MAXR; ++j)
      out[j] = gd_compute<RW, IPR, MX, XREG, PERM, FULL>(b[j], p, tab, gd_xs, xstride, xg, sm.code2s, lt, nb + j * stride, lane);
#pragma unroll
    for (int j = 0; j < MAXR; ++j)
      if (j < rounds) gd_store<RW, MX>(p, out[j], nb + j * stride, lane);
  } else {
    // Rounds past the last one load the (clamped) last row again and are never
    // computed: unconditional loads keep the waits exact (see gd_load).
    for (int j = 0; j < rounds; j += 3) {
      gd_load<RW, IPR, NESTED, LORA, FULL>(b[2], p, nb + (j + 2) * stride, lane, KB, nf);
      gd_store<RW, MX>(p, gd_compute<RW, IPR, MX, XREG, PERM, FULL>(b[0], p, tab, gd_xs, xstride, xg, sm.code2s, lt,
                                                          nb + j * stride, lane), nb + j * stride, lane);
      if (j + 1 >= rounds) break;
      gd_load<RW, IPR, NESTED, LORA, FULL>(b[0], p, nb + (j + 3) * stride, lane, KB, nf);
      gd_store<RW, MX>(p, gd_compute<RW, IPR, MX, XREG, PERM, FULL>(b[1], p, tab, gd_xs, xstride, xg, sm.code2s, lt,
                                                          nb + (j + 1) * stride, lane), nb + (j + 1) * stride, lane);
      if (j + 2 >= rounds) break;
      gd_load<RW, IPR, NESTED, LORA, FULL>(b[1], p, nb + (j + 4) * stride, lane, KB, nf);
      gd_store<RW, MX>(p, gd_compute<RW, IPR, MX, XREG, PERM, FULL>(b[2], p, tab, gd_xs, xstride, xg, sm.code2s, lt,
                                                          nb + (j + 2) * stride, lane), nb + (j + 2) * stride, lane);
    }
  }
}

// ---------------------------------------------------------------------------
// Streaming MFMA kernel: batches of up to 16 tokens over any K of whole blocks.
//
// A workgroup of 16 waves (one per CU) walks 16-row groups of W in rounds. A
// group's K range (a slice of GL_BW x `wpg` blocks, slice blockIdx.y) is split
// over wpg waves, 4 blocks each, so a wave's X fragments are 32 registers that
// it loads once; a K too short for 16 waves runs `gpr` groups side by side.
//
// The packed bytes reach LDS by buffer-load DMA, each wave streaming its own 2
// KB per round into a ring of three slots that nobody else reads: no barrier,
// only the wave's own count of outstanding loads, and up to 96 KB in flight per
// CU without a register. (Loads into registers, two rounds ahead, held the
// kernel to two waves per SIMD, whose lookups, MFMAs and waits then ran in
// turn.) A load instruction takes whole 32-byte blocks of its rows in order;
// rows are rotated in LDS so that the 16 rows a fragment read touches lie on
// different banks.
//
// Per block: 8 packed bytes a lane, 8 code pairs from the replicated LDS table
// (one v_perm_b32 each for the address), two v_mfma_f32_16x16x32_bf16 with X as
// the 16-row operand, and the block's scale applied to its 16 x 16 sums in
// fp32. Lane group g holds the block's elements 16 g .. 16 g + 15. LoRA: rank
// chunk c of 32 is one more MFMA of the group's wave c (in slice 0). The waves'
// sums are added through LDS in wave order; with several slices (K over 4096)
// each writes fp32 partials that gm_reduce_kernel adds in slice order.
//
// A single round (4096^2) is a chain: launch, X, table, first bytes, lookups, sum;
// a further round of 8 MB takes 2.3 us (3.6 TB/s). us, replayed from a graph over
// rotating weights, rank 16: weights through registers (for K = 5120, 8960 and 896
// the one-group kernel above), weights through LDS, X through LDS as well:
//            4096^2          14336 x 4096       4096 x 14336       8960 x 1536       1536 x 8960        4864 x 896
//   M = 5    7.06 6.57 6.78  13.96 13.75 14.04  17.44 16.49 16.85  10.52 7.93 7.62   14.00 10.64 10.40  7.38 6.70 6.04
//   M = 8    7.79 7.13 6.82  14.33 14.28 14.31  18.28 17.28 17.03  11.16 8.34 7.72   15.24 11.18 10.53  7.79 7.35 6.07
//   M = 16   9.11 8.46 7.44  16.13 15.53 15.06  19.90 18.48 17.91  12.64 9.44 8.32   18.04 12.21 11.04  9.01 8.64 6.50
// Since then (groups by gl_plan, B by buffer loads), one run on a box whose large shapes are 6% slower: M = 5 6.6,
// 14.7, 16.4, 7.5, 10.5, 5.1; M = 8 6.6, 14.6, 16.6, 7.5, 10.6, 5.1; M = 16 7.1, 15.7, 17.4, 7.6, 11.1, 5.4.
// Ranks that are no multiple of 8 take B by the same two loads a round; one load and address per rank cost, M = 5:
// 14336 x 4096 at rank 4 / 5 / 12 21.8 / 21.2 / 22.2 -> 14.2 / 15.4 / 13.8, 8960 x 1600 16.9 / 16.0 / 17.6 -> 9.9 /
// 10.4 / 9.7 (weights through registers, ranks by fours: 14.2 / 16.1 / 13.7, 10.7 / 10.7 / 10.9).
constexpr int GL_WAVES = 16, GL_NT = 64 * GL_WAVES, GL_BW = 4;     // GL_BW: blocks of a wave
constexpr int GL_SLOT = 16 * GL_BW * 32;                 // bytes of one wave's slot
constexpr int GL_ROT = 1;                                // row >> GL_ROT: see gl_pos

// mode 0: resolved fp32 scales; 1: nested (dq_block >= 4), one u8 code per
// block; 2: nested, the codes of 4 blocks in one 4-byte load sharing one absmax2
// entry. LV: 0 no LoRA; 1 whole groups of four ranks (r % 4 == 0, T
// rows 8-byte aligned); 2 any rank.
template <int SM, int LV>
struct GlRound {
  static constexpr int NS = SM == 2 ? 1 : SM == 1 ? 2 : GL_BW, NQ = SM == 0 ? 0 : SM == 2 ? 1 : GL_BW;
  static constexpr int NL = LV == 0 ? 0 : 2;
  static constexpr int kLoads = GL_SLOT / 1024 + NS + NQ + NL;   // vector-memory operations of a round
  uint32_t q[SM == 0 ? 1 : NQ];
  float s[NS];
  float lb[8];
};

struct GlSmem {
  // Code-pair table at a 256-byte entry stride (see GdSmem), 32 copies in the
  // first 128 bytes; the other 128 bytes of entries 0 .. 127 hold the waves'
  // partial sums, those of 128 .. 135 the nested code table.
  uint32_t tab[256 * 64];
};
MOLT_DEV float* gl_red(GlSmem& sm, int wave, int lane) {
  return reinterpret_cast<float*>(sm.tab + (wave * 8 + (lane >> 3)) * 64 + 32 + (lane & 7) * 4);
}
MOLT_DEV float* gl_code2(GlSmem& sm, uint32_t q) {
  return reinterpret_cast<float*>(sm.tab + (128 + (q >> 5)) * 64 + 32 + (q & 31));
}

// Position of 16-byte piece c (two to a block) of row R in a slot: 8 pieces to
// a row, rotated by R / 2, so that one piece of 16 rows covers 256 bytes.
MOLT_DEV int gl_pos(int R, int c) { return R * (2 * GL_BW) + ((c + (R >> GL_ROT)) & (2 * GL_BW - 1)); }

// n * k as a product of its own: folded into a 64-bit multiply-add with a
// half-defined addend, it waited for whatever load the other half was free for.
MOLT_DEV uint32_t gl_mul(int n, int k) {
  uint32_t v = (uint32_t)n * (uint32_t)k;
  asm("" : "+v"(v));
  return v;
}

// Ranks that are no groups of four: byte offset in B of half h of a lane's 8 entries of row n (16 bytes, which need
// 4-byte alignment only). Kept inside B: a load that straddled its end might lose the entries before it; moved back, it
// holds them gl_b_shift further up.
MOLT_DEV uint32_t gl_b_at(const GemvParams& p, int n, int nr, int h) { return (gl_mul(n, p.r) + (uint32_t)(p.r - nr + 4 * h)) * 4u; }
MOLT_DEV uint32_t gl_b_offset(const GemvParams& p, int n, int nr, int h) {
  return min(gl_b_at(p, n, nr, h), ((uint32_t)p.N * (uint32_t)p.r - 4u) * 4u);
}
MOLT_DEV uint32_t gl_b_shift(const GemvParams& p, int n, int nr, int h) {
  return (gl_b_at(p, n, nr, h) - gl_b_offset(p, n, nr, h)) / 4u;
}

template <int SM, int LV>
MOLT_DEV void gl_load(GlRound<SM, LV>& R, uint8_t* slot, const GemvParams& p, __amdgpu_buffer_rsrc_t wr,
                      __amdgpu_buffer_rsrc_t br, int grp, int blk, int nb, int lane, int nr) {
  // rows past N repeat the last one and feed only outputs that are not stored;
  // blocks past the slice repeat its last one and are not consumed
#pragma unroll
  for (int i = 0; i < GL_SLOT / 1024; ++i) {
    const int pc = 64 * i + lane, row = pc / (2 * GL_BW);
    const int c = ((pc & (2 * GL_BW - 1)) - (row >> GL_ROT)) & (2 * GL_BW - 1);
    const int n = min(16 * grp + row, (int)p.N - 1);
    const uint32_t off = gl_mul(n, p.K >> 1) + (32u * (uint32_t)(blk + min(c >> 1, nb - 1)) + 16u * (c & 1));
    __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (__attribute__((address_space(3))) void*)(slot + 1024 * i), 16, off, 0,
                                             0, 0);
  }
  const int n = min(16 * grp + (lane & 15), (int)p.N - 1);
  // a slice's last wave may own no block: whole units of 4 then repeat the unit before
  const uint32_t b0 = gl_mul(n, p.K >> 6) + (uint32_t)(SM == 2 && nb < 1 ? blk + nb - GL_BW : blk);
  if constexpr (SM == 2) {
    R.q[0] = *reinterpret_cast<const uint32_t*>(p.q + b0);
    R.s[0] = p.absmax2[b0 >> p.dq_shift];
  } else {
#pragma unroll
    for (int b = 0; b < GL_BW; ++b) {
      const uint32_t bb = b0 + (uint32_t)min(b, nb - 1);
      if constexpr (SM == 0) {
        R.s[b] = p.scales[bb];
      } else {
        R.q[b] = p.q[bb];
      }
    }
    if constexpr (SM == 1) {                 // 4 blocks lie in at most two groups of dq_block >= 4
      R.s[0] = p.absmax2[(b0 + (uint32_t)min(0, nb - 1)) >> p.dq_shift];
      R.s[1] = p.absmax2[(b0 + (uint32_t)(nb - 1)) >> p.dq_shift];
    }
  }
  // The lane's 8 entries of B's row (an address and a load per rank spilled registers, whose reloads waited for the
  // stream). Ranks past r read what follows and are masked where they are used. Lanes without any read zeros from past
  // B's end, without traffic, where the offset is not clamped.
  if constexpr (LV != 0) {
    const uint32_t row = LV == 1 ? gl_mul(n, p.r) * 4u + (nr > 0 ? (uint32_t)(p.r - nr) * 4u : 0x80000000u) : 0u;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint32_t off = LV == 1 ? row + 16u * h : gl_b_offset(p, n, nr, h);
      const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(br, off, 0, 0);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t w = v[e];
        R.lb[4 * h + e] = __builtin_bit_cast(float, w);
      }
    }
  }
}

// Block `blk` of X's first 8 NI rows (rows past M repeat the last one): 8 pieces to a row, as gl_pos.
template <int NI>
MOLT_DEV void gl_load_x(__amdgpu_buffer_rsrc_t xr, uint8_t* slot, const GemvParams& p, int blk, int lane) {
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int pc = 64 * i + lane, row = pc / (2 * GL_BW);
    const int c = ((pc & (2 * GL_BW - 1)) - (row >> GL_ROT)) & (2 * GL_BW - 1);
    const uint32_t off = gl_mul(min(row, p.M - 1), (int)p.ldx) * 2u + 128u * (uint32_t)blk + 16u * (uint32_t)c;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (__attribute__((address_space(3))) void*)(slot + 1024 * i), 16, off, 0,
                                             0, 0);
  }
}

template <int SM, int LV>
MOLT_DEV f32x4_t gl_compute(const GlRound<SM, LV>& R, const uint8_t* slot, const GemvParams& p, GlSmem& sm, uint32_t lb,
                            const u32x4_t (&xf)[GL_BW][2], const u32x4_t& tf, int grp, int blk, int nb, int nr, int lane) {
  const int col = lane & 15, g = lane >> 4;
  int first = 0;                       // mode 1: blocks of entry s[0]; the others are s[1]'s
  if constexpr (SM == 1) {
    const uint32_t b0 = gl_mul(min(16 * grp + col, (int)p.N - 1), p.K >> 6) + (uint32_t)blk;
    first = (1 << p.dq_shift) - (int)(b0 & ((1u << p.dq_shift) - 1));
  }
  u32x2_t w[GL_BW];
#pragma unroll
  for (int b = 0; b < GL_BW; ++b)
    w[b] = *reinterpret_cast<const u32x2_t*>(slot + 16 * gl_pos(col, 2 * b + (g >> 1)) + 8 * (g & 1));
  float sc[GL_BW];
#pragma unroll
  for (int b = 0; b < GL_BW; ++b) {
#pragma clang fp contract(off)
    if constexpr (SM == 0) {
      sc[b] = R.s[b];
    } else {
      const uint32_t q = SM == 2 ? (R.q[0] >> (8 * b)) & 0xffu : R.q[SM == 2 ? 0 : b];
      const float prod = *gl_code2(sm, q) * (SM == 2 || b < first ? R.s[0] : R.s[1]);
      sc[b] = prod + p.offset;
    }
  }
  const char* tab = reinterpret_cast<const char*>(sm.tab);
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int b = 0; b < GL_BW; ++b) {
    u32x4_t c[2];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < 4; ++j)      // bits 15:8 = byte j of the dword, bits 7:0 = the lane's copy offset
        c[h][j] = *reinterpret_cast<const uint32_t*>(tab + __builtin_amdgcn_perm(w[b][h], lb, 0x0C0C0400u | ((uint32_t)j << 8)));
    const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    f32x4_t v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8v, xf[b][0]),
                                                        __builtin_bit_cast(bf16x8v, c[0]), zero, 0, 0, 0);
    v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8v, xf[b][1]),
                                                __builtin_bit_cast(bf16x8v, c[1]), v, 0, 0, 0);
    if (b < nb) {                      // uniform: the last wave of a slice may own fewer blocks
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] += sc[b] * v[e];
    }
  }
  if constexpr (LV != 0) {
    // Only the lane's first nr ranks exist (none on waves without ranks of slice
    // 0). T is zero past them, and so is B here: the entry it was clamped to may
    // be infinite, and zero times that is not zero. Masked when it is used: at
    // its load the select would wait for it.
    u32x4_t bw;
    if constexpr (LV == 1) {               // ranks of 4: all or none
#pragma unroll
      for (int e = 0; e < 4; ++e) bw[e] = nr > 4 * (e >> 1) ? pack_bf16x2(p.s * R.lb[2 * e], p.s * R.lb[2 * e + 1]) : 0u;
    } else {
      float b[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) b[e] = R.lb[e];
      if (16 * grp + 15 >= (int)p.N - 4) {   // uniform: the rows whose loads may have been moved back
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const uint32_t sh = gl_b_shift(p, min(16 * grp + col, (int)p.N - 1), nr, h);
#pragma unroll
          for (int e = 0; e < 4; ++e) b[4 * h + e] = sh & 1 ? b[4 * h + (e < 3 ? e + 1 : 3)] : b[4 * h + e];
#pragma unroll
          for (int e = 0; e < 2; ++e) b[4 * h + e] = sh & 2 ? b[4 * h + e + 2] : b[4 * h + e];
        }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
        bw[e] = pack_bf16x2(2 * e < nr ? p.s * b[2 * e] : 0.0f, 2 * e + 1 < nr ? p.s * b[2 * e + 1] : 0.0f);
    }
    const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    const f32x4_t v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8v, tf),
                                                              __builtin_bit_cast(bf16x8v, bw), zero, 0, 0, 0);
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] += v[e];
  }
  return acc;
}

// The waves' partial sums are written and read in assembly: the compiler, which
// cannot tell this memory from the slots being filled, would wait for the whole
// stream first. gl_write's operand comes from vector arithmetic (a matrix
// instruction's result would need wait states that it does not see here) and
// the caller waits for it; gl_read4 reads four consecutive waves' entries (2 KB
// apart; past the last wave the read stays in the table and is dropped).
MOLT_DEV uint32_t gl_addr(const float* at) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const float*)at;
}
MOLT_DEV void gl_write(const float* at, const f32x4_t& v) {
  asm volatile("ds_write_b128 %0, %1" ::"v"(gl_addr(at)), "v"(v) : "memory");
}
MOLT_DEV void gl_read4(const float* at, float (&u)[4]) {
  asm volatile("ds_read_b32 %0, %4\n\tds_read_b32 %1, %4 offset:2048\n\tds_read_b32 %2, %4 offset:4096\n\t"
               "ds_read_b32 %3, %4 offset:6144\n\ts_waitcnt lgkmcnt(0)"
               : "=&v"(u[0]), "=&v"(u[1]), "=&v"(u[2]), "=&v"(u[3]) : "v"(gl_addr(at)) : "memory");
}

// slice_blocks: blocks of a K slice; wpg = ceil(slice_blocks / GL_BW) waves to a
// group; gpr groups side by side; rounds = rounds of this grid.
template <int SM, int LV, bool ONE>
__global__ __launch_bounds__(GL_NT) __attribute__((amdgpu_waves_per_eu(4)))
void nf4_gemv_lds_kernel(const GemvParams p, int slice_blocks, int wpg, int gpr, int rounds, float* part) {
  __shared__ GlSmem sm;
  __shared__ __attribute__((aligned(16))) uint8_t r0[GL_WAVES * GL_SLOT], r1[GL_WAVES * GL_SLOT], r2[GL_WAVES * GL_SLOT];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, g = lane >> 4;
  const int q = wave / wpg, wi = wave % wpg;                           // group of the round, wave within it
  const bool active = q < gpr;
  const int KB = p.K >> 6, sl = (int)blockIdx.y;
  const int b_end = min((sl + 1) * slice_blocks, KB);
  const int blk = sl * slice_blocks + (active ? wi * GL_BW : 0);
  const int nb = min(GL_BW, b_end - blk);                              // <= 0: no block of the slice is left
  const int jc = active ? 32 * wi : 0;
  const bool lora = LV != 0 && active && sl == 0 && jc < p.r;
  const int nr = lora ? p.r - jc - 8 * g : 0;                          // ranks left to this lane's 8

  typedef __attribute__((address_space(4))) const f32x4_t* cptr_t;
  const cptr_t cbp = (cptr_t)p.code;
  const f32x4_t cb0 = cbp[0], cb1 = cbp[1], cb2 = cbp[2], cb3 = cbp[3];
  float c2 = 0.0f;
  if constexpr (SM != 0) c2 = p.code2[tid & 255];
  const int mc = col < p.M ? col : p.M - 1;
  u32x4_t tf = {0u, 0u, 0u, 0u};
  uint32_t tr8[8];                         // LV 2: T's entries as loaded, packed once they have landed
  if constexpr (LV != 0) {
    // Ranks past r, and waves without ranks of this slice, load from outside the
    // buffer: zeros, no traffic (T gathered by all waves cost 0.4 us a token) and
    // no branch or select that would wait for the load here. (In the forms of one
    // round the M <= 8 side below still begins with a wait for it: the two sides
    // share registers.)
    const __amdgpu_buffer_rsrc_t tr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(p.t), (short)0, (int)(((int64_t)(p.M - 1) * p.ldt + p.r) * 2), 0x00020000);
    const int j = jc + 8 * g;
    const uint32_t row = gl_mul(mc, (int)p.ldt) * 2u;
    auto at = [&](int jj) { return lora && jj < p.r ? row + 2u * (uint32_t)jj : 0xfffffff0u; };
    if constexpr (LV == 1) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const u32x2_t v = __builtin_amdgcn_raw_buffer_load_b64(tr, at(j + 4 * h), 0, 0);
        tf[2 * h] = v[0]; tf[2 * h + 1] = v[1];
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) tr8[i] = __builtin_amdgcn_raw_buffer_load_b16(tr, at(j + i), 0, 0);
    }
  }
  __builtin_amdgcn_sched_barrier(0);       // the small loads stay ahead of the weight stream

  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(p.packed), (short)0, (int)(p.N * (p.K >> 1)), 0x00020000);
  const __amdgpu_buffer_rsrc_t br = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(p.lb), (short)0, (int)(p.N * p.r * 4), 0x00020000);
  // group of round j: rounds past the last repeat the workgroup's own last one (never computed)
  const int glast = (int)((p.N - 1) >> 4), per = (int)gridDim.x * gpr;
  auto grp = [&](int j) { return min(min(j, rounds - 1) * per + (int)blockIdx.x * gpr + q, glast); };
  GlRound<SM, LV> b0, b1, b2;
  uint8_t* s0 = r0 + wave * GL_SLOT;
  uint8_t* s1 = r1 + wave * GL_SLOT;
  uint8_t* s2 = r2 + wave * GL_SLOT;
  // X comes through LDS too: fragments straight from memory take 16 bytes of 16
  // rows in neighbouring lanes, which the load path serves a lane at a time (2.7
  // us for 16 rows), rows of 128 bytes 64 bytes a clock. Block b of 16 rows is a
  // slot's 2 KB: two go to the slots of rounds 1 and 2 and two to the table's
  // place. Up to 8 rows all four fit there, and round 1 need not wait for them.
  uint8_t* xs = reinterpret_cast<uint8_t*>(sm.tab) + wave * 2 * GL_SLOT;
  const bool x8 = p.M <= 8;
  auto pack_t = [&]() {
#pragma unroll
    for (int i = 0; i < 4; ++i) tf[i] = tr8[2 * i] | (tr8[2 * i + 1] << 16);
  };
  u32x4_t xf[GL_BW][2];
  if (active) {
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(p.x), (short)0, (int)(((int64_t)(p.M - 1) * p.ldx + p.K) * 2), 0x00020000);
    static_assert(GL_BW == 4, "four blocks of X in four places");
    if (x8) {
#pragma unroll
      for (int b = 0; b < GL_BW; ++b) gl_load_x<1>(xr, xs + 1024 * b, p, blk + min(b, nb - 1), lane);
      __builtin_amdgcn_sched_barrier(0);
      gl_load(b0, s0, p, wr, br, grp(0), blk, nb, lane, nr);
      loads_in_order();                      // round 0's wait counts every load of round 1 as younger
      if constexpr (!ONE) gl_load(b1, s1, p, wr, br, grp(1), blk, nb, lane, nr);
      __builtin_amdgcn_sched_barrier(0);
      wait_vm<(ONE ? 1 : 2) * GlRound<SM, LV>::kLoads>();
      if constexpr (LV == 2) pack_t();
      asm volatile("" ::"v"(c2), "v"(tf) : "memory");      // older loads, landed: said here, where they can still be counted
#pragma unroll
      for (int b = 0; b < GL_BW; ++b)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          xf[b][h] = *reinterpret_cast<const u32x4_t*>(xs + 1024 * b + 16 * gl_pos(col & 7, 2 * g + h));
    } else {
      gl_load_x<2>(xr, s1, p, blk + min(0, nb - 1), lane);
      gl_load_x<2>(xr, s2, p, blk + min(1, nb - 1), lane);
      gl_load_x<2>(xr, xs, p, blk + min(2, nb - 1), lane);
      gl_load_x<2>(xr, xs + GL_SLOT, p, blk + min(3, nb - 1), lane);
      __builtin_amdgcn_sched_barrier(0);
      gl_load(b0, s0, p, wr, br, grp(0), blk, nb, lane, nr);
      __builtin_amdgcn_sched_barrier(0);
      wait_vm<GlRound<SM, LV>::kLoads>();
      if constexpr (LV == 2) pack_t();
      asm volatile("" ::"v"(c2), "v"(tf) : "memory");
      const uint8_t* at[GL_BW] = {s1, s2, xs, xs + GL_SLOT};
#pragma unroll
      for (int b = 0; b < GL_BW; ++b)
#pragma unroll
        for (int h = 0; h < 2; ++h) xf[b][h] = *reinterpret_cast<const u32x4_t*>(at[b] + 16 * gl_pos(col, 2 * g + h));
      if constexpr (!ONE) {
        __builtin_amdgcn_s_waitcnt(0xC07F);    // the slot of round 1 has been read
        asm volatile("" ::: "memory");
        gl_load(b1, s1, p, wr, br, grp(1), blk, nb, lane, nr);
      }
    }
  } else {
    asm volatile("" ::"v"(c2), "v"(tf));
  }
  __builtin_amdgcn_s_waitcnt(0xC07F);        // every wave's fragments are read: the table may be built
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  {
    static_assert(GL_NT == 1024, "table build covers 256 x 32 entries, two high nibbles a pass");
    const int lo = (tid >> 5) & 15, copy = tid & 31, h0 = tid >> 9;
    auto cv = [&](int i) { return i < 4 ? cb0[i & 3] : i < 8 ? cb1[i & 3] : i < 12 ? cb2[i & 3] : cb3[i & 3]; };
    float clo = cv(0);
#pragma unroll
    for (int i = 1; i < 16; ++i) clo = lo == i ? cv(i) : clo;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int hi = 2 * k + h0;
      const float even = cv(2 * k), odd = cv(2 * k + 1);
      const float chi = h0 ? odd : even;
      const float first = p.order ? chi : clo, second = p.order ? clo : chi;
      sm.tab[(hi * 16 + lo) * 64 + copy] = pack_bf16x2(first, second);
    }
    if (SM != 0) *gl_code2(sm, tid & 255) = c2;
  }
  __builtin_amdgcn_s_waitcnt(0xC07F);        // lgkmcnt(0): the barrier waits for the table, not for the stream
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  const uint32_t lb = (uint32_t)(lane & 31) * 4;

  // Round j computes from slot j % 3 with the next two rounds in flight, then
  // adds the waves' sums in LDS.
  constexpr int kFly = ONE ? 0 : 2 * GlRound<SM, LV>::kLoads;
  const int oq = tid >> 8, om = (tid >> 4) & 15, on = tid & 15;        // this thread's output: group, row, column
  auto reduce = [&](int j, const f32x4_t* acc) {
    if (j > 0) {                             // the sums of round j - 1 have been read
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    }
    if (acc) gl_write(gl_red(sm, wave, lane), *acc);
    __builtin_amdgcn_s_waitcnt(0xC07F);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (oq < gpr) {
      float v = 0.0f;
      for (int w = 0; w < wpg; w += 4) {
        float u[4];
        gl_read4(gl_red(sm, oq * wpg + w, 16 * (om >> 2) + on) + (om & 3), u);
#pragma unroll
        for (int i = 0; i < 4; ++i) v += w + i < wpg ? u[i] : 0.0f;
      }
      const int64_t n = 16 * ((int64_t)j * per + (int64_t)blockIdx.x * gpr + oq) + on;
      if (om < p.M && n < p.N) {
        if (gridDim.y == 1) p.y[(int64_t)om * p.ldy + n] = bf16_bits(v);
        else part[((int64_t)sl * p.M + om) * p.N + n] = v;
      }
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);      // the reads above are done before the next round's first barrier
    asm volatile("" ::: "memory");
  };
  if (!active) {                             // no group left for this wave: it only helps to add
    for (int j = 0; j < rounds; ++j) reduce(j, nullptr);
    return;
  }
  auto round = [&](int j, GlRound<SM, LV>& cur, const uint8_t* slot, GlRound<SM, LV>& nxt, uint8_t* into) {
    if constexpr (!ONE) gl_load(nxt, into, p, wr, br, grp(j + 2), blk, nb, lane, nr);
    __builtin_amdgcn_sched_barrier(0);
    wait_vm<kFly>();
    asm volatile("" ::: "memory");
    const f32x4_t acc = gl_compute(cur, slot, p, sm, lb, xf, tf, grp(j), blk, nb, nr, lane);
    reduce(j, &acc);
  };
  for (int j = 0;;) {
    round(j, b0, s0, b2, s2);
    if (ONE || ++j == rounds) break;
    round(j, b1, s1, b0, s0);
    if (++j == rounds) break;
    round(j, b2, s2, b1, s1);
    if (++j == rounds) break;
  }
  wait_vm<0>();                           // the repeated rounds land before the workgroup ends
}

// Y[m, n] = bf16(sum over K slices of the fp32 partials), slices in order.
__global__ void gm_reduce_kernel(const float* __restrict__ part, int slices, int M, int64_t N,
                                 uint16_t* __restrict__ y, int64_t ldy) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (int64_t)M * N) return;
  const int m = (int)(i / N);
  const int64_t n = i - (int64_t)m * N;
  float v = 0.0f;
  for (int k = 0; k < slices; ++k) v += part[(int64_t)k * M * N + i];
  y[(int64_t)m * ldy + n] = bf16_bits(v);
}

// T[m, j] = bf16(sum_k X[m, k] * bf16(A[j, k])) for the LoRA add-on of a decode
// call: one workgroup per rank j and up to MX tokens, each thread 8 consecutive
// k of every 4096, A rounded to bf16 as it is read (a decode batch is too small
// to repay packing A first). Latency-bound: 16 ranks of 14336 floats are 0.9
// MB, so the first TK_STEPS steps of a thread load everything they need before
// any of it is used, and the only wait after them is the sum over the 8 waves.
constexpr int TK_NT = 512, TK_STEP = 8 * TK_NT, TK_STEPS = 4;

template <int MX, bool VEC>
__global__ __launch_bounds__(TK_NT) void gemv_t_kernel(const uint16_t* __restrict__ x, int64_t ldx, int M, int K,
                                                       const float* __restrict__ a, uint16_t* __restrict__ t, int r) {
  __shared__ float red[TK_NT / 64][MX];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, j = (int)blockIdx.x, m0 = MX * (int)blockIdx.y;
  const float* row = a + (int64_t)j * K;
  const uint16_t* xr[MX];
#pragma unroll
  for (int m = 0; m < MX; ++m) xr[m] = x + (int64_t)min(m0 + m, M - 1) * ldx;
  float acc[MX];
#pragma unroll
  for (int m = 0; m < MX; ++m) acc[m] = 0.0f;
  for (int base = 8 * tid; base < K; base += TK_STEP * TK_STEPS) {
    float av[TK_STEPS][8];
    u32x4_t xv[TK_STEPS][MX];
#pragma unroll
    for (int s = 0; s < TK_STEPS; ++s) {
      const int k = min(base + s * TK_STEP, K - 8);                    // past the end: loaded, not used
      if (VEC) {
        const f32x4_t lo = *reinterpret_cast<const f32x4_t*>(row + k), hi = *reinterpret_cast<const f32x4_t*>(row + k + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) { av[s][e] = lo[e]; av[s][4 + e] = hi[e]; }
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) av[s][e] = row[k + e];
      }
#pragma unroll
      for (int m = 0; m < MX; ++m) xv[s][m] = *reinterpret_cast<const u32x4_t*>(xr[m] + k);
    }
#pragma unroll
    for (int s = 0; s < TK_STEPS; ++s) {
      if (base + s * TK_STEP >= K) continue;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t ab = pack_bf16x2(av[s][2 * e], av[s][2 * e + 1]);
#pragma unroll
        for (int m = 0; m < MX; ++m) {
          const uint32_t xw = xv[s][m][e];
          acc[m] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2v, ab), __builtin_bit_cast(bf16x2v, xw),
                                                   acc[m], false);
        }
      }
    }
  }
#pragma unroll
  for (int m = 0; m < MX; ++m) {
    const float v = gd_wave_sum(acc[m]);
    if (lane == 0) red[wave][m] = v;
  }
  __syncthreads();
  if (tid < MX && m0 + tid < M) {
    float v = 0.0f;
#pragma unroll
    for (int w = 0; w < TK_NT / 64; ++w) v += red[w][tid];
    t[(int64_t)(m0 + tid) * r + j] = bf16_bits(v);
  }
}

bool aligned(const void* p, size_t a) { return ((uintptr_t)p % a) == 0; }

}  // namespace
}  // namespace molt

using namespace molt;

namespace molt {
namespace {
// Plan of the streaming MFMA kernel: K slices of slice_blocks blocks, waves per
// group, groups side by side. A workgroup holds up to four groups (as many as its
// waves allow), but only as many as pay: what counts is rounds x groups a round,
// and among equals the fewer rounds. us, M = 5, as many as fit / as many as pay:
// 4096 x 896 6.0 / 4.5 (64 workgroups or 256), 2560 x 2048 6.1 / 5.2, 8960 x 896
// 6.1 / 5.7 (rounds of four or three groups), 8960 x 2048 8.7 / 7.8 (two rounds of
// two or three of one); 6144 x 1536 5.5 with two groups in one round, 6.5 with one
// in two.
struct GlPlan { int slices, slice_blocks, wpg, gpr; };
GlPlan gl_plan(int64_t N, int64_t K) {
  const int KB = (int)(K / 64), most = GL_WAVES * GL_BW;
  const int slices = (KB + most - 1) / most;
  // slices in whole units of GL_BW blocks, as even as they come
  const int sb = (((KB + GL_BW - 1) / GL_BW + slices - 1) / slices) * GL_BW;
  const int wpg = sb / GL_BW;
  GlPlan g{(KB + sb - 1) / sb, sb, wpg, 1};
  const int64_t groups = ceil_div64(N, 16), wgs = std::max(1, molt::device_cus() / g.slices);
  int64_t best = ceil_div64(groups, wgs);
  for (int n = 2; n <= std::min(4, GL_WAVES / wpg); ++n) {
    const int64_t cost = n * ceil_div64(ceil_div64(groups, n), wgs);
    if (cost <= best) { best = cost; g.gpr = n; }
  }
  return g;
}
// K slices of the fallback MFMA kernel (nf4_gemv_kernel): narrow outputs (at
// most 128 groups of 16 rows) split K over up to 8 workgroups per group, as
// many as keep two workgroups per CU and whole 4-block units for every wave.
int gv_slices(int64_t N, int64_t K) {
  const int64_t groups = ceil_div64(N, GV_ROWS);
  if (groups > 128 || K % 256 != 0) return 1;
  const int64_t units = K / 256;                        // 4-block units
  const int64_t s = std::min<int64_t>(std::min<int64_t>(8, units / GV_WAVES), 2 * molt::device_cus() / groups);
  return s < 2 ? 1 : (int)s;
}
}  // namespace
}  // namespace molt

// Whether molt_nf4_gemv refuses less than the queried workspace: where K is 2
// to 8 slices of 3584 or 4096 and M >= 2. Elsewhere a smaller one only means
// the kernel that does not split.
static bool gemv_needs_workspace(int64_t M, int64_t K) {
  if (M < 2 || K % 512 != 0 || K == 4096) return false;
  const int64_t c = K / 512;
  return (c % 7 == 0 && c > 7 && c / 7 <= 8) || (c % 7 != 0 && c % 8 == 0 && c / 8 <= 8);
}

// Kilobyte pieces of a row, and whether the dot kernel serves a call by its
// sizes (with 16-byte aligned codes). M = 1, 2 always. Up to 8 tokens over at
// most 2048 rows and K <= 4096 (eight X rows of at most two pieces fit in LDS
// beside the code table): eight tokens per lookup, where the MFMA kernel left
// most CUs idle (M = 8: 2048^2 5.4 / 6.8 us, 1536^2 5.3 / 5.6; 1024 x 4096 6.5 /
// 6.9. With its groups side by side only where they pay that kernel takes 5.1, 4.6
// and 6.0 there, from five tokens on: this line has not been moved yet. M = 4:
// 1536^2 4.1 / 4.5, 2048 x 8192 7.9 / 8.9, 1536 x 8960 7.7 / 10.3). M = 3, 4 with three
// pieces over at most 4096 rows, two rounds of the grid, where the MFMA kernel
// runs two slices, two or more rounds and their sum (4096 x 4160 8.5 / 11.1 us, 2112
// x 5120 8.1 / 9.5, 4096 x 6144 8.8 / 11.1; but 4608 x 5120 13.0 / 11.3, and with
// two or four pieces 4096^2 7.0 / 6.4, 2560 x 7168 11.5 / 10.9). The
// MOLT_TUNE_GEMV_DOT_M setting (0..8) replaces the rule by a plain bound on M.
static int64_t dot_pieces(int64_t K) { return ceil_div64(K, 2048); }
static bool dot_serves(int64_t M, int64_t N, int64_t K) {
  const int64_t pieces = dot_pieces(K);
  if (pieces > 7 || (M > 4 && pieces > 2)) return false;
  const int most = (int)molt::tuning_value(MOLT_TUNE_GEMV_DOT_M);
  if (most >= 0) return M <= most;
  return M <= 2 || (M <= 8 && N <= 2048) || (M <= 4 && N <= 4096 && pieces == 3);
}

extern "C" size_t molt_nf4_gemv_workspace(int64_t M, int64_t N, int64_t K) {
  // fp32 partials of the K slices when the streaming MFMA kernel, or the
  // fallback kernel of a narrow output, splits K
  const int ks = K >= 64 && (gemv_needs_workspace(M, K) || !dot_serves(M, N, K)) ? gl_plan(N, K).slices : 0;
  const int vs = gv_slices(N, K);
  const int s = std::max(ks, vs);
  return s > 1 ? (size_t)s * (size_t)M * (size_t)N * sizeof(float) : 0;
}

extern "C" int molt_nf4_gemv(const uint16_t* x, int64_t ldx, int64_t M, const molt_nf4_weight* w,
                             const uint16_t* t, int64_t ldt, const float* lora_b, int32_t r, float scaling,
                             uint16_t* y, int64_t ldy, void* workspace, size_t workspace_bytes,
                             void* stream) {
  const char* who = "molt_nf4_gemv";
  MOLT_REQUIRE(w && w->packed && w->code && x && y, MOLT_EINVAL, "%s: null argument", who);
  MOLT_REQUIRE(M >= 1 && M <= 16, MOLT_EUNSUPPORTED, "%s: M=%lld outside 1..16", who, (long long)M);
  MOLT_REQUIRE(w->block_size == 64 && w->cols % 64 == 0, MOLT_EUNSUPPORTED,
               "%s: needs block_size 64 and cols %% 64 == 0", who);
  MOLT_REQUIRE(w->cols < (1ll << 30), MOLT_EUNSUPPORTED, "%s: cols too large", who);
  MOLT_REQUIRE(w->rows * (w->cols / 2) < (1ll << 31) && M * ldx < (1ll << 30), MOLT_EUNSUPPORTED,
               "%s: weight or activations too large for 32-bit offsets", who);
  MOLT_REQUIRE(w->rows > 0 && ldx >= w->cols && ldy >= w->rows, MOLT_EINVAL, "%s: bad shape/stride", who);
  MOLT_REQUIRE(ldx % 8 == 0 && aligned(x, 16) && aligned(w->packed, 8) && aligned(w->code, 16), MOLT_EINVAL,
               "%s: X rows and the codebook must be 16-byte aligned and packed data 8-byte aligned", who);
  MOLT_REQUIRE(r >= 0 && (r == 0 || (t && lora_b && ldt >= r)), MOLT_EINVAL, "%s: bad LoRA operands", who);
  MOLT_REQUIRE(r <= GV_RMAX, MOLT_EUNSUPPORTED, "%s: LoRA rank %d > %d", who, r, GV_RMAX);
  const bool nested = w->nested != 0;
  MOLT_REQUIRE(nested ? (w->absmax_q && w->absmax2 && w->code2 && w->dq_block > 0) : (w->scales != nullptr),
               MOLT_EINVAL, "%s: scale statistics missing", who);
  int shift = 0;
  if (nested) {
    MOLT_REQUIRE((w->dq_block & (w->dq_block - 1)) == 0, MOLT_EUNSUPPORTED,
                 "%s: nested block %d is not a power of two", who, w->dq_block);
    while ((1 << shift) < w->dq_block) ++shift;
  }
  GemvParams p{};
  p.x = x; p.ldx = ldx; p.M = (int)M; p.packed = w->packed; p.N = w->rows; p.K = (int)w->cols;
  p.scales = nested ? nullptr : w->scales;
  p.q = w->absmax_q; p.absmax2 = w->absmax2; p.code2 = nested ? w->code2 : nullptr; p.offset = w->offset;
  p.dq_shift = shift;
  p.code = w->code; p.order = w->nibble_order;
  p.t = t; p.ldt = ldt; p.lb = lora_b; p.r = r; p.s = scaling; p.y = y; p.ldy = ldy;
  const int64_t groups = ceil_div64(p.N, GV_ROWS);
  MOLT_REQUIRE(groups < (1ll << 31), MOLT_EINVAL, "%s: problem too large", who);
  hipStream_t st = (hipStream_t)stream;
  // Decode: streaming dot-product kernel, one row per wave per round, as many
  // workgroups as fit on the GPU at once (two per CU at K = 4096 with up to two
  // tokens, else one; at K = 14336 three rounds of 7 KB per wave need ~190
  // registers); the waves loop over the rounds. M = 2 runs with two X rows, 3
  // and 4 with four. It serves the calls of dot_serves, and up to four tokens
  // without the workspace for the MFMA kernel's slices. Elsewhere that kernel is
  // the faster one (M = 4: 4096 x 14336 17.6 / 16.6 us).
  // Any K (a multiple of 64, at most 7 pieces of 2048): a row is IPR pieces of
  // 1 KB, the last possibly partial; IPR is rounded up to an instantiated
  // value (a wholly idle piece re-reads the row's last bytes and is dropped).
  const GlPlan gl = gl_plan(w->rows, w->cols);
  const size_t gl_need = gl.slices > 1 ? (size_t)gl.slices * (size_t)M * (size_t)w->rows * sizeof(float) : 0;
  const bool gl_ws = gl_need == 0 || (workspace && workspace_bytes >= gl_need && aligned(workspace, 16));
  const int ipr_need = (int)dot_pieces(w->cols);
  const bool dot_m = dot_serves(M, w->rows, w->cols) ||
                     (M <= 4 && ipr_need <= 7 && !gl_ws && molt::tuning_value(MOLT_TUNE_GEMV_DOT_M) < 0);
  if (dot_m && aligned(w->packed, 16)) {
    const int ipr = ipr_need <= 3 ? ipr_need : (ipr_need <= 5 ? 5 : 7);
    const int cus = molt::device_cus();
    const int rw = 1;                                         // rows per wave per round
    const int mx = M == 1 ? 1 : (M == 2 ? 2 : (M <= 4 ? 4 : 8));   // X rows held by the kernel
    // One workgroup per CU, so that each wave has more rounds over the same
    // set-up work (code table, X, LoRA operands): one token 4096^2 5.2 -> 4.95
    // us, 14336 x 4096 10.5-11.2 -> 10.1-10.2 us, 8960 x 1536 6.4 -> 5.4 us;
    // two tokens 14336 x 4096 12.8-13.1 -> 12.1-12.5 us, 8960 x 1536 7.6 ->
    // 6.4 us. Two (the kernel then fits in 128 registers) for two tokens over
    // at most 4096 rows, where one measured slower (4096^2: 5.35 -> 5.6 us).
    const int per_cu = ipr <= 2 && mx == 2 && w->rows <= 4096 ? 2 : 1;
    const int64_t waves = std::min<int64_t>(ceil_div64(w->rows, rw), (int64_t)cus * GD_WAVES * per_cu);
    const int64_t wgs = ceil_div64(waves, GD_WAVES);
    const int rounds = (int)ceil_div64(w->rows, wgs * GD_WAVES * rw);
    const size_t dyn = ipr == 2 && mx == 1 ? 0 : (size_t)mx * (ipr * 2048 + GD_XPAD) * 2;   // X in registers
    // rows of whole pieces (K = 4096, 14336) skip the partial-piece clamps and masks
    const bool full = w->cols == (int64_t)ipr * 2048;
#define MOLT_GDK(IPRv, MXv, NE, LO, MR)                                                                        \
  do {                                                                                                          \
    if ((IPRv == 2 || IPRv == 7) && full)                                                                       \
      hipLaunchKernelGGL((nf4_gemv_dot_kernel<1, IPRv, MXv, NE, LO, MR, (IPRv == 2 || IPRv == 7)>),             \
                         dim3((unsigned)wgs), dim3(GD_NT), dyn, st, p, rounds);                                 \
    else                                                                                                        \
      hipLaunchKernelGGL((nf4_gemv_dot_kernel<1, IPRv, MXv, NE, LO, MR, false>), dim3((unsigned)wgs), dim3(GD_NT), \
                         dyn, st, p, rounds);                                                                   \
  } while (0)
    // nested statistics with at most 4 rounds per wave (every cfg5 decode shape): straight-line rounds
#define MOLT_GDS(IPRv, MXv, LO)                                                   \
  do {                                                                            \
    if (rounds == 1) MOLT_GDK(IPRv, MXv, true, LO, 1);                                       \
    else if (rounds == 2) MOLT_GDK(IPRv, MXv, true, LO, 2); else MOLT_GDK(IPRv, MXv, true, LO, 4); \
  } while (0)
#define MOLT_GD(IPRv, MXv)                                                                                  \
  do {                                                                                                      \
    if (nested && rounds <= 4) { if (r > 0) MOLT_GDS(IPRv, MXv, true); else MOLT_GDS(IPRv, MXv, false); } \
    else if (nested) { if (r > 0) MOLT_GDK(IPRv, MXv, true, true, 0); else MOLT_GDK(IPRv, MXv, true, false, 0); } \
    else { if (r > 0) MOLT_GDK(IPRv, MXv, false, true, 0); else MOLT_GDK(IPRv, MXv, false, false, 0); }     \
  } while (0)
#define MOLT_GDI(IPRv)                                                                               \
  do {                                                                                                 \
    if (mx == 1) MOLT_GD(IPRv, 1);                                                                     \
    else if (mx == 2) MOLT_GD(IPRv, 2);                                                                \
    else if (mx == 4) MOLT_GD(IPRv, 4);                                                                \
    else MOLT_GD((IPRv <= 2 ? IPRv : 2), 8);   /* eight rows: at most two pieces (see dot_m) */       \
  } while (0)
    switch (ipr) {
      case 1: MOLT_GDI(1); break;
      case 2: MOLT_GDI(2); break;
      case 3: MOLT_GDI(3); break;
      case 5: MOLT_GDI(5); break;
      default: MOLT_GDI(7); break;
    }
#undef MOLT_GDI
#undef MOLT_GD
#undef MOLT_GDS
#undef MOLT_GDK
    return check_launch(who);
  }
  // Any other batch: the streaming MFMA kernel, one workgroup per CU, K split
  // over the waves (and, past 4096, over workgroups with fp32 partials). Each
  // LoRA rank chunk of 32 needs a wave of its own, the DMA 16-byte aligned rows,
  // and a wave's four blocks at most two nested groups; what is left (and a
  // workspace below the query) goes to the one-group kernel, which was the
  // slower one at every size measured (see nf4_gemv_lds_kernel).
  MOLT_REQUIRE(gl_ws || !gemv_needs_workspace(M, w->cols), MOLT_EWORKSPACE,
               "%s: workspace of %zu bytes (16-byte aligned) needed, got %zu", who, gl_need, workspace_bytes);
  if (gl_ws && r <= 32 * gl.wpg && M * ldt < (1ll << 30) && w->rows * r < (1ll << 29) && (r == 0 || w->rows * r >= 4) && aligned(w->packed, 16) && (!nested || w->dq_block >= 4)) {
    const int64_t sets = ceil_div64(ceil_div64(w->rows, 16), gl.gpr);
    const int64_t wgs = std::max<int64_t>(1, std::min<int64_t>(sets, molt::device_cus() / gl.slices));
    const int rounds = (int)ceil_div64(sets, wgs);
    const bool q4u = nested && w->dq_block >= 4 && (w->cols / 64) % 4 == 0 && aligned(w->absmax_q, 4);
    float* part = gl.slices > 1 ? static_cast<float*>(workspace) : nullptr;
    const dim3 grid((unsigned)wgs, (unsigned)gl.slices);
    // whole groups of four ranks: nothing to shift at B's end, T as 8-byte vectors
    const int lv = r == 0 ? 0 : (r % 4 == 0 && ldt % 4 == 0 && aligned(t, 8) ? 1 : 2);
#define MOLT_GL(SMv, LVv) \
  do {                                                                                                                  \
    if (rounds == 1)                                                                                                    \
      hipLaunchKernelGGL((nf4_gemv_lds_kernel<SMv, LVv, true>), grid, dim3(GL_NT), 0, st, p, gl.slice_blocks, gl.wpg,   \
                         gl.gpr, rounds, part);                                                                         \
    else                                                                                                                \
      hipLaunchKernelGGL((nf4_gemv_lds_kernel<SMv, LVv, false>), grid, dim3(GL_NT), 0, st, p, gl.slice_blocks, gl.wpg,  \
                         gl.gpr, rounds, part);                                                                         \
  } while (0)
#define MOLT_GLS(SMv) \
  do { if (lv == 0) MOLT_GL(SMv, 0); else if (lv == 1) MOLT_GL(SMv, 1); else MOLT_GL(SMv, 2); } while (0)
    if (!nested) MOLT_GLS(0); else if (q4u) MOLT_GLS(2); else MOLT_GLS(1);
#undef MOLT_GLS
#undef MOLT_GL
    if (gl.slices > 1) {
      const int rc = check_launch(who);
      if (rc) return rc;
      const int64_t n = M * w->rows;
      hipLaunchKernelGGL(gm_reduce_kernel, dim3((unsigned)ceil_div64(n, 256)), dim3(256), 0, st, part, gl.slices,
                         (int)M, w->rows, y, ldy);
    }
    return check_launch(who);
  }
  const bool q4 = nested && (w->cols / 64) % 4 == 0 && w->dq_block >= 4 && aligned(w->absmax_q, 4);
  // narrow outputs split K over workgroups (fp32 partials summed in slice order)
  int vs = gv_slices(w->rows, w->cols);
  if (vs > 1) {
    const size_t need = (size_t)vs * (size_t)M * (size_t)w->rows * sizeof(float);
    if (!(workspace && aligned(workspace, 16) && workspace_bytes >= need)) vs = 1;   // a smaller workspace: unsplit
  }
  float* part = vs > 1 ? static_cast<float*>(workspace) : nullptr;
  const dim3 grid((unsigned)groups, (unsigned)vs);
  if (q4) hipLaunchKernelGGL((nf4_gemv_kernel<true>), grid, dim3(GV_NT), 0, st, p, part);
  else hipLaunchKernelGGL((nf4_gemv_kernel<false>), grid, dim3(GV_NT), 0, st, p, part);
  if (vs > 1) {
    const int rc = check_launch(who);
    if (rc) return rc;
    const int64_t n = M * w->rows;
    hipLaunchKernelGGL(gm_reduce_kernel, dim3((unsigned)ceil_div64(n, 256)), dim3(256), 0, st, part, vs, (int)M,
                       w->rows, y, ldy);
  }
  return check_launch(who);
}

static size_t gemv_t_bytes(int64_t M, int32_t r) { return ((size_t)M * (size_t)r * 2 + 255) / 256 * 256; }

extern "C" size_t molt_nf4_lora_gemv_workspace(int64_t M, int64_t N, int64_t K, int32_t r) {
  return M > 0 && r > 0 ? gemv_t_bytes(M, r) + molt_nf4_gemv_workspace(M, N, K) : 0;
}

extern "C" int molt_nf4_lora_gemv(const uint16_t* x, int64_t ldx, int64_t M, const molt_nf4_weight* w,
                                  const float* lora_a, const float* lora_b, int32_t r, float scaling, uint16_t* y,
                                  int64_t ldy, void* workspace, size_t workspace_bytes, void* stream) {
  const char* who = "molt_nf4_lora_gemv";
  MOLT_REQUIRE(w && x && y && lora_a && lora_b, MOLT_EINVAL, "%s: null argument", who);
  MOLT_REQUIRE(M >= 1 && M <= 16, MOLT_EUNSUPPORTED, "%s: M=%lld outside 1..16", who, (long long)M);
  MOLT_REQUIRE(r >= 1 && r <= GV_RMAX, MOLT_EUNSUPPORTED, "%s: LoRA rank %d outside 1..%d", who, r, GV_RMAX);
  MOLT_REQUIRE(w->cols >= 64 && w->cols % 64 == 0 && w->cols < (1ll << 30), MOLT_EUNSUPPORTED,
               "%s: needs cols %% 64 == 0", who);
  MOLT_REQUIRE(ldx >= w->cols && ldx % 8 == 0 && aligned(x, 16), MOLT_EINVAL, "%s: X rows must be 16-byte aligned",
               who);
  const size_t need = molt_nf4_lora_gemv_workspace(M, w->rows, w->cols, r);
  MOLT_REQUIRE(workspace && workspace_bytes >= need && aligned(workspace, 256), MOLT_EWORKSPACE,
               "%s: workspace of %zu bytes (256-byte aligned) needed, got %zu", who, need, workspace_bytes);
  uint16_t* t = static_cast<uint16_t*>(workspace);
  const int K = (int)w->cols, mx = M == 1 ? 1 : M == 2 ? 2 : 4;
  const dim3 grid((unsigned)r, (unsigned)ceil_div64(M, mx));
  hipStream_t st = (hipStream_t)stream;
#define MOLT_TK(MXv, VECv) \
  hipLaunchKernelGGL((gemv_t_kernel<MXv, VECv>), grid, dim3(TK_NT), 0, st, x, ldx, (int)M, K, lora_a, t, r)
  if (aligned(lora_a, 16)) {
    if (mx == 1) MOLT_TK(1, true); else if (mx == 2) MOLT_TK(2, true); else MOLT_TK(4, true);
  } else {
    if (mx == 1) MOLT_TK(1, false); else if (mx == 2) MOLT_TK(2, false); else MOLT_TK(4, false);
  }
#undef MOLT_TK
  const int rc = check_launch(who);
  if (rc) return rc;
  const size_t tb = gemv_t_bytes(M, r);
  return molt_nf4_gemv(x, ldx, M, w, t, r, lora_b, r, scaling, y, ldy, (char*)workspace + tb, workspace_bytes - tb,
                       stream);
}

// ---------------------------------------------------------------------------
// molt_nf4_gemv_noalloc: molt_nf4_gemv with its split-K partials in a static
// device array instead of a caller workspace, for callers that cannot allocate.
// ---------------------------------------------------------------------------
namespace {
constexpr size_t GEMV_SCRATCH_BYTES = size_t(8) << 20;   // 2 Mi fp32 partials
constexpr int GEMV_SCRATCH_DEVICES = 64;

// One copy per device, held until the process ends. Host code never uses this
// name as an address: it is the host-side handle of the symbol, and only the
// per-device address that hipGetSymbolAddress returns is passed to kernels.
static __device__ __align__(256) unsigned char scratch[GEMV_SCRATCH_BYTES];

std::mutex g_scratch_mu;
void* g_scratch_addr[GEMV_SCRATCH_DEVICES];
// Per device: an event recorded after the last call that used the scratch, and
// the stream that call ran on. A call on another stream waits on the event
// first, so calls from different streams are ordered instead of racing.
hipEvent_t g_scratch_done[GEMV_SCRATCH_DEVICES];
hipStream_t g_scratch_stream[GEMV_SCRATCH_DEVICES];
bool g_scratch_used[GEMV_SCRATCH_DEVICES];

// Set-up on the first call on a device (with it current): the address of
// `scratch` and the ordering event, both kept until the process ends. Returns
// the device index through `dev_out`. The caller holds g_scratch_mu.
int scratch_setup(int* dev_out, const char* who) {
  int dev = -1;
  const hipError_t de = hipGetDevice(&dev);
  MOLT_REQUIRE(de == hipSuccess && dev >= 0 && dev < GEMV_SCRATCH_DEVICES, MOLT_ELAUNCH,
               "%s: no current device (%s)", who, hipGetErrorString(de));
  if (g_scratch_addr[dev] == nullptr) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    MOLT_REQUIRE(e == hipSuccess && p != nullptr, MOLT_ELAUNCH, "%s: scratch symbol lookup failed on device %d: %s",
                 who, dev, hipGetErrorString(e));
    hipEvent_t ev = nullptr;
    const hipError_t ee = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
    MOLT_REQUIRE(ee == hipSuccess, MOLT_ELAUNCH, "%s: scratch ordering event on device %d: %s", who, dev,
                 hipGetErrorString(ee));
    g_scratch_done[dev] = ev;
    g_scratch_addr[dev] = p;
  }
  *dev_out = dev;
  return MOLT_OK;
}

// True when `stream` is being captured into a graph. The legacy null stream
// cannot be captured, so it is not asked.
bool capturing(hipStream_t stream) {
  if (stream == nullptr) return false;
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  return hipStreamIsCapturing(stream, &st) == hipSuccess && st != hipStreamCaptureStatusNone;
}

// The calls that take the shared scratch. Everything that shares it is ordered by an event, and captured calls not even
// that, so a call takes it only where it has to (no kernel serves the shape unsplit) or where a narrow output would
// leave the GPU idle; elsewhere the dot kernel or the unsplit one-group kernel runs, on any number of streams at once.
bool noalloc_splits(int64_t M, const molt_nf4_weight* w) {
  const bool dot = aligned(w->packed, 16) &&
                   (dot_serves(M, w->rows, w->cols) ||
                    (M <= 4 && dot_pieces(w->cols) <= 7 && (w->cols == 14336 || !gemv_needs_workspace(M, w->cols)) &&
                     molt::tuning_value(MOLT_TUNE_GEMV_DOT_M) < 0));
  return !dot && (gemv_needs_workspace(M, w->cols) || gv_slices(w->rows, w->cols) > 1);
}
}  // namespace

extern "C" size_t molt_nf4_gemv_noalloc_limit(void) { return GEMV_SCRATCH_BYTES; }

extern "C" int molt_nf4_gemv_noalloc(const uint16_t* x, int64_t ldx, int64_t M, const molt_nf4_weight* w,
                                     const uint16_t* t, int64_t ldt, const float* lora_b, int32_t r, float scaling,
                                     uint16_t* y, int64_t ldy, void* stream) {
  const char* who = "molt_nf4_gemv_noalloc";
  MOLT_REQUIRE(w != nullptr, MOLT_EINVAL, "%s: null weight", who);
  MOLT_REQUIRE(M >= 1 && M <= 16 && w->rows > 0 && w->cols > 0, MOLT_EUNSUPPORTED, "%s: M=%lld outside 1..16 or empty weight",
               who, (long long)M);
  const size_t need = molt_nf4_gemv_workspace(M, w->rows, w->cols);
  MOLT_REQUIRE(need <= GEMV_SCRATCH_BYTES || !gemv_needs_workspace(M, w->cols), MOLT_EUNSUPPORTED,
               "%s: M=%lld, %lld x %lld needs %zu bytes of split-K partials, more than the %zu-byte static scratch "
               "(use molt_nf4_gemv with a workspace)",
               who, (long long)M, (long long)w->rows, (long long)w->cols, need, GEMV_SCRATCH_BYTES);
  if (need > GEMV_SCRATCH_BYTES || !noalloc_splits(M, w)) return molt_nf4_gemv(x, ldx, M, w, t, ldt, lora_b, r, scaling, y, ldy, nullptr, 0, stream);
  // Wait, launch and record under one lock, so calls from several host threads
  // are ordered as they take it. Under graph capture the graph's own order
  // applies and the event is neither waited on nor recorded.
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  int dev = -1;
  const int rc = scratch_setup(&dev, who);
  if (rc != MOLT_OK) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool order = !capturing(s);
  if (order && g_scratch_used[dev] && g_scratch_stream[dev] != s) {
    const hipError_t e = hipStreamWaitEvent(s, g_scratch_done[dev], 0);
    MOLT_REQUIRE(e == hipSuccess, MOLT_ELAUNCH, "%s: wait for the previous scratch user: %s", who,
                 hipGetErrorString(e));
  }
  // Nothing in the scratch has to start at zero: every partial the reduction
  // reads is written earlier in the same call.
  const int lrc = molt_nf4_gemv(x, ldx, M, w, t, ldt, lora_b, r, scaling, y, ldy, g_scratch_addr[dev], need, stream);
  if (lrc != MOLT_OK || !order) return lrc;
  const hipError_t e = hipEventRecord(g_scratch_done[dev], s);
  MOLT_REQUIRE(e == hipSuccess, MOLT_ELAUNCH, "%s: record the scratch ordering event: %s", who, hipGetErrorString(e));
  g_scratch_stream[dev] = s;
  g_scratch_used[dev] = true;
  return MOLT_OK;
}
