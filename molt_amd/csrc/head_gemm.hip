// GEMMs of the frozen LM head over one chunk of tokens (gfx950):
//
//   dH[M, H] = D[M, V] . W[V, H]      (the hidden gradient of a chunk)
//
// D are the chunk's dL/dlogits (bf16, row stride ldd) and W is the head as it
// lies in memory, so the contraction runs down W's rows: its tiles are 64 rows
// of 256 consecutive columns, brought in by DMA as they are and read as MFMA
// fragments by transposing LDS reads (ds_read_b64_tr_b16), with no transposed
// copy of the head.
//
// A chunk has few rows and an enormous contraction (256 x 1536 outputs over
// V = 151,936): six output tiles. V is split so that tiles x ranges fill the
// CUs; every range writes an fp32 partial and head_sum_kernel adds the ranges
// in order, so the result does not depend on which finishes first. The bound is
// the stream of W (467 MB a chunk, once), with the partials (S x M x H fp32,
// written and read) on top: a chunk of 256, V = 151,936, H = 1536 takes 135 us
// in all (the library GEMM, which does not split here, 496; W alone at the
// card's copy rate 91).
#include <algorithm>

#include "tile256.h"

namespace molt {
namespace {

using namespace big;

struct HeadGradParams {
  const uint16_t* d; int64_t ldd, M;
  const uint16_t* w; int64_t V, H;
  float* part;              // [S][M][H]
  int steps, split_steps;   // whole 64-deep steps in V, and in a range
  int tiles, nt_n;          // output tiles, and column tiles
};

typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4_t* tr_ptr_t;

// W tile in LDS: contraction row k at 256 k, its 32 16-byte chunks at position
// c ^ ((k & 7) << 1). A transposing read takes 16 lanes as 4 rows of 16
// columns: the swizzle puts the 4 rows' 32 bytes on different banks.
MOLT_DEV int wt_pos(int k, int c) { return k * 256 + ((c ^ ((k & 7) << 1)) << 3); }

// Fragments of 16-deep sub-step kk. a[i]: lane l holds column 32 i + l % 32 of
// the wave's 128 and contraction elements 8 (l / 32) .. + 7 as two transposing
// reads of 4 rows; lane l addresses row (l % 16) / 4 and columns 4 (l % 4) .. + 3
// of its 16 lanes' 4 x 16 block and receives column l % 16 of it. `ao` are the
// lane's offsets of the two reads at i = 0, kk = 0; subtile i flips position
// bits 2, 3 only (element offset bits 5, 6), sub-step kk adds 16 rows.
MOLT_DEV void load_frags_nn(const uint16_t* __restrict__ ws, const uint16_t* __restrict__ ds, const int (&ao)[2], int bo,
                            int kk, bf16x8_t (&a)[TM], bf16x8_t (&b)[TN]) {
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr_t)(ws + (ao[0] ^ (i << 5)) + 4096 * kk));
    const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr_t)(ws + (ao[1] ^ (i << 5)) + 4096 * kk));
    a[i] = __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  }
  const int bk = bo ^ (kk << 4);
#pragma unroll
  for (int j = 0; j < TN; ++j) b[j] = *reinterpret_cast<const bf16x8_t*>(ds + bk + 2048 * j);
}

__global__ __launch_bounds__(NT) void head_grad_kernel(const HeadGradParams p) {
  __shared__ __attribute__((aligned(16))) uint16_t wb0[BUF], wb1[BUF], wb2[BUF], db0[BUF], db1[BUF];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave % WAVES_M, wn = wave / WAVES_M;
  // The output tiles of one range are neighbours: they read the same columns
  // of D, which meet in their XCD's L2.
  const uint32_t b = blockIdx.x, per = gridDim.x / 8, more = gridDim.x % 8, xcd = b % 8;   // xcd_tile in 32 bits
  const uint32_t t = xcd * per + min(xcd, more) + b / 8;
  const int split = (int)(t / (uint32_t)p.tiles), tile = (int)(t % (uint32_t)p.tiles);
  const int64_t m0 = (int64_t)(tile / p.nt_n) * BM, n0 = (int64_t)(tile % p.nt_n) * BN;
  const int sbeg = split * p.split_steps, n = min(p.split_steps, p.steps - sbeg);

  // D rows past M repeat the last row and columns past H the last chunk: they
  // feed only outputs that are not stored.
  const __amdgpu_buffer_rsrc_t dr = make_rsrc(p.d, ((p.M - 1) * p.ldd + p.V) * 2);
  const __amdgpu_buffer_rsrc_t wr = make_rsrc(p.w, p.V * p.H * 2);
  uint32_t doff[4], woff[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    int R, k;
    dma_slot(wave * 4 + c, lane, R, k);
    doff[c] = (uint32_t)((min(m0 + R, p.M - 1) * p.ldd + k) * 2);
    const int kw = 2 * (wave * 4 + c) + (lane >> 5), ch = (lane & 31) ^ ((kw & 7) << 1);
    woff[c] = (uint32_t)((kw * p.H + min(n0 + 8 * ch, p.H - 8)) * 2);
  }
  // indices past the end repeat the last step (loaded, never read)
  auto d_load = [&](uint16_t* dst, int j) {
    const uint32_t so = (uint32_t)(sbeg + min(j, n - 1)) * (BK * 2);
#pragma unroll
    for (int c = 0; c < 4; ++c) buf_load_lds16(dr, dst + (wave * 4 + c) * 512, doff[c], so);
  };
  auto w_load = [&](uint16_t* dst, int j) {
    const uint32_t so = (uint32_t)(sbeg + min(j, n - 1)) * (uint32_t)(BK * 2 * p.H);
#pragma unroll
    for (int c = 0; c < 4; ++c) buf_load_lds16(wr, dst + (wave * 4 + c) * 512, woff[c], so);
  };

  const int q = (lane & 15) >> 2, c0 = wn * 16 + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
  int ao[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) ao[h] = wt_pos(8 * (lane >> 5) + 4 * h + q, c0) + 4 * (lane & 1);
  const int bo = loff(wm * WCOLS + (lane & 31), lane >> 5);

  f32x16_t acc[TM][TN];
  zero_acc(acc);
  bf16x8_t a[2][TM], bf[2][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i) a[1][i] = bf16x8_t{};
#pragma unroll
  for (int j = 0; j < TN; ++j) bf[1][j] = bf16x8_t{};

  if (n > 0) {
    // W streams from memory and is loaded two steps ahead into a ring of three;
    // D, shared by the range's tiles, one step ahead into two. The last
    // sub-step's MFMAs run under the next step's first reads.
    w_load(wb0, 0);
    d_load(db0, 0);
    loads_in_order();
    w_load(wb1, 1);
    wait_vm<kStageDma>();
    step_barrier();
    auto step = [&](int j, const uint16_t* wc, const uint16_t* dc, uint16_t* w2, uint16_t* dnx) {
      load_frags_nn(wc, dc, ao, bo, 0, a[0], bf[0]);
      mfma_set(a[1], bf[1], acc);
      d_load(dnx, j + 1);
      loads_in_order();
      w_load(w2, j + 2);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kk = 0; kk < 3; ++kk) {
        load_frags_nn(wc, dc, ao, bo, kk + 1, a[(kk + 1) & 1], bf[(kk + 1) & 1]);
        mfma_set(a[kk & 1], bf[kk & 1], acc);
        __builtin_amdgcn_sched_barrier(0);
      }
      wait_vm<kStageDma>();                  // D(j + 1), W(j + 1) landed; W(j + 2) may fly
      step_barrier();
    };
    ring_steps(n, step, wb0, wb1, wb2, db0, db1);
    wait_vm<0>();
    __syncthreads();
    mfma_set(a[1], bf[1], acc);
  }
  // The contraction's end past the whole steps (V % 64, a multiple of 8), by
  // the last range: element loads of what lies inside, zeros outside.
  const int64_t k0 = (int64_t)p.steps * BK;
  if (k0 < p.V && (int)gridDim.x == (split + 1) * p.tiles) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      int R, k;
      dma_slot(wave * 4 + c, lane, R, k);
      u32x4_t dv = {0u, 0u, 0u, 0u}, wv = {0u, 0u, 0u, 0u};
      if (m0 + R < p.M && k0 + k < p.V) dv = *reinterpret_cast<const u32x4_t*>(p.d + (m0 + R) * p.ldd + k0 + k);
      const int kw = 2 * (wave * 4 + c) + (lane >> 5), ch = (lane & 31) ^ ((kw & 7) << 1);
      if (k0 + kw < p.V && n0 + 8 * ch < p.H)
        wv = *reinterpret_cast<const u32x4_t*>(p.w + (k0 + kw) * p.H + n0 + 8 * ch);
      *reinterpret_cast<u32x4_t*>(db0 + (wave * 4 + c) * 512 + 8 * lane) = dv;
      *reinterpret_cast<u32x4_t*>(wb0 + (wave * 4 + c) * 512 + 8 * lane) = wv;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      load_frags_nn(wb0, db0, ao, bo, kk, a[0], bf[0]);
      mfma_set(a[0], bf[0], acc);
    }
  }

  float* part = p.part + (int64_t)split * p.M * p.H;
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int64_t m = m0 + wm * WCOLS + j * 32 + (lane & 31);
    if (m >= p.M) continue;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int64_t nn = n0 + wn * WROWS + i * 32 + 8 * g + 4 * (lane >> 5);
        if (nn < p.H)
          *reinterpret_cast<f32x4_t*>(part + m * p.H + nn) =
              f32x4_t{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
      }
  }
}

// out = the sum of the partials in range order, 4 consecutive values a thread,
// HS_BATCH ranges' loads issued together.
constexpr int HS_BATCH = 8;
template <bool OUT_F32>
__global__ void head_sum_kernel(const float* __restrict__ part, int splits, int64_t total, void* __restrict__ out) {
  const int64_t e = 4 * ((int64_t)blockIdx.x * blockDim.x + threadIdx.x);
  if (e >= total) return;
  f32x4_t v = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int s0 = 0; s0 < splits; s0 += HS_BATCH) {
    f32x4_t w[HS_BATCH];
#pragma unroll
    for (int i = 0; i < HS_BATCH; ++i)
      w[i] = *reinterpret_cast<const f32x4_t*>(part + (int64_t)min(s0 + i, splits - 1) * total + e);
#pragma unroll
    for (int i = 0; i < HS_BATCH; ++i)
      if (s0 + i < splits)
#pragma unroll
        for (int c = 0; c < 4; ++c) v[c] += w[i][c];
  }
  if (OUT_F32) *reinterpret_cast<f32x4_t*>(reinterpret_cast<float*>(out) + e) = v;
  else *reinterpret_cast<u32x2_t*>(reinterpret_cast<uint16_t*>(out) + e) =
      u32x2_t{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
}

bool aligned(const void* p, size_t a) { return ((uintptr_t)p % a) == 0; }

// Ranges of V: as many as fill the CUs, each of at least 8 steps.
int head_splits(int64_t M, int64_t V, int64_t H, int& split_steps) {
  const int64_t tiles = ceil_div64(M, BM) * ceil_div64(H, BN), steps = V / BK;
  int64_t S = std::min<int64_t>(device_cus() / std::max<int64_t>(tiles, 1), steps / 8);
  S = std::max<int64_t>(S, 1);
  split_steps = (int)std::max<int64_t>(ceil_div64(steps, S), 1);
  return (int)std::max<int64_t>(ceil_div64(steps, split_steps), 1);
}

}  // namespace
}  // namespace molt

using namespace molt;

extern "C" size_t molt_head_grad_workspace(int64_t M, int64_t V, int64_t H) {
  if (M <= 0 || V <= 0 || H <= 0) return 0;
  int ss;
  return (size_t)head_splits(M, V, H, ss) * (size_t)M * (size_t)H * sizeof(float);
}

extern "C" int molt_head_grad(const uint16_t* dlogits, int64_t ldd, int64_t M, const uint16_t* w, int64_t V, int64_t H,
                              void* out, int32_t out_dtype, void* workspace, size_t workspace_bytes, void* stream) {
  const char* who = "molt_head_grad";
  MOLT_REQUIRE(M >= 0 && V > 0 && H > 0 && ldd >= V, MOLT_EINVAL, "%s: bad shape", who);
  MOLT_REQUIRE(out_dtype == MOLT_DTYPE_BF16 || out_dtype == MOLT_DTYPE_F32, MOLT_EINVAL, "%s: bad dtype", who);
  if (M == 0) return MOLT_OK;
  MOLT_REQUIRE(dlogits && w && out, MOLT_EINVAL, "%s: null argument", who);
  MOLT_REQUIRE(V % 8 == 0 && H % 8 == 0 && ldd % 8 == 0 && aligned(dlogits, 16) && aligned(w, 16) && aligned(out, 16),
               MOLT_EUNSUPPORTED, "%s: rows must be 16-byte aligned (V %% 8 == 0, H %% 8 == 0)", who);
  const int64_t lim = 0x7fffffffll;   // 32-bit buffer offsets
  MOLT_REQUIRE(((M - 1) * ldd + V) * 2 <= lim && V * H * 2 <= lim, MOLT_EUNSUPPORTED, "%s: operands above 2 GiB", who);
  const size_t need = molt_head_grad_workspace(M, V, H);
  MOLT_REQUIRE(workspace && workspace_bytes >= need && aligned(workspace, 16), MOLT_EWORKSPACE,
               "%s: workspace of %zu bytes (16-byte aligned) needed, got %zu", who, need, workspace_bytes);
  HeadGradParams p{};
  p.d = dlogits; p.ldd = ldd; p.M = M; p.w = w; p.V = V; p.H = H; p.part = (float*)workspace;
  p.steps = (int)(V / BK);
  const int S = head_splits(M, V, H, p.split_steps);
  p.nt_n = (int)ceil_div64(H, BN);
  p.tiles = (int)ceil_div64(M, BM) * p.nt_n;
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL(head_grad_kernel, dim3((unsigned)(p.tiles * S)), dim3(NT), 0, st, p);
  const int rc = check_launch(who);
  if (rc) return rc;
  const int64_t total = M * H;
  const dim3 grid((unsigned)ceil_div64(total / 4, 256));
  if (out_dtype == MOLT_DTYPE_F32)
    hipLaunchKernelGGL((head_sum_kernel<true>), grid, dim3(256), 0, st, p.part, S, total, out);
  else
    hipLaunchKernelGGL((head_sum_kernel<false>), grid, dim3(256), 0, st, p.part, S, total, out);
  return check_launch(who);
}
