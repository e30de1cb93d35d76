// The 256 x 256 workgroup tile shared by the NF4 GEMMs and the LM head's GEMMs
// (gfx950): operand buffers of 256 rows x 64 contraction elements in LDS, filled
// by buffer-load DMA and read as v_mfma_f32_32x32x16_bf16 fragments by 8 waves
// of 128 x 64 outputs.
#pragma once

#include "mfma_core.h"

namespace molt {
namespace {
namespace big {

constexpr int BM = 256, BN = 256, NT = 512, WAVES_M = 4;
constexpr int WROWS = 128, WCOLS = 64, TM = 4, TN = 2, LD = 64;
constexpr int GROUP_M = 4;
constexpr int BUF = BM * LD;     // bf16 elements of one operand buffer (32 KB)

// Operand buffer layout. A tile row holds its 64 contraction elements as 8
// chunks of 16 B in one 128-byte line, row R at 128 R, chunk c at position
// c ^ f(R) with f(R) = (R ^ ((R >> 3) & 3)) & 7. Then
//  * a ds_read_b128 of one chunk over 16 consecutive rows (served 16 lanes per
//    cycle over 64 banks) hits 16 distinct 16-byte bank groups: rows R and
//    R + 8 of the group differ in R & 1 or in f (the fragment reads);
//  * a 1 KB DMA block is 8 whole rows, so each 128-byte line of X is one
//    request (half-line requests doubled the L1 traffic);
//  * f(R + 32) = f(R), so the subtiles of a fragment read are one per-lane
//    base offset (XOR-ed with the sub-step) plus an immediate of 32 rows.
MOLT_DEV int lswz(int R) { return (R ^ ((R >> 3) & 3)) & 7; }
MOLT_DEV int loff(int R, int c) { return R * 64 + ((c ^ lswz(R)) << 3); }

// Global -> LDS DMA writes lane l's 16 bytes to (block base + 16 l): block blk
// (1 KB) of a buffer holds rows 8 blk .. 8 blk + 7, lane l filling position
// l % 8 of row 8 blk + l / 8. Returns the tile row and first contraction
// element the lane must fetch.
// DMA instructions that fill one operand buffer (16 bytes per lane each).
constexpr int kStageDma = BUF * 2 / (NT * 16);
static_assert(kStageDma == 4, "x_load and the staged W DMA issue 4 instructions per buffer");

// Value selects for the staged kernels' per-step sources. A conditional
// expression over two lvalues (captured variables, array elements) selects an
// address and loads through it, from scratch memory, which also makes the
// result look divergent; by-value parameters keep it a register select.
template <typename T>
MOLT_DEV T pick(bool c, T a, T b) { return c ? a : b; }

// Steps 0 .. n - 1 of a staged kernel: step j reads X buffer j % 3 and W
// buffer j % 2 and loads X(j + 2), W(j + 1) into the buffers read at step
// j - 1. The pattern repeats every 6 steps; every call names its buffers
// statically (the compiler then tells the LDS reads of one buffer from the
// DMA into another and inserts no waits between them).
template <typename Step>
MOLT_DEV void ring_steps(int n, Step& step, uint16_t* x0, uint16_t* x1, uint16_t* x2, uint16_t* w0, uint16_t* w1) {
  int j = 0;
  for (; j + 6 <= n; j += 6) {
    step(j, x0, w0, x2, w1);
    step(j + 1, x1, w1, x0, w0);
    step(j + 2, x2, w0, x1, w1);
    step(j + 3, x0, w1, x2, w0);
    step(j + 4, x1, w0, x0, w1);
    step(j + 5, x2, w1, x1, w0);
  }
  if (j < n) step(j, x0, w0, x2, w1);
  if (j + 1 < n) step(j + 1, x1, w1, x0, w0);
  if (j + 2 < n) step(j + 2, x2, w0, x1, w1);
  if (j + 3 < n) step(j + 3, x0, w1, x2, w0);
  if (j + 4 < n) step(j + 4, x1, w0, x0, w1);
}

MOLT_DEV void dma_slot(int blk, int lane, int& R, int& k) {
  R = 8 * blk + (lane >> 3);
  k = 8 * ((lane & 7) ^ lswz(R));
}

typedef __attribute__((address_space(3))) void* lds_ptr_t;

// Buffer resource over [p, p + bytes): loads through it are bounds-checked by
// the hardware (out-of-range lanes read zero) and take a 32-bit per-lane byte
// offset plus a uniform scalar offset, so no per-step 64-bit address math.
MOLT_DEV __amdgpu_buffer_rsrc_t make_rsrc(const void* p, int64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}
MOLT_DEV u32x4_t buf_load16(__amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t soff) {
  return __builtin_amdgcn_raw_buffer_load_b128(r, off, soff, 0);
}
MOLT_DEV uint32_t buf_load4(__amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t soff) {
  return __builtin_amdgcn_raw_buffer_load_b32(r, off, soff, 0);
}
// 16 bytes per lane from global straight into LDS at dst + 16 * lane (dst uniform).
MOLT_DEV void buf_load_lds16(__amdgpu_buffer_rsrc_t r, void* dst, uint32_t off, uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr_t)dst, 16, off, soff, 0, 0);
}
// Workgroup barrier without __syncthreads()'s release fence: the fence makes
// the compiler drain every outstanding vector-memory op, including register
// loads of packed weight bytes that are only used a step later. The caller
// waits explicitly (vmcnt) for the DMA other waves will read; this wave's own
// LDS stores are waited for here, and the empty asm statements keep the
// compiler from moving memory accesses across the barrier.
MOLT_DEV void step_barrier() {
  __builtin_amdgcn_s_waitcnt(0xC07F);              // lgkmcnt(0)
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Per-lane fragment offsets: lane l supplies row (l % 32) of each 32-row
// subtile and the 8-element half (l / 32) of a 16-deep sub-step. Sub-step kk
// reads chunk 2 kk + l / 32, whose position is (h ^ f(R)) ^ 2 kk: its offset
// is base ^ (kk << 4) (the XOR touches only the position bits); subtile i adds
// 32 rows = 2048 elements.
struct FragOff { int a, b; };

MOLT_DEV void frag_offsets(FragOff& f, int arow0, int brow0, int lane) {
  const int h = lane >> 5;
  f.a = loff(arow0 + (lane & 31), h);
  f.b = loff(brow0 + (lane & 31), h);
}

MOLT_DEV void load_frags(const uint16_t* __restrict__ ws, const uint16_t* __restrict__ xs, const FragOff& f, int kk,
                         bf16x8_t (&a)[TM], bf16x8_t (&b)[TN]) {
  const int ao = f.a ^ (kk << 4), bo = f.b ^ (kk << 4);
#pragma unroll
  for (int i = 0; i < TM; ++i)
    a[i] = *reinterpret_cast<const bf16x8_t*>(ws + ao + 2048 * i);
#pragma unroll
  for (int j = 0; j < TN; ++j)
    b[j] = *reinterpret_cast<const bf16x8_t*>(xs + bo + 2048 * j);
}

MOLT_DEV void mfma_set(const bf16x8_t (&a)[TM], const bf16x8_t (&b)[TN], f32x16_t (&acc)[TM][TN]) {
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
      acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
}

// One BK step from LDS (used by the LoRA steps): four 16-deep sub-steps, the
// fragment reads of sub-step kk+1 issued before the MFMAs of kk.
MOLT_DEV void compute(const uint16_t* __restrict__ ws, const uint16_t* __restrict__ xs, const FragOff& f,
                      f32x16_t (&acc)[TM][TN]) {
  bf16x8_t a[2][TM], b[2][TN];
  load_frags(ws, xs, f, 0, a[0], b[0]);
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) {
    if (kk < 3) load_frags(ws, xs, f, kk + 1, a[(kk + 1) & 1], b[(kk + 1) & 1]);
    mfma_set(a[kk & 1], b[kk & 1], acc);
    __builtin_amdgcn_sched_barrier(0);
  }
}

}  // namespace big
}  // namespace
}  // namespace molt
