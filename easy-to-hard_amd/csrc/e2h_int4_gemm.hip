// int4 group-wise matmul for many rows of x (prefill, scoring): MFMA-bound, 32x32 tiles.
//
// Same contract and data layouts as e2h_int4_mm.hip (torch.ops.aten._weight_int4pack_mm as called by
// linear_forward_int4, reference models/quantize.py:445-453), inner_k_tiles = 8, group size 32 / 64 / 128, and 256 as pairs of groups of 128
// that share a scale and a zero.
//
//   y[m,n] = sum_g  s[g,n] * sum_{k in g} x[m,k] * (16 + q[n,k])  +  sum_g (z[g,n] - 24 s[g,n]) * X[m,g]
//
// with X[m,g] = sum_{k in g} x[m,k] taken from a pre-pass (launch_x_group_sums).  Codes enter the matrix cores as the exact
// bfloat16 16 + q (rotate, and-or per two codes), so products are exact and sums float32.
//
// Scales.  An accumulator is kept in units of its column's current scale: entering group g it is multiplied by
// s[g-1,n] / s[g,n], and the group's products then add to it directly.  No second set of registers for the sums of one group,
// which is what lets a wave own 128 rows x 64 columns, so that one unpacked fragment feeds four MFMAs and one activation
// fragment two.  In a group whose scale is zero a column's operands are zeros and its unit stays.  Scales between 2^-100 and 2^13 (the
// quantizer's lie between 2^-24 and a few units) run like that: rescaling by up to 2^113 loses at most 2^-136 of a sum, below the smallest
// bfloat16.  A workgroup that meets any other (infinities, NaN) forms every group's sum by itself in a plain loop, which takes five to nine
// times as long (8192 x 11008 x 4096, group size 128, such a scale in every workgroup: 5850 us beside 680).  So does a wave whose
// sums leave float32's range in units of the scales although they may not by themselves (a zero of 2^100 beside a scale of 2^-20,
// activations near the type's end): an infinity or NaN in an accumulator stays one to the end, where it is looked for, but for the
// rows that have one in x.
// Group size 32 keeps that second set of registers (64 rows per workgroup, so they fit): rescaling 64 sums every two steps costs the same
// multiplications as adding 64 group sums, and the quotients and masks on top, 6 % of the kernel.  Every finite scale runs like that.
//
// The zero-point term is a matrix product over the groups.  It starts the accumulators: X and z - 24 s are each split into three
// bfloat16 parts (exact: 3 x 8 bits), and eight of the nine products of parts (all but low x low, 2^-32) fill one lane's eight k values,
// two groups per v_mfma_f32_32x32x16_bf16.  That is half the matrix time of the float32 instruction for the same two groups.
//
// Main loop, k in natural order: lane L = 32 h + n supplies column n0 + n and the eight k values 16 s + 8 h .. + 7 of step s.  A packed
// word (column, j, span p) holds the codes at k = 32 p + 8 i + 2 j + {0, 1} in nibbles i and i + 4, so dword j of the operand of step
// 2 p + a is word[j][p] rotated right by 8 a + 4 h - 3, masked to bits 3 .. 6 and 19 .. 22, over two bfloat16 sixteens.
// Four waves, 64, 96 or 128 rows x 256 columns per workgroup (kRT row tiles of 32), two workgroups per CU: one's start and end run under the
// other's matrix work.
// Operands reach LDS by 16-byte loads that write LDS directly:
//   activations, 128 rows x 64 k per chunk, three stages: 1 KB block b holds rows 8 b .. 8 b + 7, the 16-byte pieces of a row stored at
//   piece ^ ((row >> 1) & 7);
//   weights, 64 columns of one wave x 128 k, two stages: 64 bytes per column, pieces at piece ^ ((column >> 2) & 3), read by the wave
//   that loaded them.
// A gated launch (both matrices of silu(x w1) * (x w3)) gives a wave 32 columns of each, so that a lane holds both products of its outputs and multiplies them on the way out.
// One barrier per 64 k.  Where the row count leaves the chip short of workgroups, S of them share K and leave float32 sums for a
// second kernel to add in order.
//
// Workgroup -> tile mapping: workgroup w runs on XCD w % 8; each XCD owns the column blocks cb = xcd (mod 8) and
// walks them for one row block before moving to the next, so its L2 keeps that slice of the weights.
#include <algorithm>

#include "e2h_common.h"
#include "e2h_int4_unpack.h"

namespace e2h {
namespace {

typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void lds_void;

constexpr int kCols = 256, kCT = 2;

__device__ __forceinline__ uint32_t high_halves(float hi, float lo) {  // (bfloat16 bits of lo) | (of hi) << 16, truncated
  return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, hi), __builtin_bit_cast(uint32_t, lo), 0x07060302u);
}

// v = p[0] + p[1] + p[2], every part a bfloat16 value
__device__ __forceinline__ void split3(float v, float (&p)[3]) {
  p[0] = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, v) & 0xFFFF0000u);
  const float r = v - p[0];
  p[1] = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, r) & 0xFFFF0000u);
  p[2] = r - p[1];
}

// a / b, correctly rounded, for bfloat16 values between 2^-100 and 2^13: the first guess is a few units in the last place off, its residual
// is exact, and a quotient of two 8-bit significands is no closer to a rounding boundary than 2^-33 of itself.  (A division takes ten
// instructions; with one per group and column the kernel took 1.2 % longer at group size 64.)
__device__ __forceinline__ float quotient(float a, float b) {
  const float rcp = __builtin_amdgcn_rcpf(b), q = a * rcp;
  return __builtin_fmaf(__builtin_fmaf(-q, b, a), rcp, q);
}

// F.silu(a) * b on bfloat16 tensors, before the last rounding
__device__ __forceinline__ float gated(float a, float b) {
  const float gate = bf16_round(a);
  return bf16_round(gate / (1.0f + expf(-gate))) * bf16_round(b);
}

struct GemmArgs {
  const uint16_t *x;
  const uint32_t *wp, *sz, *wp2, *sz2;  // wp2, sz2: the second matrix of a gated launch
  uint16_t *y;
  float *partials;  // [S][M][N] when K is shared, else null
  const float *xsum;
  int xsum_stride, M, N, K, n_col_blocks, cbx;
  int shared;         // 1: two neighbouring groups have one (scale, zero) pair (group size 256), else 0
  const int *run_if, *row_flag;  // not null: run_if[0] = 1 asks for everything, 2 for the rows m with row_flag[m] only, 0 for nothing
};

// kRT row tiles of 32 per wave: 32 kRT rows x 256 columns per workgroup.  GATE: 128 columns of each of two matrices, a wave's first column tile from
// the one and its second from the other, so that a lane ends up with both products of its outputs: y = bf16( bf16(silu(bf16 a)) * bf16 b ).
template <int G, int kRT, bool GATE>
__global__ __launch_bounds__(256, 2) void int4_gemm_kernel(const GemmArgs a) {
  constexpr int kRows = 32 * kRT, kXStage = kRows * 128, kWStage = kCols * 64, kLdsW = 3 * kXStage, kLdsBytes = kLdsW + 2 * kWStage;
  static_assert(2 * kLdsBytes <= 160 * 1024, "two workgroups per CU");
  constexpr int NGRP = 128 / G, SPG = G / 16;  // groups per 128 k, MFMA steps per group
  constexpr bool kGroupSums = G == 32;         // a group's products in registers of their own, scaled when it ends
  __shared__ __attribute__((aligned(1024))) uint8_t lds[kLdsBytes];
  const int M = a.M, N = a.N, K = a.K;
  const int xcd = blockIdx.x & 7;
  const int slot = blockIdx.x >> 3;
  const int cb = xcd + 8 * (slot % a.cbx), rb = slot / a.cbx;
  if (cb >= a.n_col_blocks) return;  // grid padding; uniform, before any barrier

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, h = lane >> 5;
  constexpr int kWide = GATE ? 32 : 64;  // columns of a matrix per wave
  const int row0 = rb * kRows, col0 = cb * (4 * kWide) + kWide * wave;
  const auto column = [&](int ct) { return col0 + (GATE ? 0 : 32 * ct); };  // first one of a column tile
  const int *only = nullptr;
  if (a.run_if) {
    const int asked = *a.run_if;
    if (asked == 0) return;  // the whole grid
    if ((asked & 1) == 0) {
      int any = 0;
      for (int r = lane; r < kRows; r += 64) any |= row0 + r < M ? a.row_flag[row0 + r] : 0;
      if (__builtin_amdgcn_ballot_w64(any != 0) == 0) return;  // the whole workgroup
      only = a.row_flag;
    }
  }
  const int KT = K >> 7;
  const int blk0 = static_cast<int>((static_cast<int64_t>(KT) * blockIdx.y) / gridDim.y);
  const int blk1 = static_cast<int>((static_cast<int64_t>(KT) * (blockIdx.y + 1)) / gridDim.y);
  const int g_begin = blk0 * NGRP, g_end = blk1 * NGRP;

  const __amdgpu_buffer_rsrc_t w_rsrc = make_rsrc(a.wp, static_cast<uint32_t>(static_cast<size_t>(N) * K / 2));
  const __amdgpu_buffer_rsrc_t sz_rsrc = make_rsrc(a.sz, static_cast<uint32_t>(static_cast<size_t>((K / G) >> a.shared) * N * 4));
  const __amdgpu_buffer_rsrc_t w2_rsrc = make_rsrc(GATE ? a.wp2 : a.wp, static_cast<uint32_t>(static_cast<size_t>(N) * K / 2));
  const __amdgpu_buffer_rsrc_t sz2_rsrc = make_rsrc(GATE ? a.sz2 : a.sz, static_cast<uint32_t>(static_cast<size_t>((K / G) >> a.shared) * N * 4));
  const __amdgpu_buffer_rsrc_t x_rsrc = make_rsrc(a.x, static_cast<uint32_t>(static_cast<size_t>(M) * K * 2));
  const __amdgpu_buffer_rsrc_t xs_rsrc = make_rsrc(a.xsum, static_cast<uint32_t>(static_cast<size_t>(K / G) * a.xsum_stride * 4));

  // ---- what this lane loads: activation block wave + 4 i, row 8 (wave + 4 i) + lane / 8; weight column 16 i + lane / 4 of the wave's 64
  uint32_t xsrc[4], wsrc[4];
#pragma unroll
  for (int i = 0; i < kRT; ++i) {
    int row = row0 + 8 * (wave + 4 * i) + (lane >> 3);
    row = row < M ? row : M - 1;
    xsrc[i] = static_cast<uint32_t>((static_cast<size_t>(row) * K + ((lane & 7) ^ (((lane >> 4) + 4 * wave) & 7)) * 8) * 2);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    int col = col0 + (GATE ? 16 * (i & 1) : 16 * i) + (lane >> 2);
    col = col < N ? col : N - 1;
    wsrc[i] = static_cast<uint32_t>(static_cast<size_t>(col >> 3) * KT * 512 + (col & 7) * 64 + ((lane & 3) ^ ((lane >> 4) & 3)) * 16);
  }
  const int last_chunk = 2 * blk1 - 1;
  const auto load_x = [&](int chunk, uint32_t stage) {  // past the slice: its last chunk again, which nobody uses
    const uint32_t off = static_cast<uint32_t>(chunk < last_chunk ? chunk : last_chunk) * 128u;
#pragma unroll
    for (int i = 0; i < kRT; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(x_rsrc, (lds_void *)(lds + stage + (wave + 4 * i) * 1024), 16, xsrc[i], off, 0, 0);
  };
  const auto load_w = [&](int blk, uint32_t stage) {
    const uint32_t off = static_cast<uint32_t>(blk < blk1 - 1 ? blk : blk1 - 1) * 512u;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(GATE && i >= 2 ? w2_rsrc : w_rsrc, (lds_void *)(lds + stage + (4 * wave + i) * 1024), 16, wsrc[i], off, 0, 0);
  };
  uint32_t szlane[kCT];  // this lane's columns inside one [N] row of (scale, zero) pairs
#pragma unroll
  for (int ct = 0; ct < kCT; ++ct) {
    int col = column(ct) + n;
    col = col < N ? col : N - 1;
    szlane[ct] = static_cast<uint32_t>(col) * 4u;
  }
  const auto load_sz = [&](int ct, int g) {
    return __builtin_amdgcn_raw_buffer_load_b32(GATE && ct > 0 ? sz2_rsrc : sz_rsrc, szlane[ct], static_cast<uint32_t>((g < g_end - 1 ? g : g_end - 1) >> a.shared) * N * 4u, 0);
  };

  load_w(blk0, kLdsW);
  load_x(2 * blk0, 0);
  load_x(2 * blk0 + 1, kXStage);

  // ---- accumulators start as the zero-point term -----------------------------------------------------------------------
  f32x16_t acc[kCT][kRT];
#pragma unroll
  for (int ct = 0; ct < kCT; ++ct)
#pragma unroll
    for (int rt = 0; rt < kRT; ++rt)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[ct][rt][e] = 0.f;
  bool odd_scale = false;
  float not_finite[kRT] = {};  // NaN once this lane met a group sum of its row that is not finite
  struct Zero {
    float xs[4];
    uint32_t szw[kCT];
  };
  constexpr int kBatch = 4;  // pairs of groups per round, requested a round ahead
  const auto dead = [&](int g0) { return g0 + h < g_end ? 0u : 0x80000000u; };  // lanes with h = 1 take group g0 + 1; past the end: zeros
  const auto load_zero = [&](Zero (&z)[kBatch], int g0) {
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      const int g = g0 + 2 * i;
      const uint32_t out = dead(g), gs = static_cast<uint32_t>(g < g_end ? g : g_begin);
#pragma unroll
      for (int rt = 0; rt < kRT; ++rt) {
        const int row = row0 + 32 * rt + n;  // past M: zeros, so that nothing there overflows
        z[i].xs[rt] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xs_rsrc, row < M ? static_cast<uint32_t>(h * a.xsum_stride + row) * 4u | out : 0x80000000u,
                                                                                     gs * a.xsum_stride * 4u, 0));
      }
#pragma unroll
      for (int ct = 0; ct < kCT; ++ct)
        z[i].szw[ct] = __builtin_amdgcn_raw_buffer_load_b32(GATE && ct > 0 ? sz2_rsrc : sz_rsrc, (szlane[ct] + ((gs + h) >> a.shared) * static_cast<uint32_t>(N) * 4u) | out, 0, 0);
    }
  };
  Zero za[kBatch], zb[kBatch];
  load_zero(za, g_begin);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll 1
  for (int g0 = g_begin; g0 < g_end; g0 += 2 * kBatch) {
    load_zero(zb, g0 + 2 * kBatch);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      bf16x8_t zf[kCT];
#pragma unroll
      for (int ct = 0; ct < kCT; ++ct) {
        const float scale = __builtin_bit_cast(float, za[i].szw[ct] << 16), zero = __builtin_bit_cast(float, za[i].szw[ct] & 0xFFFF0000u);
        const bool carried = kGroupSums ? __builtin_isfinite(scale) && __builtin_isfinite(zero)
                                        : scale == 0.f || (__builtin_fabsf(scale) >= 0x1p-100f && __builtin_fabsf(scale) <= 0x1p13f);
        odd_scale |= !dead(g0 + 2 * i) && !carried;
        float p[3];
        split3(__builtin_fmaf(-24.0f, scale, zero), p);
        const uint32_t hm = high_halves(p[1], p[0]);
        zf[ct] = __builtin_bit_cast(bf16x8_t, u32x4_t{hm, hm, high_halves(p[0], p[2]), high_halves(p[1], p[2])});
      }
#pragma unroll
      for (int rt = 0; rt < kRT; ++rt) {
        float p[3];
        not_finite[rt] = __builtin_fmaf(za[i].xs[rt], 0.f, not_finite[rt]);
        split3(za[i].xs[rt], p);
        const bf16x8_t xf = __builtin_bit_cast(bf16x8_t, u32x4_t{high_halves(p[0], p[0]), high_halves(p[1], p[1]), high_halves(p[2], p[0]), high_halves(p[2], p[1])});
#pragma unroll
        for (int ct = 0; ct < kCT; ++ct) acc[ct][rt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xf, zf[ct], acc[ct][rt], 0, 0, 0);
      }
    }
#pragma unroll
    for (int i = 0; i < kBatch; ++i) za[i] = zb[i];
  }

  uint32_t odd_rows[kRT];  // bit r: row r of the tile has a value that is not finite
#pragma unroll
  for (int rt = 0; rt < kRT; ++rt) {
    const uint64_t lanes = __builtin_amdgcn_ballot_w64(!(not_finite[rt] == 0.f));
    odd_rows[rt] = static_cast<uint32_t>(lanes) | static_cast<uint32_t>(lanes >> 32);
  }

  // do all waves know the same?  (the third activation stage is free until the loop)
  uint32_t *const votes = reinterpret_cast<uint32_t *>(lds + 2 * kXStage);
  const bool odd_wave = __builtin_amdgcn_ballot_w64(odd_scale) != 0;
  if (lane == 0) votes[wave] = odd_wave;
  lds_barrier();
  bool plain = __builtin_amdgcn_readfirstlane(votes[0] | votes[1] | votes[2] | votes[3]) != 0;
  if (!plain) {
    // ---- fragments: activation (row tile rt, step s): row 32 rt + n, piece 2 s + h; weights (column tile ct): pieces j of column 32 ct + n
    uint32_t a_lane[4], w_lane[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) a_lane[s] = static_cast<uint32_t>(n * 128 + (((2 * s + h) ^ ((n >> 1) & 7)) << 4));
#pragma unroll
    for (int j = 0; j < 4; ++j) w_lane[j] = static_cast<uint32_t>(wave * 4096 + n * 64 + ((j ^ ((n >> 2) & 3)) << 4));
    bf16x8_t af[2][kRT], wf[2][kCT];
    u32x4_t wq[kCT][4];
    const auto read_a = [&](bf16x8_t (&f)[kRT], uint32_t stage, int s) {
#pragma unroll
      for (int rt = 0; rt < kRT; ++rt) f[rt] = *reinterpret_cast<const bf16x8_t *>(lds + stage + a_lane[s] + rt * 4096);
    };
    const auto read_w = [&](uint32_t stage) {
#pragma unroll
      for (int ct = 0; ct < kCT; ++ct)
#pragma unroll
        for (int j = 0; j < 4; ++j) wq[ct][j] = *reinterpret_cast<const u32x4_t *>(lds + stage + w_lane[j] + ct * 2048);
    };
    // registers, so that each pair of codes is one and-or; per column, both zero where a group's scale is zero: it adds nothing
    uint32_t mask[kCT], magic[kCT];
    if constexpr (kGroupSums) {
      asm volatile("s_mov_b32 %0, 0x00780078" : "=s"(mask[0]));
      asm volatile("v_mov_b32 %0, 0x41804180" : "=v"(magic[0]));
      mask[1] = mask[0];
      magic[1] = magic[0];
    }
    const auto enter = [&](int ct, uint32_t pair) {
      if constexpr (!kGroupSums) {
        const bool live = (pair & 0x7FFFu) != 0;
        mask[ct] = live ? 0x00780078u : 0u;
        magic[ct] = live ? 0x41804180u : 0u;
        asm volatile("" : "+v"(mask[ct]), "+v"(magic[ct]));  // no select behind every pair
      }
    };
    const uint32_t rot0 = (4 * h - 3) & 31, rot1 = (4 * h + 5) & 31;
    const auto convert = [&](bf16x8_t (&f)[kCT], int s8) {
#pragma unroll
      for (int ct = 0; ct < kCT; ++ct) {
        u32x4_t u;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const uint32_t w = wq[ct][j][s8 >> 1];
          u[j] = (__builtin_amdgcn_alignbit(w, w, s8 & 1 ? rot1 : rot0) & mask[ct]) | magic[ct];
        }
        f[ct] = __builtin_bit_cast(bf16x8_t, u);
      }
    };

    float unit[kCT] = {1.f, 1.f};  // what one step of the accumulators is worth (group sums: the group's scale)
    [[maybe_unused]] f32x16_t part[kCT][kGroupSums ? kRT : 1];
    constexpr int kSc = NGRP < 2 ? NGRP : 2;  // pairs held ahead
    uint32_t sc[kCT][kSc];
#pragma unroll
    for (int ct = 0; ct < kCT; ++ct)
#pragma unroll
      for (int g = 0; g < kSc; ++g) sc[ct][g] = load_sz(ct, g_begin + g);
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    asm volatile("s_barrier" ::: "memory");
    read_w(kLdsW);
    read_a(af[0], 0, 0);
#pragma unroll
    for (int ct = 0; ct < kCT; ++ct) enter(ct, sc[ct][0]);
    convert(wf[0], 0);
    uint32_t s0 = 0, s1 = kXStage, s2 = 2 * kXStage;  // stage of the chunk in use, of the next one, of the one after
    uint32_t w_next = kLdsW + kWStage;

    for (int blk = blk0; blk < blk1; ++blk) {
      load_w(blk + 1, w_next);
      load_x(2 * blk + 2, s2);
#pragma unroll
      for (int s8 = 0; s8 < 8; ++s8) {
        const int cur = s8 & 1;
        if (s8 == 4) load_x(2 * blk + 3, s0);  // every wave left that stage at the barrier below
        // The second chunk is in: loads issued after it are this block's words, its next chunk and the scale pairs of the last half block of each kind.  The
        // next block's words and first chunk are in: after them came one chunk and this block's scale pairs.
        if (s8 == 3) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(4 + kRT + (NGRP == 1 ? 2 : 2 * NGRP)) : "memory");
        if (s8 == 7) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kRT + 2 * NGRP) : "memory");
        if (s8 == 7) read_w(w_next);
        if (!kGroupSums) __builtin_amdgcn_sched_barrier(0);  // the counts of the waits above hold for this order of loads
        read_a(af[cur ^ 1], s8 < 3 ? s0 : s8 < 7 ? s1 : s2, (s8 + 1) & 3);
        if (kGroupSums) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ct = 0; ct < kCT; ++ct) {
          float r = 1.f;
          if (s8 % SPG == 0) {
            const float scale = __builtin_bit_cast(float, sc[ct][s8 / SPG % kSc] << 16), s = kGroupSums || scale != 0.f ? scale : unit[ct];
            if (!kGroupSums) r = quotient(unit[ct], s);
            unit[ct] = s;
            sc[ct][s8 / SPG % kSc] = load_sz(ct, blk * NGRP + s8 / SPG + kSc);
          }
#pragma unroll
          for (int rt = 0; rt < kRT; ++rt) {
            if constexpr (kGroupSums) {
              part[ct][rt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[cur][rt], wf[cur][ct], s8 % SPG == 0 ? f32x16_t{} : part[ct][rt], 0, 0, 0);
            } else {
              if (s8 % SPG == 0) {
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[ct][rt][e] *= r;
              }
              acc[ct][rt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[cur][rt], wf[cur][ct], acc[ct][rt], 0, 0, 0);
            }
          }
        }
        if constexpr (kGroupSums)
          if ((s8 + 1) % SPG == 0)
#pragma unroll
            for (int ct = 0; ct < kCT; ++ct)
#pragma unroll
              for (int rt = 0; rt < kRT; ++rt)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[ct][rt][e] = __builtin_fmaf(unit[ct], part[ct][rt][e], acc[ct][rt][e]);
        if ((s8 + 1) % SPG == 0)
#pragma unroll
          for (int ct = 0; ct < kCT; ++ct) enter(ct, sc[ct][(s8 + 1) % 8 / SPG % kSc]);
        convert(wf[cur ^ 1], (s8 + 1) & 7);
        // A product takes 32 clocks and leaves its wave's vector unit free.  Left to itself the compiler issues a step's products in a
        // row and its vector work behind them, so a wave pays for both; in this order (entering a group first, then a product, an LDS
        // read, three vector instructions) most of the unpacking runs under the products.  With the 96-row form
        // 471 x 12288 x 4096, group size 128, went from 69 to 58 us.
        if constexpr (!kGroupSums) {
#pragma unroll
          for (int i = 0; i < kCT * kRT; ++i) {
            if (s8 % SPG == 0) __builtin_amdgcn_sched_group_barrier(0x2, 16, 0);
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
            if (s8 == 7) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            else __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x2, 3, 0);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      const uint32_t t = s0;  // two chunks on
      s0 = s2;
      s2 = s1;
      s1 = t;
      w_next ^= kLdsW ^ (kLdsW + kWStage);
    }
    // the loads issued past the last block still write LDS: drain them before the stages are reused
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    // Is a sum not finite in its column's units?  A row whose x is not finite stays out: nothing could make it so.
    bool over = false;
#pragma unroll
    for (int rt = 0; rt < (kGroupSums ? 0 : kRT); ++rt) {
#pragma unroll
      for (int ct = 0; ct < kCT; ++ct) {
        float t[2] = {0.f, 0.f};  // zero times an infinity or a NaN is a NaN
        if (odd_rows[rt] == 0) {
#pragma unroll
          for (int e = 0; e < 16; ++e) t[e & 1] = __builtin_fmaf(acc[ct][rt][e], 0.f, t[e & 1]);
        } else {
          const uint32_t mine = odd_rows[rt] >> (4 * h);
#pragma unroll
          for (int e = 0; e < 16; ++e) t[e & 1] = __builtin_fmaf(mine >> (8 * (e >> 2) + (e & 3)) & 1 ? 0.f : acc[ct][rt][e], 0.f, t[e & 1]);
        }
        over |= !(t[0] + t[1] == 0.f);
      }
    }
    plain = __builtin_amdgcn_ballot_w64(over) != 0;
    if (!plain) {
#pragma unroll
      for (int ct = 0; ct < (kGroupSums ? 0 : kCT); ++ct)
#pragma unroll
        for (int rt = 0; rt < kRT; ++rt)
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[ct][rt][e] *= unit[ct];

      // ---- store: lane (h, n) holds column col0 + 32 ct + n, rows 8 (e / 4) + 4 h + e % 4 of each tile -----------
      if (a.partials) {
        float *out = a.partials + static_cast<size_t>(blockIdx.y) * M * N;
#pragma unroll
        for (int ct = 0; ct < kCT; ++ct) {
          const int col = column(ct) + n;
          if (col >= N) continue;
#pragma unroll
          for (int rt = 0; rt < kRT; ++rt)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
              const int m = row0 + 32 * rt + 8 * (e >> 2) + 4 * h + (e & 3);
              if (m < M) out[static_cast<size_t>(m) * N + col] = acc[ct][rt][e];
            }
        }
        return;
      }
      int late = lane;
      asm volatile("" : "+v"(late));  // keeps the rows' addresses out of the registers of the main loop (the 128-row form of group size 64 would spill two)
      const bool pieces = (N & 7) == 0 && (reinterpret_cast<uintptr_t>(a.y) & 15) == 0;
      if constexpr (GATE) {
        const float no_scale[1] = {};
        uint8_t *const tile = lds + wave * TileStore<1>::kBytesPerWave;
#pragma unroll
        for (int rt = 0; rt < kRT; ++rt) {
          f32x16_t out[1][1];
#pragma unroll
          for (int e = 0; e < 16; ++e) out[0][0][e] = gated(acc[0][rt][e], acc[1][rt][e]);
          store_tiles_via_lds<1, 1, false>(out, no_scale, tile, a.y, row0 + 32 * rt, col0, M, N, late, pieces, only);
        }
      } else {
        const float no_scale[kCT] = {};
        store_tiles_via_lds<kRT, kCT, false>(acc, no_scale, lds + wave * TileStore<kCT>::kBytesPerWave, a.y, row0, col0, M, N, late, pieces, only);
      }
      return;
    }
  }

  // Every group's sum by itself, two row tiles at a time, operands straight from memory, nothing shared with the other waves.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the first loads still write LDS
  [[maybe_unused]] f32x16_t first[2];
#pragma unroll 1
  for (int t = 0; t < kCT * ((kRT + 1) / 2); ++t) {  // (gated: the two tiles of the same outputs after each other)
    const bool second = GATE && (t & 1);
    int r0 = row0 + 64 * (t / kCT);
    asm volatile("" : "+s"(r0));  // keeps the addresses of all rows out of the registers of the loops
    int col = column(t % kCT) + n;
    const bool live = col < N;
    col = live ? col : N - 1;
    const uint32_t wo = static_cast<uint32_t>(static_cast<size_t>(col >> 3) * KT * 512 + (col & 7) * 64);
    uint32_t xo[2];
    f32x16_t sum[2] = {};
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      const int row = r0 + 32 * rt + n;
      xo[rt] = static_cast<uint32_t>(static_cast<size_t>(row < M ? row : M - 1) * K * 2) + 16u * h;
    }
#pragma unroll 1
    for (int g = g_begin; g < g_end; ++g) {
      f32x16_t part[2] = {};
#pragma unroll 4
      for (int s = 0; s < SPG; ++s) {
        const int step = g * SPG + s;  // of 16 k
        u32x4_t u;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const uint32_t w = __builtin_amdgcn_raw_buffer_load_b32(second ? w2_rsrc : w_rsrc, wo + 16u * j, static_cast<uint32_t>(step >> 3) * 512u + ((step >> 1) & 3) * 4u, 0);
          u[j] = (__builtin_amdgcn_alignbit(w, w, (8 * (step & 1) + 4 * h - 3) & 31) & 0x00780078u) | 0x41804180u;
        }
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
          const bf16x8_t xf = __builtin_bit_cast(bf16x8_t, __builtin_amdgcn_raw_buffer_load_b128(x_rsrc, xo[rt], static_cast<uint32_t>(step) * 32u, 0));
          part[rt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xf, __builtin_bit_cast(bf16x8_t, u), part[rt], 0, 0, 0);
        }
      }
      const uint32_t szw = __builtin_amdgcn_raw_buffer_load_b32(second ? sz2_rsrc : sz_rsrc, static_cast<uint32_t>(col) * 4u, static_cast<uint32_t>(g >> a.shared) * N * 4u, 0);
      const float scale = __builtin_bit_cast(float, szw << 16), zero = __builtin_bit_cast(float, szw & 0xFFFF0000u);
      const float zc = __builtin_fmaf(-24.0f, scale, zero);
#pragma unroll
      for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int q = 0; q < 4; ++q) {  // rows 8 q + 4 h .. + 3 of the tile
          const f32x4_t xg = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(xs_rsrc, static_cast<uint32_t>(r0 + 32 * rt + 8 * q + 4 * h) * 4u,
                                                                                              static_cast<uint32_t>(g) * a.xsum_stride * 4u, 0));
#pragma unroll
          for (int e = 0; e < 4; ++e) sum[rt][4 * q + e] = __builtin_fmaf(zc, xg[e], __builtin_fmaf(scale, part[rt][4 * q + e], sum[rt][4 * q + e]));
        }
    }
    if (GATE && !second) {
      first[0] = sum[0];
      first[1] = sum[1];
      continue;
    }
    if (!live) continue;
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int m = r0 + 32 * rt + 8 * (e >> 2) + 4 * h + (e & 3);
        if (m >= M || m >= row0 + kRows || (only && !only[m])) continue;
        if (a.partials) a.partials[(static_cast<size_t>(blockIdx.y) * M + m) * N + col] = sum[rt][e];
        else a.y[static_cast<size_t>(m) * N + col] = f32_to_bf16_rne(GATE ? gated(first[rt][e], sum[rt][e]) : sum[rt][e]);
      }
  }
}

constexpr int kMostSlices = 8;

// y = bf16(sum over the K slices), a balanced tree in the order of K; four columns per thread (N % 8 == 0)
__global__ __launch_bounds__(256) void add_slices_kernel(const float *__restrict__ partials, uint16_t *__restrict__ y, int64_t quads, int64_t slice, int S) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= quads) return;
  f32x4_t v[kMostSlices];
#pragma unroll
  for (int s = 0; s < kMostSlices; ++s) v[s] = s < S ? *reinterpret_cast<const f32x4_t *>(partials + s * slice + 4 * i) : f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int step = 1; step < kMostSlices; step *= 2)
#pragma unroll
    for (int s = 0; s < kMostSlices; s += 2 * step) v[s] += v[s + step];
#pragma unroll
  for (int j = 0; j < 4; ++j) y[4 * i + j] = f32_to_bf16_rne(v[0][j]);
}

}  // namespace

// Time of a whole call in us, group sums of x included, within 3 to 5 % (one standard deviation) of 9600 measured calls of 27 shapes, 65 to 2600 rows: a workgroup of 64, 96 or 128 rows
// takes `one` per 128 k when it has its CU to itself and two that share a CU take `two`; slices what their sums cost to write and add.
double expected_us(int M, int N, int KT, int groupsize, int rows, int slices) {
  constexpr double kOne32[] = {1.81}, kTwo32[] = {2.69}, kOne64[] = {1.42, 1.74, 2.06}, kTwo64[] = {2.18, 2.8, 3.55}, kOne128[] = {1.1, 1.37, 1.65}, kTwo128[] = {1.85, 2.36, 3.08};
  constexpr double kCall[] = {7.75, 8.7, 9.8}, kSlices[] = {2.6, 3.2, 3.6}, kSlice[] = {0.13, 0.25, 0.25}, kSum[] = {2.06e-6, 1.55e-6, 1.47e-6};
  const int r = rows / 32 - 2;
  const double one = (groupsize == 32 ? kOne32 : groupsize == 64 ? kOne64 : kOne128)[r], two = (groupsize == 32 ? kTwo32 : groupsize == 64 ? kTwo64 : kTwo128)[r];
  const int64_t per_cu = (static_cast<int64_t>((M + rows - 1) / rows) * (((N + kCols - 1) / kCols + 7) / 8) * slices + 31) / 32;
  return (static_cast<double>(per_cu / 2) * two + (per_cu & 1 ? one : 0)) * KT / slices + kCall[r] +
         (slices > 1 ? kSlices[r] + slices * (kSlice[r] + kSum[r] * static_cast<double>(M) * N) : 0);
}

// Rows per workgroup and K slices by the least cost in us of the product alone, from what was measured at 65 .. 8192 rows of the 7B and 34B shapes:
// a workgroup takes `one` per 128 k when it has its CU to itself and two that share a CU take `two` (64 rows: 1.2 and 1.95, 96 rows:
// 1.47 and 2.42, 128 rows: 1.85 and 3.3), a call 3 more, and slices what their sums cost to write and add.  128 rows win once the chip is full (8192 x 12288 x 4096:
// 688 us, 64 rows 795), 64 rows with one slice or several below (471 x 4096 x 4096: two slices 34 us, one 41, 128 rows 63).
Int4GemmShape int4_gemm_shape(int M, int N, int K, int groupsize, int64_t scratch_bytes) {
  const int KT = K >> 7;
  const int64_t fit = scratch_bytes / (static_cast<int64_t>(M) * N * 4);
  const int want_rows = options().int4_gemm_tile, most = options().int4_k_slices > 0 ? options().int4_k_slices : kMostSlices;
  const auto possible = [&](int s) { return s <= kMostSlices && s <= KT && s <= most && (s == 1 || s <= fit); };
  int forced = 0;  // the option's count, or the largest one below it that there is
  if (options().int4_k_slices > 0)
    for (int s = 1; possible(s); s *= 2) forced = s;
  Int4GemmShape best = {64, 1, -1.0};
  double least = -1;
  for (int rows = 64; rows <= (groupsize == 32 ? 64 : 128); rows += 32) {
    // group size 32 at 128 rows does not fit the registers
    if ((want_rows == 96 || want_rows == 128) && groupsize != 32 && rows != want_rows) continue;
    const int64_t per_xcd = static_cast<int64_t>((M + rows - 1) / rows) * (((N + kCols - 1) / kCols + 7) / 8);  // one slice; 32 CUs each
    for (int s = 1; possible(s); s *= 2) {
      if (forced && s != forced) continue;
      const int64_t per_cu = (per_xcd * s + 31) / 32;
      const double one = rows == 64 ? 1.2 : rows == 96 ? 1.47 : 1.85, two = rows == 64 ? 1.95 : rows == 96 ? 2.42 : 3.3;
      const double cost = (static_cast<double>(per_cu / 2) * two + (per_cu & 1 ? one : 0)) * KT / s + 3 +
                          (s > 1 ? 4 + s * (0.6 + 0.9e-6 * static_cast<double>(M) * N) : 0);
      if (least < 0 || cost < least) {
        least = cost;
        best = Int4GemmShape{rows, s, expected_us(M, N, KT, groupsize, rows, s)};
      }
    }
  }
  return best;
}

template <int G, bool GATE>
void launch_gemm(const GemmArgs &a, int rows, dim3 grid, hipStream_t stream) {
  if constexpr (G != 32) {
    if (rows != 64) {
      if (rows == 128) hipLaunchKernelGGL((int4_gemm_kernel<G, 4, GATE>), grid, dim3(256), 0, stream, a);
      else hipLaunchKernelGGL((int4_gemm_kernel<G, 3, GATE>), grid, dim3(256), 0, stream, a);
      return;
    }
  }
  hipLaunchKernelGGL((int4_gemm_kernel<G, 2, GATE>), grid, dim3(256), 0, stream, a);
}

template <bool GATE>
int launch_gemm(const GemmArgs &args, int groupsize, Int4GemmShape shape, hipStream_t stream) {
  GemmArgs a = args;
  const int wide = GATE ? kCols / 2 : kCols;
  a.n_col_blocks = (a.N + wide - 1) / wide;
  a.cbx = (a.n_col_blocks + 7) / 8;
  const long long wgs = 8LL * a.cbx * ((a.M + shape.rows - 1) / shape.rows);
  if (wgs > 0x7FFFFFFFLL) return E2H_ERR_BAD_SHAPE;
  const dim3 grid(static_cast<unsigned>(wgs), static_cast<unsigned>(shape.slices));
  switch (groupsize) {
    case 32: launch_gemm<32, GATE>(a, shape.rows, grid, stream); break;
    case 64: launch_gemm<64, GATE>(a, shape.rows, grid, stream); break;
    case 128: launch_gemm<128, GATE>(a, shape.rows, grid, stream); break;
    default: return E2H_ERR_BAD_GROUPSIZE;
  }
  return E2H_OK;
}

int int4_gemm(const uint16_t *x, const int32_t *packed, const uint16_t *sz, uint16_t *y, const float *xsum, int xsum_stride,
              float *partials, Int4GemmShape shape, int M, int N, int K, int groupsize, hipStream_t stream, const int *run_if, const int *row_flag) {
  if (K % 128 != 0 || N % 8 != 0) return E2H_ERR_BAD_SHAPE;
  const int shared = groupsize == 256;
  if (shared) groupsize = 128;
  const GemmArgs a = {x, reinterpret_cast<const uint32_t *>(packed), reinterpret_cast<const uint32_t *>(sz), nullptr, nullptr, y, shape.slices > 1 ? partials : nullptr,
                      xsum, xsum_stride, M, N, K, 0, 0, shared, run_if, row_flag};
  const int rc = launch_gemm<false>(a, groupsize, shape, stream);
  if (rc != E2H_OK) return rc;
  if (shape.slices > 1 && y) {
    const int64_t quads = static_cast<int64_t>(M) * N / 4;
    hipLaunchKernelGGL(add_slices_kernel, dim3(static_cast<unsigned>((quads + 255) / 256)), dim3(256), 0, stream, partials, y, quads,
                       static_cast<int64_t>(M) * N, shape.slices);
  }
  return launch_status();
}

int int4_gemm_gate(const uint16_t *x, const int32_t *packed, const uint16_t *sz, const int32_t *packed2, const uint16_t *sz2, uint16_t *y, const float *xsum,
                   int xsum_stride, Int4GemmShape shape, int M, int N, int K, int groupsize, hipStream_t stream, const int *run_if, const int *row_flag) {
  if (K % 128 != 0 || N % 8 != 0 || shape.slices != 1) return E2H_ERR_BAD_SHAPE;
  const int shared = groupsize == 256;
  const GemmArgs a = {x, reinterpret_cast<const uint32_t *>(packed), reinterpret_cast<const uint32_t *>(sz), reinterpret_cast<const uint32_t *>(packed2),
                      reinterpret_cast<const uint32_t *>(sz2), y, nullptr, xsum, xsum_stride, M, N, K, 0, 0, shared, run_if, row_flag};
  const int rc = launch_gemm<true>(a, shared ? 128 : groupsize, shape, stream);
  return rc != E2H_OK ? rc : launch_status();
}

}  // namespace e2h

namespace e2h {
int64_t int4_unpacked_bytes(int64_t M, int64_t N, int64_t K, int groupsize, int inner_k_tiles);
int64_t int4_gate_unpacked_bytes(int64_t M, int64_t N, int64_t K, int groupsize, int inner_k_tiles);
int int4_unpacked_gate(const uint16_t *x, const int32_t *packed, const uint16_t *sz, const int32_t *packed2, const uint16_t *sz2, uint16_t *y, int M, int N, int K, int groupsize,
                       void *scratch, hipStream_t stream);
constexpr int kUnpackRows = 1024;  // from here on callers offer memory for unpacked operands

// Scratch of a gated call: for unpacked operands (int4_gate_unpacked_bytes) or the group sums of x; or 0 where two calls of the 32x32-tile kernel and a pass that multiplies are expected to be no slower or a form is asked for by an
// option.  The launch of both matrices has twice the workgroups, spares one pass over x for its group sums, the two products' way to memory and back, and a launch.
int64_t int4_gate_rows_bytes(int64_t M, int64_t N, int64_t K, int groupsize, int inner_k_tiles) {
  if (inner_k_tiles != 8 || (groupsize != 32 && groupsize != 64 && groupsize != 128 && groupsize != 256)) return 0;
  if (M <= 64 || N < 8 || N % 8 != 0 || K < 128 || K % 128 != 0 || K % groupsize != 0 || M > INT32_MAX / 64 || N > INT32_MAX / 64 || K > INT32_MAX / 64) return 0;
  if (M * K * 2 >= (int64_t{1} << 32) || N * K / 2 >= (int64_t{1} << 32) || K / groupsize * N * 4 >= (int64_t{1} << 32)) return 0;
  const int G = groupsize == 256 ? 128 : groupsize;
  const int64_t bytes = K / G * ((M + 63) / 64 * 64) * 4;
  if (bytes >= (int64_t{1} << 32)) return 0;
  const Options &o = options();
  if (o.int4_no_gemm32 || o.int4_gemm_tile || o.int4_gemm32_min_rows || o.int4_no_xsum || o.int4_k_slices || o.int4_rows_per_wave || o.row_tiles) return 0;
  const int m = static_cast<int>(M), n = static_cast<int>(N), k = static_cast<int>(K);
  if (const int64_t unpacked = int4_gate_unpacked_bytes(M, N, K, groupsize, inner_k_tiles)) return unpacked;
  if (M >= kUnpackRows && int4_unpacked_bytes(M, N, K, groupsize, inner_k_tiles) > 0) return 0;
  const double calls = 2 * int4_gemm_shape(m, n, k, G, int64_t{32} << 20).us + 3 + static_cast<double>(M) * static_cast<double>(N) * 6 / 5e6;  // the pass moves six bytes an output
  return 1.07 * int4_gemm_shape(m, 2 * n, k, G, 0).us < calls ? bytes : 0;
}

// Whether a model's calls gain by it: sizes that are taken, beside calls of whichever kernel they would run (small weights, of group size 256 above all: the one of 16 x 16 tiles).  The
// gated launch takes 5 us and a tenth more than expected of a product of both widths.  Measured, us, two calls and the pass / here: 2 x 11008 x 4096 g128 65 rows 61 / 54, 128 rows
// 72 / 51, 471 rows 117 / 97, 1500 rows 298 / 273; g64 471 rows 141 / 112; 2 x 5504 x 2048 g128 256 rows 51 / 31; left to the calls: 2 x 2816 x 1024 g256 72 rows 17 / 21, 2 x 2048 x 4096
// g256 192 rows 35 / 47, 2 x 1024 x 512 g256 192 rows 15 / 16.  Of 834 shapes and rows (65 .. 4096) that are taken 779 pay, 19 % less on average and 3 % more at most; the other 55 would
// take up to 34 % more and none 2 % less.
bool int4_gate_rows_pay(int64_t M, int64_t N, int64_t K, int groupsize, int inner_k_tiles) {
  if (int4_gate_rows_bytes(M, N, K, groupsize, inner_k_tiles) == 0) return false;
  if (int4_gate_unpacked_bytes(M, N, K, groupsize, inner_k_tiles) > 0) return true;
  const int G = groupsize == 256 ? 128 : groupsize, m = static_cast<int>(M), n = static_cast<int>(N), k = static_cast<int>(K);
  double call = int4_gemm_shape(m, n, k, G, int64_t{32} << 20).us;
  if (groupsize == 256 || (M + 127) / 128 * ((N + 127) / 128) < 320) {  // as e2h_int4_mm chooses
    const int tiles = groupsize != 256 && (N + 127) / 128 * ((M + 63) / 64) >= 256 ? 2 : 1;
    call = std::min(call, int4_rows_us(m, n, k, groupsize, tiles));
  }
  return 1.03 * int4_gemm_shape(m, 2 * n, k, G, 0).us + 6 < 2 * call + 3 + static_cast<double>(M) * static_cast<double>(N) * 6 / 5e6;
}

// The K slices of e2h_int4_mm_rows, 0 where it takes no such call: 65 to 1023 rows that e2h_int4_mm, given a workspace of the usual size, would run on this file's kernel, with the same
// rows per workgroup and slices.
Int4GemmShape int4_rows_shape(int64_t m, int64_t n, int64_t k, int groupsize, int inner_k_tiles) {
  const Int4GemmShape none = {0, 0, 0.};
  if (inner_k_tiles != 8 || (groupsize != 32 && groupsize != 64 && groupsize != 128 && groupsize != 256)) return none;
  if (m <= 64 || m >= kUnpackRows || n < 8 || n % 8 != 0 || k < 128 || k % 128 != 0 || k % groupsize != 0 || n > INT32_MAX / 64 || k > INT32_MAX / 64) return none;
  if (m * k * 2 >= (int64_t{1} << 32) || n * k / 2 >= (int64_t{1} << 32) || k / groupsize * n * 4 >= (int64_t{1} << 32)) return none;
  const Options &o = options();
  if (o.int4_no_gemm32 || o.int4_gemm_tile || o.int4_gemm32_min_rows || o.int4_no_xsum || o.int4_k_slices || o.int4_rows_per_wave || o.int4_k_groups || o.int4_col_waves || o.row_tiles)
    return none;
  const int M = static_cast<int>(m), N = static_cast<int>(n), K = static_cast<int>(k), G = groupsize == 256 ? 128 : groupsize;
  const Int4GemmShape shape = int4_gemm_shape(M, N, K, G, (int64_t{32} << 20) - k / G * ((m + 63) / 64 * 64) * 4);
  if (groupsize != 256 && (m + 127) / 128 * ((n + 127) / 128) >= 320) return shape;
  const int tiles = groupsize != 256 && (N + 127) / 128 * ((M + 63) / 64) >= 256 ? 2 : 1;
  return shape.us < int4_rows_us(M, N, K, groupsize, tiles) ? shape : none;
}
}  // namespace e2h

extern "C" int e2h_int4_mm_rows_slices(int64_t m, int64_t n, int64_t k, int groupsize, int inner_k_tiles) {
  return e2h::int4_rows_shape(m, n, k, groupsize, inner_k_tiles).slices;
}

extern "C" int e2h_int4_mm_rows(const uint16_t *x, const int32_t *packed, const uint16_t *scales_and_zeros, float *sums, int sums_there, uint16_t *y, float *partials, int64_t m, int64_t n,
                                int64_t k, int groupsize, int inner_k_tiles, void *stream) {
  using namespace e2h;
  if (!x || !packed || !scales_and_zeros || !sums) return E2H_ERR_NULL_POINTER;
  const Int4GemmShape shape = int4_rows_shape(m, n, k, groupsize, inner_k_tiles);
  if (shape.slices == 0) return E2H_ERR_BAD_SHAPE;
  if (shape.slices > 1 ? !partials : !y) return E2H_ERR_NULL_POINTER;
  if (!aligned16(x) || !aligned16(packed) || !aligned16(scales_and_zeros) || !aligned16(sums) || !aligned16(partials) || (reinterpret_cast<uintptr_t>(y) & 7u)) return E2H_ERR_MISALIGNED;
  const int M = static_cast<int>(m), N = static_cast<int>(n), K = static_cast<int>(k), stride = (M + 63) / 64 * 64;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (!sums_there) {
    const int rc = launch_x_group_sums(x, sums, M, K, stride, groupsize == 256 ? 128 : groupsize, s);
    if (rc != E2H_OK) return rc;
  }
  return int4_gemm(x, packed, scales_and_zeros, y, sums, stride, partials, shape, M, N, K, groupsize, s);
}

extern "C" int64_t e2h_int4_mm_silu_gate_rows_scratch_bytes(int64_t m, int64_t n, int64_t k, int groupsize, int inner_k_tiles) {
  return e2h::int4_gate_rows_bytes(m, n, k, groupsize, inner_k_tiles);
}

extern "C" int e2h_int4_mm_silu_gate_rows_pays(int64_t m, int64_t n, int64_t k, int groupsize, int inner_k_tiles) {
  return e2h::int4_gate_rows_pay(m, n, k, groupsize, inner_k_tiles);
}

namespace e2h {
namespace {
int gate_rows(const uint16_t *x, const int32_t *packed_gate, const uint16_t *sz_gate, const int32_t *packed_up, const uint16_t *sz_up, uint16_t *y, int64_t m, int64_t n, int64_t k,
              int groupsize, int inner_k_tiles, void *scratch, int64_t scratch_bytes, bool sums_there, void *stream) {
  if (!x || !packed_gate || !sz_gate || !packed_up || !sz_up || !y || !scratch) return E2H_ERR_NULL_POINTER;
  if (groupsize != 32 && groupsize != 64 && groupsize != 128 && groupsize != 256) return E2H_ERR_BAD_GROUPSIZE;
  if (inner_k_tiles != 8) return E2H_ERR_BAD_INNER_K_TILES;
  const int64_t need = int4_gate_rows_bytes(m, n, k, groupsize, inner_k_tiles);
  if (need == 0) return E2H_ERR_BAD_SHAPE;
  if (scratch_bytes < need) return E2H_ERR_SCRATCH_TOO_SMALL;
  if (!aligned16(x) || !aligned16(packed_gate) || !aligned16(sz_gate) || !aligned16(packed_up) || !aligned16(sz_up) || !aligned16(scratch) ||
      (reinterpret_cast<uintptr_t>(y) & 1u))
    return E2H_ERR_MISALIGNED;
  const int M = static_cast<int>(m), N = static_cast<int>(n), K = static_cast<int>(k), G = groupsize == 256 ? 128 : groupsize, stride = (M + 63) / 64 * 64;
  if (aligned16(y) && int4_gate_unpacked_bytes(m, n, k, groupsize, inner_k_tiles) > 0)
    return sums_there ? E2H_ERR_BAD_SHAPE
                      : int4_unpacked_gate(x, packed_gate, sz_gate, packed_up, sz_up, y, M, N, K, groupsize, scratch, static_cast<hipStream_t>(stream));
  float *xsum = static_cast<float *>(scratch);
  const int rc = sums_there ? E2H_OK : launch_x_group_sums(x, xsum, M, K, stride, G, static_cast<hipStream_t>(stream));
  if (rc != E2H_OK) return rc;
  return int4_gemm_gate(x, packed_gate, sz_gate, packed_up, sz_up, y, xsum, stride, int4_gemm_shape(M, 2 * N, K, G, 0), M, N, K, groupsize,
                        static_cast<hipStream_t>(stream));
}
}  // namespace
}  // namespace e2h

extern "C" int e2h_int4_mm_silu_gate_rows(const uint16_t *x, const int32_t *packed_gate, const uint16_t *sz_gate, const int32_t *packed_up, const uint16_t *sz_up,
                                          uint16_t *y, int64_t m, int64_t n, int64_t k, int groupsize, int inner_k_tiles, void *scratch, int64_t scratch_bytes,
                                          void *stream) {
  return e2h::gate_rows(x, packed_gate, sz_gate, packed_up, sz_up, y, m, n, k, groupsize, inner_k_tiles, scratch, scratch_bytes, false, stream);
}

extern "C" int e2h_int4_mm_silu_gate_rows_sums(const uint16_t *x, const int32_t *packed_gate, const uint16_t *sz_gate, const int32_t *packed_up, const uint16_t *sz_up,
                                               uint16_t *y, int64_t m, int64_t n, int64_t k, int groupsize, int inner_k_tiles, void *sums, int64_t sums_bytes, void *stream) {
  return m >= e2h::kUnpackRows ? E2H_ERR_BAD_SHAPE
                               : e2h::gate_rows(x, packed_gate, sz_gate, packed_up, sz_up, y, m, n, k, groupsize, inner_k_tiles, sums, sums_bytes, true, stream);
}
