// int4 group-wise dequant GEMV for decode batches (M <= 64) on activations handed over in matrix-core operand order.
//
// Replaces torch.ops.aten._weight_int4pack_mm as called by linear_forward_int4 (reference models/quantize.py:445-453)
// for the one-token-per-sequence steps of the decode loop (reference inference_generate.py:123-157), where every
// quantized linear is a stream over its weights with a few rows of activations.  The activations arrive "staged"
// (layout in e2h_staged.h), written by e2h_int4_stage_x or directly by the kernel that produces them.
//
// Arithmetic per output: y[m,n] = sum_g s[g,n] * P[m,n,g] + sum_g (z[g,n] - 136 s[g,n]) * X[m,g] with
// P = sum_k x[m,k] (128 + q[n,k]) over the group (exact products, float32 accumulation in the matrix cores) and X the
// group sum of x taken from the staged buffer.  The second sum is a small float32 matrix product over the groups
// (v_mfma_f32_16x16x4_f32, four groups per instruction).
//
// Decomposition: a workgroup is eight waves (four, two workgroups on a CU, where there is more than a round of them) that split K (each wave a contiguous run of
// 128-wide chunks of the workgroup's K slice)
// and all work on the same T tiles of 16 weight rows and on all rows of the batch, so that weights are read once (small weights beside 33
// and more rows: on half of them, see plan).  No wave shares anything with another until the end.  The waves' partial tiles meet in LDS; wave w adds and finishes the (column tile, row
// tile) units w, w + 8, .. (w + 4, ..) in a fixed order, so results are deterministic; the order of a sum follows from the number of waves and the chunk they begin with, which
// another epilogue of the same weights may have otherwise (a gated launch has twice the tiles of a plain one).  S workgroups may split K further (partial epilogue
// only): their float32 sums go to slice s of a [S][M][N] array for the consumer to add in slice order.
//
// What a wave needs passes in units of 1 KB through a ring of its own in LDS, written by loads that touch no register: per chunk the
// packed words of T tiles, their (scale, zero) pairs, then the activation operands 32 k at a time.  A unit is 16 rows of four 16-byte
// pieces, placed in an order (turned below) that keeps the four lanes of a request on one 64-byte segment and the
// operand reads free of bank conflicts.  Units move from the ring into registers as they land and their places are refilled at once, so
// 16 KB per wave are on their way while the matrix cores work on a group.  Waits count loads; there is no barrier in the loop.
//
// What bounds it: up to 32 rows the stream of the words (4.2 - 5 TB/s where a launch has a full round of workgroups), at 33 .. 64 rows
// the unpacking and the matrix cores as well.  Loads straight into registers, 16 rows of 64 bytes apart per request and at most two
// chunks ahead, left the short k runs waiting for memory; slabs of 32 rows read the words twice.  Measured on MI355X, weights from HBM,
// loads in registers -> ring (rows; N x K, group size):
//   1 row:    q|k|v 10240 x 8192, g64 16.4 -> 12.6 us; w1|w3 22016 x 8192 46.5 -> 40.4; w2 8192 x 22016 29.6 -> 21.8; head 34.3 -> 28.6
//   32 rows:  w1|w3 11008 x 4096, g128 16.2 -> 15.9 us; w2 4096 x 11008 10.3 -> 9.7; w2 8192 x 22016, g64 37.8 -> 27.0; head 41.9 -> 34.4
//   64 rows:  q|k|v 10240 x 8192, g64 36.4 -> 25.8 us; wo 8192 x 8192 21.2 -> 17.3; w1|w3 102 -> 78.3; w2 48.5 -> 42.8; head 76 -> 55
// At 64 rows no one unit is full: without the vector work of the scales, without the products, without the operands' loads, without their LDS reads the launch of
// w1|w3 takes 9, 9, 10 and 5 % less, with everything but the products and the words left out still 55 %.  Reading a step's operands and unpacking a tile ahead, with products and
// vector instructions interleaved one to four, took 84.5 for 86 us there with eight waves and 76.4 for 78.3 with four, but 1 us more per launch at 32 rows and less.
#pragma once

#include <type_traits>

#include "e2h_int4_staged.h"
#include "e2h_int4_unpack.h"

namespace e2h {
namespace staged {
namespace {

constexpr int kNt = 2;  // "nt" cache policy: weights are streamed once

typedef __attribute__((address_space(3))) void lds_void;

// Piece b of row r stands at b ^ turned(r / 4 mod 4) of the row's four places.  An LDS read of 16 bytes per lane serves lanes 0 - 3, 12 - 15, 20 - 23 and 24 - 27
// together, then the sixteen between them, then the same of the upper half: in this order each sixteen cover the 64 banks once (with b ^ (r / 4 mod 4), which does
// so for sixteen lanes in a row, 35 - 41 % of the cycles were conflicts).
__device__ __forceinline__ int turned(int k) { return ((k << 1) ^ ((k >> 1) * 3)) & 3; }

// until at most n (a constant once the loop around the call is unrolled) of this wave's loads are out
__device__ __forceinline__ void wait_units(int n) {
  switch (n) {
#define E2H_WAIT(N) \
  case N: asm volatile("s_waitcnt vmcnt(" #N ")" ::: "memory"); break;
    E2H_WAIT(1) E2H_WAIT(2) E2H_WAIT(3) E2H_WAIT(4) E2H_WAIT(5) E2H_WAIT(6) E2H_WAIT(7) E2H_WAIT(8) E2H_WAIT(9) E2H_WAIT(10) E2H_WAIT(11)
    E2H_WAIT(12) E2H_WAIT(13) E2H_WAIT(14) E2H_WAIT(15)
#undef E2H_WAIT
    default: asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
}

// until at most n of this wave's LDS reads are out
__device__ __forceinline__ void wait_reads(int n) {
  switch (n) {
#define E2H_WAIT(N) \
  case N: asm volatile("s_waitcnt lgkmcnt(" #N ")" ::: "memory"); break;
    E2H_WAIT(0) E2H_WAIT(1) E2H_WAIT(2) E2H_WAIT(3) E2H_WAIT(4) E2H_WAIT(5) E2H_WAIT(6) E2H_WAIT(7) E2H_WAIT(8) E2H_WAIT(9) E2H_WAIT(10)
    E2H_WAIT(11) E2H_WAIT(12) E2H_WAIT(13) E2H_WAIT(14)
#undef E2H_WAIT
    default: asm volatile("s_waitcnt lgkmcnt(15)" ::: "memory");
  }
}

// operands of the zero-point term: the groups' sums of 16 (16 bytes each) and their (scale, zero) pairs
template <int RB, int MT, int T, int L>
struct ZeroPoint {
  u32x4_t xs[RB][MT][L];
  uint32_t sz[RB][T];
};

// G group size; MT row tiles of 16 (all rows of the batch, or one of its halves); T weight tiles of 16 rows per workgroup (GATE: T/2 of each matrix).
template <int G, int MT, int T, int EPI, int kWaves>
__global__ __launch_bounds__(64 * kWaves, 2) void int4_staged_mm_kernel(const StagedArgs a) {
  constexpr bool GATE = EPI == kStGate;
  static_assert(!GATE || T % 2 == 0, "gate mode pairs the tiles of two matrices");
  constexpr int TC = GATE ? T / 2 : T;     // distinct column tiles per workgroup
  constexpr int NGRP = 128 / G;            // groups per 128-wide chunk
  constexpr int SPG = G / 32;              // MFMA steps per group
  constexpr int RB = 4 / SPG;              // rounds of four groups whose zero-point operands are requested together: 512 k
  constexpr int kUnits = TC * MT;          // (column tile, row tile) pairs, each finished by one wave
  constexpr int kUnitsPerWave = (kUnits + kWaves - 1) / kWaves;
  // units of a chunk in the order of their use: pairs, operands, words
  constexpr int kSz = GATE ? 2 : (T * NGRP + 15) / 16, kHead = kSz + 4 * MT, UC = kHead + T;
  constexpr int kRing = 16;                      // units of 1 KB per wave
  constexpr int kAhead = (kRing + UC - 1) / UC;  // chunks that the ring reaches into, at most
  constexpr int kLate = kAhead * UC - kRing;     // units of the last kAhead chunks that are issued while those run
  static_assert(kSz + MT < kRing && TC * NGRP <= 16 * (GATE ? 1 : kSz), "ring");
  constexpr bool kTwoSteps = T * MT > 16;        // the parts do not fit LDS at once
  constexpr int kParts = kTwoSteps ? kWaves / 2 : kWaves;
  constexpr int kRedBytes = kParts * T * MT * 1024, kRingBytes = kWaves * kRing * 1024;

  constexpr int kBestAt = kRedBytes > kRingBytes ? kRedBytes : kRingBytes;

  // One object for everything: beside a second one the compiler tells loads into LDS from reads by object and puts a wait for all loads
  // in front of the reads (the arg-max kernel with an array of its own behind the ring: 19 such waits for 5, 32000 x 4096 at 32 rows 27.6 us
  // for 20).
  __shared__ __attribute__((aligned(1024))) uint8_t lds[kBestAt + (EPI == kStArgmax ? kUnits * 128 : 0)];
  unsigned long long *const unit_best = reinterpret_cast<unsigned long long *>(lds + kBestAt);  // arg-max: [unit][row of its tile]

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int kg = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave = k part
  const int c = lane & 15, b = lane >> 4;
  const int N = a.N, K = a.K, M = a.M;
  const int KT = K >> 7;  // packed k-blocks (inner_k_tiles = 8) = chunks
  const int S = gridDim.y, ks = blockIdx.y;
  const int C0 = static_cast<int>((static_cast<unsigned>(KT) * static_cast<unsigned>(ks)) / static_cast<unsigned>(S));
  const int C1 = static_cast<int>((static_cast<unsigned>(KT) * static_cast<unsigned>(ks + 1)) / static_cast<unsigned>(S));
  const int c0 = C0 + ((C1 - C0) * kg) / kWaves;
  const int nloc = C0 + ((C1 - C0) * (kg + 1)) / kWaves - c0;
  const int col_block = blockIdx.x;
  // Rows of a multiple of 32 KB: workgroups that all start with their first chunk ask few of the memory's channels at a time, so each starts with another one
  // (w1|w3 22016 x 8192, g64, 1 row 48.5 -> 40.4 us, 32 rows 55.7 -> 50.4; head 32000 x 8192, 1 row 35.2 -> 28.6; 12288 x 4096, which has rows of 16 KB, 7.8 either way).
  // Workgroups of four waves begin alike: turned chunks make no difference to them (w1|w3, g64, 33 rows 73.2 us, turned 73.1, 64 rows 75.5 and 76.3; head, 64 rows 54.0 and 53.4).
  const int turn = kWaves == 8 && KT % 64 == 0 && nloc > 0 ? static_cast<int>(static_cast<unsigned>(col_block) % static_cast<unsigned>(nloc)) : 0;
  const int row0 = blockIdx.z * (16 * MT);
  const int tile16_0 = col_block * TC;
  const int tiles = (N >> 4) - tile16_0 < TC ? (N >> 4) - tile16_0 : TC;  // N % 16 == 0
  const uint32_t row_block = static_cast<uint32_t>(a.Mpad) * 64u;  // bytes of one k segment of all rows

  // this workgroup's tiles are consecutive in the packed words; a (scale, zero) pair of group g and column n is dword g N + n
  const size_t w_base = static_cast<size_t>(tile16_0) * KT * 1024;
  const uint32_t w_bytes = static_cast<uint32_t>(tiles) * KT * 1024u;
  const uint32_t sz_bytes = static_cast<uint32_t>(static_cast<size_t>(K / G) * N * 4);
  const __amdgpu_buffer_rsrc_t w_rsrc = make_rsrc(reinterpret_cast<const uint8_t *>(a.wp) + w_base, w_bytes);
  const __amdgpu_buffer_rsrc_t sz_rsrc = make_rsrc(a.sz, sz_bytes);
  const __amdgpu_buffer_rsrc_t w2_rsrc = make_rsrc(reinterpret_cast<const uint8_t *>(GATE ? a.wp2 : a.wp) + w_base, w_bytes);
  const __amdgpu_buffer_rsrc_t sz2_rsrc = make_rsrc(GATE ? a.sz2 : a.sz, sz_bytes);
  const __amdgpu_buffer_rsrc_t x_rsrc = make_rsrc(a.frag, static_cast<uint32_t>(static_cast<size_t>(K / 32) * row_block));
  const __amdgpu_buffer_rsrc_t xs_rsrc = make_rsrc(a.sums, static_cast<uint32_t>(static_cast<size_t>(KT) * a.Mpad * 32));

  uint8_t *const ring = lds + kg * (kRing * 1024);
  // what lane 4 q + s brings: piece s ^ turned(q / 4 mod 4) of row q
  const int q4 = lane >> 2;
  const uint32_t piece = static_cast<uint32_t>((lane & 3) ^ turned(lane >> 4)) * 16u;
  const uint32_t w_lane = static_cast<uint32_t>(q4 >> 3) * KT * 512u + (q4 & 7) * 64u + piece;  // rows 0 .. 7, 8 .. 15: two packed tiles
  const uint32_t x_lane = static_cast<uint32_t>(row0 + q4) * 64u + piece;
  const auto column_of = [&](int t) { return 16 * (tile16_0 + (t < tiles ? t : tiles - 1)); };  // past the end: any valid one
  // unit p (static) of a chunk into ring place `at`
  const auto issue = [&](int p, uint32_t chunk, int at) {
    lds_void *const dst = (lds_void *)(ring + at * 1024);
    if (p < kSz) {
      // 16 bytes (four columns) per lane: pair block q4 = (tile, group) of this unit's sixteen
      const int blk = q4 + (GATE ? 0 : 16 * p), t = blk / NGRP, g = blk % NGRP;
      const uint32_t off = (static_cast<uint32_t>(g) * N + column_of(t) + 4u * (lane & 3)) * 4u;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(GATE && p > 0 ? sz2_rsrc : sz_rsrc, dst, 16, off, chunk * (NGRP * 4u) * static_cast<uint32_t>(N), 0, 0);
    } else if (p < kHead) {
      const int s = (p - kSz) / MT, mt = (p - kSz) % MT;
      const uint32_t off = row0 + 16 * mt + q4 < M ? x_lane + 1024u * mt : 0x80000000u;  // rows past M: out of the buffer's range, zeros
      __builtin_amdgcn_raw_ptr_buffer_load_lds(x_rsrc, dst, 16, off, (chunk * 4u + s) * row_block, 0, 0);
    } else {
      const int t = p - kHead;  // past N: out of the buffer's range, zeros
      __builtin_amdgcn_raw_ptr_buffer_load_lds(t < TC ? w_rsrc : w2_rsrc, dst, 16, w_lane + static_cast<uint32_t>(t % TC) * KT * 1024u, chunk * 512u, 0, kNt);
    }
  };

  f32x4_t acc[T][MT];
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[t][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const UnpackConsts uc = unpack_consts();

  // ---- the zero-point term: four groups per float32 MFMA, lane (b, .) owns group 4 r + b of the wave's run ---------------
  const int ngroups = nloc * NGRP;
  typedef ZeroPoint<RB, MT, T, NGRP == 1 ? 2 : 1> Zero;
  const auto zero_point_load = [&](Zero &z, int r0) {
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      const int gi = 4 * (r0 + r) + b;
      const int gcl = gi < ngroups ? gi : 0;
      int chunk = c0 + gcl / NGRP;
      chunk = chunk < KT ? chunk : KT - 1;
      const int sub = gcl % NGRP;
      // chunk and sub differ between lanes: everything goes into the vector offset
      const uint32_t so = static_cast<uint32_t>(chunk) * static_cast<uint32_t>(a.Mpad) * 32u;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        // the group's 8 / NGRP sums of 16
        const uint32_t off = so + static_cast<uint32_t>((row0 + 16 * mt + c) * 32 + sub * (32 / NGRP));
        if constexpr (NGRP == 1) {
          z.xs[r][mt][0] = __builtin_amdgcn_raw_buffer_load_b128(xs_rsrc, off, 0, 0);
          z.xs[r][mt][1] = __builtin_amdgcn_raw_buffer_load_b128(xs_rsrc, off + 16, 0, 0);
        } else if constexpr (NGRP == 2) {
          z.xs[r][mt][0] = __builtin_amdgcn_raw_buffer_load_b128(xs_rsrc, off, 0, 0);
        } else {
          const u32x2_t lo = __builtin_amdgcn_raw_buffer_load_b64(xs_rsrc, off, 0, 0);
          z.xs[r][mt][0] = u32x4_t{lo[0], lo[1], 0u, 0u};
        }
      }
#pragma unroll
      for (int t = 0; t < T; ++t)
        z.sz[r][t] = __builtin_amdgcn_raw_buffer_load_b32(GATE && t >= TC ? sz2_rsrc : sz_rsrc, static_cast<uint32_t>(column_of(t % TC) + c) * 4u +
                                                             static_cast<uint32_t>(chunk * NGRP + sub) * static_cast<uint32_t>(N) * 4u, 0, 0);
    }
  };
  const auto zero_point_use = [&](const Zero &z, int r0) {
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      const bool live = 4 * (r0 + r) + b < ngroups;
      float xsum[MT];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const f32x4_t lo = __builtin_bit_cast(f32x4_t, z.xs[r][mt][0]);
        float v;
        if constexpr (NGRP == 1) {
          const f32x4_t hi = __builtin_bit_cast(f32x4_t, z.xs[r][mt][1]);
          v = ((lo[0] + lo[1]) + (lo[2] + lo[3])) + ((hi[0] + hi[1]) + (hi[2] + hi[3]));
        } else if constexpr (NGRP == 2) {
          v = (lo[0] + lo[1]) + (lo[2] + lo[3]);
        } else {
          v = lo[0] + lo[1];
        }
        xsum[mt] = live ? v : 0.f;
      }
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const float scale = __builtin_bit_cast(float, z.sz[r][t] << 16);
        const float zero = __builtin_bit_cast(float, z.sz[r][t] & 0xFFFF0000u);
        const float zc = live ? __builtin_fmaf(-136.0f, scale, zero) : 0.f;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[t][mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(xsum[mt], zc, acc[t][mt], 0, 0, 0);
      }
    }
  };

  Zero z0, z1;
  zero_point_load(z0, 0);
  __builtin_amdgcn_sched_barrier(0);
  uint32_t ahead[kAhead + 1];  // the chunk at hand and those behind it
  const auto behind = [&](uint32_t chunk) { return chunk + 1 == static_cast<uint32_t>(c0 + nloc) ? static_cast<uint32_t>(c0) : chunk + 1; };
  ahead[0] = static_cast<uint32_t>(c0 + turn);
#pragma unroll
  for (int d = 0; d < kAhead; ++d) ahead[d + 1] = behind(ahead[d]);
#pragma unroll
  for (int u = 0; u < kRing; ++u)
    if (u / UC < nloc) issue(u % UC, ahead[u / UC], u);
  if (4 * RB < ngroups) zero_point_load(z1, RB);
  __builtin_amdgcn_sched_barrier(0);

  // RoPE epilogue: the rotation's cos / sin depend on a position read from memory; both are fetched now, behind the
  // first loads, for the units this wave will finish
  int rope_pos = -1;
  float rope_cs[kUnitsPerWave], rope_sn[kUnitsPerWave];
#pragma unroll
  for (int u = 0; u < kUnitsPerWave; ++u) {
    rope_cs[u] = 1.f;
    rope_sn[u] = 0.f;
  }
  if constexpr (EPI == kStRope) {
    const int64_t p = a.rope.input_pos[0];
    rope_pos = p >= 0 && p < a.rope.S ? static_cast<int>(p) : -1;
#pragma unroll
    for (int u = 0; u < kUnitsPerWave; ++u) {
      const int unit = kg + u * kWaves;
      const int ncol = 16 * (tile16_0 + unit / MT) + c;
      if (unit < kUnits && ncol < N && rope_pos >= 0 && ncol < (a.rope.H + a.rope.Hkv) * a.rope.D) {
        const uint32_t f = reinterpret_cast<const uint32_t *>(a.rope.freqs)[static_cast<size_t>(rope_pos) * (a.rope.D / 2) + ((ncol % a.rope.D) >> 1)];
        rope_cs[u] = __builtin_bit_cast(float, f << 16);
        rope_sn[u] = __builtin_bit_cast(float, f & 0xFFFF0000u);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  zero_point_use(z0, 0);
  if (4 * RB < ngroups) {
    for (int r0 = 2 * RB; 4 * r0 < ngroups; r0 += RB) {
      zero_point_load(z0, r0);
      zero_point_use(z1, r0 - RB);
      z1 = z0;
    }
    zero_point_use(z1, (ngroups - 1) / (4 * RB) * RB);
  }
  __builtin_amdgcn_sched_barrier(0);

  // ---- the chunks -------------------------------------------------------------------------------------------------
  const uint32_t read_lane = c * 64u + ((b ^ turned(c >> 2)) * 16u);  // lane (b, c): piece b of row c
  // kTail -1: a chunk with kAhead or more behind it; 0 .. kAhead - 1: the last ones, for which ever less is left to issue; kAhead: all has landed
  const auto chunk = [&](auto tail, int i, int at0) {
    constexpr int kTail = decltype(tail)::value;
    constexpr bool kSteady = kTail < 0, kDone = kTail == kAhead;
    // A batch of n units from p0 on, behind one of `before` units whose places are refilled only once this batch's reads are on their
    // way, so that no wave waits for its own reads.  Loads that may still be out: the ring's younger units.
    const auto landed = [&](int p0, int n, int before) {
      if (kDone) return;
      const int issued = kTail * UC + p0 - before + kRing, all = kAhead * UC;
      const int younger = kSteady ? kRing - before - n : (issued < all ? issued : all) - (kTail * UC + p0 + n);
      wait_units(younger);
    };
    const auto at = [&](int p) { return (at0 + p) & (kRing - 1); };
    // the places of units p0 .. p0 + n - 1 of chunk j, whose reads are followed by `later` newer ones; j_tail: kTail of that chunk
    const auto refill = [&](int before, int j_tail, int j_at0, int p0, int n, int later) {  // (of the chunk at hand or, before = 1, the one before it)
      if (kDone) return;
      wait_reads(later);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int p = p0; p < p0 + n; ++p)
        if (j_tail < 0 || j_tail * UC + p < kLate) issue((p + kRing) % UC, ahead[(p + kRing) / UC - before], (j_at0 + p) & (kRing - 1));
      __builtin_amdgcn_sched_barrier(0);
    };
    uint32_t sz[T][NGRP];
    landed(0, kSz, 1);
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int g = 0; g < NGRP; ++g) {
        const int blk = (t % TC) * NGRP + g;
        sz[t][g] = *reinterpret_cast<const uint32_t *>(ring + at(GATE ? t / TC : blk / 16) * 1024 + (blk % 16) * 64 + c * 4);
      }
    if (i > 0) refill(1, kTail < 0 ? -1 : kTail - 1, at0 - UC, UC - 1, 1, T * NGRP);  // the previous chunk's last batch
    bf16x8_t x[4][MT];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int p0 = kSz + s * MT, before = s == 0 ? kSz : MT;
      landed(p0, MT, before);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) x[s][mt] = *reinterpret_cast<const bf16x8_t *>(ring + at(p0 + mt) * 1024 + read_lane);
      refill(0, kTail, at0, p0 - before, before, MT);
    }
    u32x4_t w[2];
#pragma unroll
    for (int t = 0; t < T + 1; ++t) {
      if (t < T) {
        const int before = t > 0 ? 1 : MT;
        landed(kHead + t, 1, before);
        w[t & 1] = *reinterpret_cast<const u32x4_t *>(ring + at(kHead + t) * 1024 + read_lane);
        refill(0, kTail, at0, kHead + t - before, before, 1);
      }
      if (t == 0) continue;
#pragma unroll
      for (int g = 0; g < NGRP; ++g) {
        f32x4_t part[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) part[mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < SPG; ++s) {
          const bf16x8_t wf = unpack_word(w[(t - 1) & 1][g * SPG + s], uc);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) part[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[g * SPG + s][mt], wf, part[mt], 0, 0, 0);
        }
        const float scale = __builtin_bit_cast(float, sz[t - 1][g] << 16);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int q = 0; q < 4; ++q) acc[t - 1][mt][q] = __builtin_fmaf(scale, part[mt][q], acc[t - 1][mt][q]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  int i = 0, at0 = 0;
  const auto run = [&](auto tail) {
    chunk(tail, i, at0);
    at0 = (at0 + UC) & (kRing - 1);
    ++i;
#pragma unroll
    for (int d = 0; d < kAhead; ++d) ahead[d] = ahead[d + 1];
    ahead[kAhead] = behind(ahead[kAhead]);
  };
#pragma unroll 1
  while (i < nloc - kAhead) run(std::integral_constant<int, -1>{});
  if (nloc >= kAhead) {
    run(std::integral_constant<int, 0>{});
    if constexpr (kAhead > 1) run(std::integral_constant<int, 1>{});
    if constexpr (kAhead > 2) run(std::integral_constant<int, 2>{});
    static_assert(kAhead <= 3, "ring");
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll 1
  while (i < nloc) run(std::integral_constant<int, kAhead>{});  // a wave with fewer chunks than the ring holds

  // ---- the waves' K parts meet in LDS as a balanced tree in the order of K; wave w finishes units w, w + kWaves, .. -------
  float *const red = reinterpret_cast<float *>(lds);
  const auto put = [&](int part) {
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) *reinterpret_cast<f32x4_t *>(red + ((part * T * MT + t * MT + mt) * 64 + lane) * 4) = acc[t][mt];
  };
  const auto get = [&](int part, int t, int mt) { return *reinterpret_cast<const f32x4_t *>(red + ((part * T * MT + t * MT + mt) * 64 + lane) * 4); };
  lds_barrier();  // the rings are done with
  if constexpr (kTwoSteps) {
    if (kg & 1) put(kg >> 1);
    lds_barrier();
    if (!(kg & 1)) {
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[t][mt] += get(kg >> 1, t, mt);
    }
    lds_barrier();
    if (!(kg & 1)) put(kg >> 1);
  } else {
    put(kg);
  }
  lds_barrier();
#pragma unroll
  for (int u = 0; u < kUnitsPerWave; ++u) {
    const int unit = kg + u * kWaves;
    if (unit >= kUnits) break;  // uniform per wave
    const int tc = unit / MT, mt = unit % MT;
    f32x4_t v[GATE ? 2 : 1];
#pragma unroll
    for (int h = 0; h < (GATE ? 2 : 1); ++h) {
      const int t = tc + h * TC;
      f32x4_t pair[kWaves / 2];
#pragma unroll
      for (int w = 0; w < kWaves / 2; ++w) pair[w] = kTwoSteps ? get(w, t, mt) : get(2 * w, t, mt) + get(2 * w + 1, t, mt);
      v[h] = pair[0] + pair[1];
      if constexpr (kWaves == 8) v[h] += pair[2] + pair[3];
    }
    const int n = 16 * (tile16_0 + tc) + c;
    if constexpr (EPI == kStPartial) {
      float *out = a.partials + static_cast<size_t>(ks) * M * N;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int m = row0 + 16 * mt + 4 * b + q;
        if (n < N && m < M) out[static_cast<size_t>(m) * N + n] = v[0][q];
      }
    } else if constexpr (EPI == kStGate) {
      // bf16(bf16(silu(bf16 gate)) * bf16 up): the rounding points of F.silu(w1(x)) * w3(x) on bfloat16 tensors
      // (reference models/model.py:359-360)
      const bool tile_live = 16 * (tile16_0 + tc) < N;  // whole tiles: N % 16 == 0 on this path
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int m = row0 + 16 * mt + 4 * b + q;
        const float gate = bf16_round(v[0][q]), up = bf16_round(v[1][q]);
        const float act = bf16_round(gate / (1.0f + expf(-gate)));
        const uint16_t o = f32_to_bf16_rne(act * up);
        if (a.y && n < N && m < M) a.y[static_cast<size_t>(m) * N + n] = o;
        // staged form for the next linear: whole 16-lane groups store (rows past M hold values nobody reads)
        if (a.out.frag && tile_live && m < a.out.mpad) staged_store_run16(a.out, m, n, o);
      }
    } else if constexpr (EPI == kStRope) {
      // the product is the fused q | k | v projection, rounded to bfloat16; the interleaved pairs of the q and k heads
      // are rotated in float32 (reference models/model.py:400-412); q goes to q_out [B, H, D], k and v into the caches
      // [B, Hkv, S, D] at the position (KVCache.update, reference models/model.py:121-129)
      const StagedRope &rp = a.rope;
      const int Dh = rp.D, H = rp.H, Hkv = rp.Hkv;
      const int pos = rope_pos;
      const int head = n / Dh, d = n % Dh;
      const bool in_range = n < N && pos >= 0;
      const bool rotated = head < H + Hkv;
      const float cs = rope_cs[u], sn = rope_sn[u];
      uint16_t *dst;
      size_t row_stride;
      if (head < H) {
        dst = rp.q_out + static_cast<size_t>(head) * Dh + d;
        row_stride = static_cast<size_t>(H) * Dh;
      } else {
        const int hk = rotated ? head - H : head - H - Hkv;
        dst = (rotated ? rp.kc : rp.vc) + (static_cast<size_t>(hk) * rp.S + (pos < 0 ? 0 : pos)) * Dh + d;
        row_stride = static_cast<size_t>(Hkv) * rp.S * Dh;
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int m = row0 + 16 * mt + 4 * b + q;
        const float own = bf16_round(v[0][q]);
        const float other = __shfl_xor(own, 1);  // the pair's other column lives in the neighbouring lane
        const float r = (c & 1) ? own * cs + other * sn : own * cs - other * sn;
        if (in_range && m < M) dst[static_cast<size_t>(m) * row_stride] = f32_to_bf16_rne(rotated ? r : own);
      }
    } else if constexpr (EPI == kStArgmax) {
      // greedy token straight from the LM head: the logit is rounded to bfloat16 as the plain epilogue would store it and
      // offered as (order-preserving key << 32 | ~column), so that the maximum is the largest value and, among equals,
      // the lowest column; a NaN counts as the largest value (torch.argmax over the float32 view of bfloat16 logits,
      // reference inference_generate.py:110-120 with sampling switched off).  First over the tile's 16 columns ...
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t u = static_cast<uint32_t>(f32_to_bf16_rne(v[0][q])) << 16;
        const uint32_t key = (u & 0x7FFFFFFFu) > 0x7F800000u ? 0xFFFFFFFFu : ((u & 0x80000000u) ? ~u : (u | 0x80000000u));
        unsigned long long best = n < N ? ((static_cast<unsigned long long>(key) << 32) | static_cast<uint32_t>(~static_cast<uint32_t>(n))) : 0ull;
#pragma unroll
        for (int off = 1; off < 16; off <<= 1) {
          const unsigned long long other = __shfl_xor(best, off);
          best = other > best ? other : best;
        }
        if (c == 0) unit_best[unit * 16 + 4 * b + q] = best;
      }
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int m = row0 + 16 * mt + 4 * b + q;
        if (n < N && m < M) a.y[static_cast<size_t>(m) * N + n] = f32_to_bf16_rne(v[0][q]);
      }
    }
  }
  if constexpr (EPI == kStArgmax) {
    // ... then over the workgroup's column tiles: one candidate per row and column block for the reduction kernel
    __syncthreads();
    if (tid < 16 * MT) {
      const int mt = tid >> 4, m = row0 + tid;
      unsigned long long best = 0ull;
#pragma unroll
      for (int tc = 0; tc < TC; ++tc) {
        const unsigned long long other = unit_best[(tc * MT + mt) * 16 + (tid & 15)];
        best = other > best ? other : best;
      }
      if (m < M) a.cand[static_cast<size_t>(col_block) * M + m] = best;
    }
  }
}

template <int G, int MT, int T, int EPI>
int launch_staged(const StagedArgs &a, const Geometry &g, hipStream_t stream) {
  if constexpr (T > max_tiles(G, MT, EPI == kStGate)) {
    return E2H_ERR_BAD_SHAPE;
  } else {
    const dim3 grid(a.col_blocks, g.slices, g.halves);
    if (g.waves == 4) hipLaunchKernelGGL((int4_staged_mm_kernel<G, MT, T, EPI, 4>), grid, dim3(256), 0, stream, a);
    else hipLaunchKernelGGL((int4_staged_mm_kernel<G, MT, T, EPI, 8>), grid, dim3(512), 0, stream, a);
    return launch_status();
  }
}

template <int G, int MT, int EPI>
int dispatch_tiles(const StagedArgs &a, const Geometry &g, hipStream_t stream) {
  switch (g.t) {
    case 2: return launch_staged<G, MT, 2, EPI>(a, g, stream);
    case 4: return launch_staged<G, MT, 4, EPI>(a, g, stream);
    case 6: return launch_staged<G, MT, 6, EPI>(a, g, stream);
    case 8: return launch_staged<G, MT, 8, EPI>(a, g, stream);
  }
  if constexpr (EPI == kStGate) {
    if (g.t == 12) return launch_staged<G, MT, 12, EPI>(a, g, stream);
  } else {
    if (g.t == 1) return launch_staged<G, MT, 1, EPI>(a, g, stream);
    if (g.t == 3) return launch_staged<G, MT, 3, EPI>(a, g, stream);
  }
  return E2H_ERR_BAD_SHAPE;
}

template <int G, int EPI>
int dispatch_rows(const StagedArgs &a, const Geometry &g, hipStream_t stream) {
  switch (g.mt) {
    case 1: return dispatch_tiles<G, 1, EPI>(a, g, stream);
    case 2: return dispatch_tiles<G, 2, EPI>(a, g, stream);
    case 4: return dispatch_tiles<G, 4, EPI>(a, g, stream);
  }
  return E2H_ERR_BAD_SHAPE;
}

}  // namespace

template <int G>
int launch_group(int epilogue, const StagedArgs &a, const Geometry &g, hipStream_t stream) {
  switch (epilogue) {
    case kStPlain: return dispatch_rows<G, kStPlain>(a, g, stream);
    case kStGate: return dispatch_rows<G, kStGate>(a, g, stream);
    case kStRope: return dispatch_rows<G, kStRope>(a, g, stream);
    case kStPartial: return dispatch_rows<G, kStPartial>(a, g, stream);
    case kStArgmax: return dispatch_rows<G, kStArgmax>(a, g, stream);
  }
  return E2H_ERR_BAD_SHAPE;
}

}  // namespace staged
}  // namespace e2h
