// Matrix product of two 16-bit operands, 256 x 256 outputs per tile: the loop that the many-row kernels share.
//
//   out[row][col] = sum_k x[row][k] w[col][k]      x rows and w rows of K values, K a multiple of 64 and at least 192
//
// What bounds it: the matrix pipelines (busy 75 - 78 % of a launch that fills the chip, the library's kernel 83 %), and with all of them at work the chip's power (1.75 - 1.85 GHz instead of
// 2.4), so that everything that costs energy beside the products costs time.  One workgroup per CU of four waves, each 128 x 128 outputs in 256 accumulation registers
// (an LDS read of 16 values per lane feeds 64 products of 16 x 16 x 32; 256 x 64 per wave would read 1.25 times as much).  Operands reach LDS by
// 16-byte loads that write LDS directly, in units of 256 rows x 64 k (32 KB, whole 128-byte lines: units of 32 k, which ask the L2 for every line
// twice, ran at 1300 TFLOP/s where this runs at 1420 - 1520).  All 160 KB of LDS are a ring of five such units, x_0 w_0 x_1 w_1 ..: a unit's place
// is free as soon as the fragments of its second half are in registers, so that a chunk of 64 k is requested two chunks ahead of its use.
// One barrier per chunk, in its middle.  The walk over tiles is one pipeline: the first chunks of a tile are on their way while the
// one before it is finished and stored.
// A tile's first products take zero as their third operand instead of 256 registers set to it, and its loop runs at least once behind
// the first chunk, which is what lets the compiler count the loads behind those of `dest`: of a scoring pass of 49152 rows 1.1 %.
//   8192 rows, bfloat16: 12288 x 4096 545 us (1510 TFLOP/s), 4096 x 11008 480 us (1540).
//
// 16-byte pieces of a row stand at position piece ^ f(row) of its 128 bytes, f chosen so that the 16 rows of a fragment read fall on different
// bank groups: rows of x in order, f = (row / 2) % 8; of w the fragments i = 2 p and 2 p + 1 of a wave hold columns 32 p + 8 (r / 4) + 4 (i % 2) + r % 4
// (r: the fragment's row), so that a lane ends up with eight neighbouring outputs of a row, f = (column / 2) % 2 + 2 ((column / 8) % 4).
#pragma once

#include <type_traits>

#include "e2h_common.h"

namespace e2h {
namespace gemm256 {

constexpr int kSide = 256, kLeastK = 192;
constexpr uint32_t kUnit = 256 * 128, kRing = 5 * kUnit;
constexpr uint32_t kNowhere = 0xFFFFFFF0u;  // an offset past every buffer: the store is dropped

#if defined(__HIP_DEVICE_COMPILE__)
typedef __attribute__((address_space(3))) void lds_void_t;

// In-place accumulation on an accumulation register: left to itself the register allocator, with all 256 of them taken, moves
// accumulators about inside the loop (twice the time).
// FIRST: a tile's first product of these outputs, which needs no register set to zero.
template <bool F16, bool FIRST>
__device__ __forceinline__ void mma(f32x4_t &d, u32x4_t a, u32x4_t b) {
  if constexpr (FIRST && F16) asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, 0" : "=a"(d) : "v"(a), "v"(b));
  else if constexpr (FIRST) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(d) : "v"(a), "v"(b));
  else if constexpr (F16) asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(d) : "v"(a), "v"(b));
  else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(d) : "v"(a), "v"(b));
}

// P names the tiles and what surrounds them.  P::Tile holds uniform values.
//   static constexpr bool kHalves             whether tiles may have 128 rows and fewer, bool half(Tile): whether this one does; only the products of those are
//                                             formed then, and the rows 32 j + 16 wm + r of a tile are wave wm's instead of 128 wm + 16 j + r
//   static constexpr bool kPairs              whether the upper 64 columns of a wave's 128 belong to the lower ones, as up to gate
//   bool first(Tile &), bool next(Tile &)     the workgroup's tiles, false: no more
//   int chunks()                              K / 64
//   rsrc x_rsrc(Tile), w_rsrc(Tile)           the operands
//   Fetch, fetch(Tile, lane, wave, Fetch &)   what the two below need from memory (requested a tile ahead)
//   uint32_t x_at(Tile, Fetch, i, row), w_at(Tile, col)   byte offset of row (0 .. 255, the i-th of this lane) and column of the tile, inside the buffer
//   Dest, dest(Tile, row of the lane's first output, col, Dest &)   what store needs from memory
//   store(Tile, Dest, j, p, row, col, v)      stores the eight outputs (row, col .. col + 7), one vector store in every case
//   store(Tile, Dest, j, p, row, col, v, u)   with kPairs: v, and u of the columns 64 further on
template <bool F16, class P>
__device__ __forceinline__ void walk(P &p, uint8_t *lds) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave & 1, wn = wave >> 1, chunks = p.chunks();
  // a wave's 16-row blocks: neighbours, or every second one where tiles may be half empty
  constexpr int kXWave = P::kHalves ? 16 : 128, kXStep = P::kHalves ? 32 : 16;
  constexpr int kStores = P::kPairs ? 16 : 32;  // vector stores of a wave per tile, exactly (see below)
  typename P::Tile cur, nxt;
  if (!p.first(cur)) return;  // uniform, before any barrier

  // loads: wave w brings the 1 KB blocks w, w + 4, .. of a unit (8 rows each), lane l position l % 8 of row l / 8
  const uint32_t xpiece = ((lane & 7) ^ ((4 * (wave & 1) + (lane >> 4)) & 7)) * 16, wpiece = ((lane & 7) ^ (((lane >> 4) & 1) + 2 * wave)) * 16;
  uint32_t xsrc[8], wsrc[8];
  typename P::Fetch fetched;
  __amdgpu_buffer_rsrc_t xr = p.x_rsrc(cur), wr = p.w_rsrc(cur);
  auto aim_x = [&](const typename P::Tile &t) {
    xr = p.x_rsrc(t);
#pragma unroll
    for (int i = 0; i < 8; ++i) xsrc[i] = p.x_at(t, fetched, i, 8 * (wave + 4 * i) + (lane >> 3)) + xpiece;
  };
  auto aim_w = [&](const typename P::Tile &t) {
    wr = p.w_rsrc(t);
#pragma unroll
    for (int i = 0; i < 8; ++i) wsrc[i] = p.w_at(t, P::kPairs ? 32 * i + ((8 * wave + (lane >> 3)) & 31) : 8 * (wave + 4 * i) + (lane >> 3)) + wpiece;  // (the same: pairs want bit 6 a constant)
  };
  auto load_x = [&](int chunk, uint32_t unit, int i) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_void_t *)(lds + unit + (wave + 4 * i) * 1024), 16, xsrc[i], static_cast<uint32_t>(chunk) * 128, 0, 0);
  };
  auto load_w = [&](int chunk, uint32_t unit, int i) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lds_void_t *)(lds + unit + (wave + 4 * i) * 1024), 16, wsrc[i], static_cast<uint32_t>(chunk) * 128, 0, 0);
  };

  // fragments of a half chunk: lane (h, n) reads piece 4 s + h of its rows
  const int n = lane & 15, h = lane >> 4;
  const uint32_t xa = (kXWave * wm + n) * 128 + ((h ^ ((n >> 1) & 7)) << 4);
  const uint32_t wa = (128 * wn + 8 * (n >> 2) + (n & 3)) * 128 + ((h ^ (((n >> 1) & 1) + 2 * (n >> 2))) << 4);
  u32x4_t xf[2][8], wf[2][8];
  auto read_x = [&](uint32_t unit, int s, int i) { return *reinterpret_cast<const u32x4_t *>(lds + unit + (xa ^ (64 * s)) + i * (kXStep * 128)); };
  auto read_w = [&](uint32_t unit, int s, int i) {
    return *reinterpret_cast<const u32x4_t *>(lds + unit + (wa ^ (64 * s)) + (i >> 1) * 4096 + (i & 1) * 512);
  };
  auto after = [](uint32_t unit) { return unit + kUnit == kRing ? 0u : unit + kUnit; };

  p.fetch(cur, lane, wave, fetched);
  aim_x(cur);
  aim_w(cur);
#pragma unroll
  for (int i = 0; i < 8; ++i) load_x(0, 0, i);
#pragma unroll
  for (int i = 0; i < 8; ++i) load_w(0, kUnit, i);
#pragma unroll
  for (int i = 0; i < 8; ++i) load_x(1, 2 * kUnit, i);
#pragma unroll
  for (int i = 0; i < 8; ++i) load_w(1, 3 * kUnit, i);
  asm volatile("s_waitcnt vmcnt(16)\n\ts_barrier" ::: "memory");
  nxt = cur;
  bool more = p.next(nxt);
  if (more) p.fetch(nxt, lane, wave, fetched);
  typename P::Dest dest;
  const int row0 = kXWave * wm + n, col0 = 128 * wn + 8 * h;
  p.dest(cur, row0, col0, dest);
#pragma unroll
  for (int i = 0; i < 8; ++i) xf[0][i] = read_x(0, 0, i);
#pragma unroll
  for (int i = 0; i < 8; ++i) wf[0][i] = read_w(kUnit, 0, i);

  uint32_t xu = 0, wu = kUnit, loading = 3 * kUnit;
  int ahead = 2;         // the chunk that the next loads bring, of this tile or (once it has come round) of the next one
  bool stored = false;   // this tile's first chunk has the stores of another one in front of its loads
  auto chunk = [&](auto first, auto blocks, f32x4_t (&acc)[8][8]) {
    constexpr bool kFirst = decltype(first)::value;  // of a tile
    constexpr int kBlocks = decltype(blocks)::value;  // of 16 rows per wave
    const uint32_t nxu = after(wu), nwu = after(nxu);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      if (s == 1) {
        // The next chunk has landed once at most what was issued behind it is open: the eight loads of the first half, and in a tile's first
        // chunk the stores of the tile before it.  Behind the barrier nobody reads this chunk's units any more.
        if (kFirst && stored) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(8 + kStores) : "memory");
        else asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      }
      loading = after(loading);
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < kBlocks; ++j) {
          if (kFirst && s == 0) mma<F16, true>(acc[i][j], wf[s][i], xf[s][j]);
          else mma<F16, false>(acc[i][j], wf[s][i], xf[s][j]);
          const int slot = kBlocks * i + j, r = slot / 2;
          if (slot % 2 == 0 && r < 16) {  // the next half's fragments, in the order of their use
            if (r == 0) wf[s ^ 1][0] = read_w(s ? nwu : wu, s ^ 1, 0);
            else if (r <= 8) xf[s ^ 1][r - 1] = read_x(s ? nxu : xu, s ^ 1, r - 1);
            else wf[s ^ 1][r - 8] = read_w(s ? nwu : wu, s ^ 1, r - 8);
          }
          if (slot % 4 == 1 && slot < 32) {
            if (s == 0) load_x(ahead, loading, slot / 4);
            else load_w(ahead, loading, slot / 4);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      // behind the last tile the loads go on reading it: nobody uses them
      if (s == 0 && ahead + 1 == chunks && more) aim_x(nxt);
      if (s == 1 && ++ahead == chunks) {
        ahead = 0;
        if (more) aim_w(nxt);
      }
    }
    xu = nxu;
    wu = nwu;
  };
  while (true) {
    const auto chunks_of = [&](auto blocks) {
      f32x4_t acc[8][8];
      chunk(std::true_type{}, blocks, acc);
      int c = 1;
      do chunk(std::false_type{}, blocks, acc);  // at least three chunks: whoever waits for what a tile's start has requested can count on that
      while (++c < chunks);
      asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");  // the last products' results can be read
      __builtin_amdgcn_sched_barrier(0);
      int row = row0, col = col0;
      asm volatile("" : "+v"(row), "+v"(col));  // what is derived from them is formed here: held through the tiles, it would not fit the registers
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int q = 0; q < (P::kPairs ? 2 : 4); ++q) {
          float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};  // rows that are not there: stored nowhere, but counted
          if (j < decltype(blocks)::value) {
            asm volatile("" : "+a"(acc[2 * q][j]), "+a"(acc[2 * q + 1][j]));  // read here: all 256 at once would not fit
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = acc[2 * q + (e >> 2)][j][e & 3];
          }
          if constexpr (P::kPairs) {
            float u[8];
            asm volatile("" : "+a"(acc[2 * q + 4][j]), "+a"(acc[2 * q + 5][j]));
#pragma unroll
            for (int e = 0; e < 8; ++e) u[e] = acc[2 * q + 4 + (e >> 2)][j][e & 3];
            p.store(cur, dest, j, q, row + kXStep * j, col + 32 * q, v, u);
          } else {
            p.store(cur, dest, j, q, row + kXStep * j, col + 32 * q, v);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
    };
    if constexpr (P::kHalves) {
      if (p.half(cur)) chunks_of(std::integral_constant<int, 4>{});
      else chunks_of(std::integral_constant<int, 8>{});
    } else {
      chunks_of(std::integral_constant<int, 8>{});
    }
    if (!more) break;
    stored = true;
    cur = nxt;
    more = p.next(nxt);
    if (more) p.fetch(nxt, lane, wave, fetched);
    int row = row0, col = col0;
    asm volatile("" : "+v"(row), "+v"(col));
    p.dest(cur, row, col, dest);
    __builtin_amdgcn_sched_barrier(0);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // loads past the last tile must land before the workgroup gives its LDS away
}
#endif

#if defined(__HIPCC__)
// ---- activations behind a tile ------------------------------------------------------------------------------------------------------------
// A lane activates 128 values behind its tile with nothing beside it (35 instructions each, what expf and a division take, are 9 us a tile).  So they are formed by a few instructions that end
// within kNear units in the last place of the form that a pass over memory has, and where a value lies that close to a boundary of its rounding to bfloat16 that form decides: all results
// are bit for bit those of the pass.  One in eight of a wave's stores of 512 has such a value; they are taken one per lane and round.  A scoring pass of 49152 rows through two int8 7B layers
// takes 31.00 ms, without the look at the rounding (one gate of 65536 rounds otherwise) 30.82, with passes of their own 32.18.
constexpr uint32_t kNear = 8;
typedef float f32x8_t __attribute__((ext_vector_type(8)));

__device__ __forceinline__ bool undecided(uint32_t bits) { return ((bits + 0x8000u + kNear) & 0xFFFFu) < 2 * kNear; }

// v: close to form(the eight bfloat16 values of `of`); those near a boundary become that.  (Vectors: of arrays the compiler makes memory, whose waits would be counted as a tile's loads.)
template <class Form>
__device__ __forceinline__ f32x8_t settled(f32x8_t v, u32x4_t of, Form form) {
  typedef uint16_t u16x2_t __attribute__((ext_vector_type(2)));
  typedef uint32_t u32x8_t __attribute__((ext_vector_type(8)));
  const u32x8_t bits = __builtin_bit_cast(u32x8_t, v);
  u16x2_t least = {0xFFFF, 0xFFFF};
#pragma unroll
  for (int i = 0; i < 4; ++i) {  // the lower halves of two values at a time
    const uint32_t low = __builtin_amdgcn_perm(bits[2 * i + 1], bits[2 * i], 0x05040100u);
    const u16x2_t at = __builtin_bit_cast(u16x2_t, low) + static_cast<uint16_t>(0x8000u + kNear);
    least = __builtin_elementwise_min(least, at);
  }
  if (__builtin_expect(__builtin_amdgcn_ballot_w64(least[0] < 2 * kNear || least[1] < 2 * kNear) == 0, 1)) return v;
  uint32_t todo = 0;
#pragma unroll
  for (int e = 0; e < 8; ++e) todo |= undecided(bits[e]) ? 1u << e : 0u;
  while (todo) {
    const int next = __builtin_ctz(todo), pair = next >> 1;
    uint32_t two = pair == 1 ? of[1] : of[0];
    two = pair == 2 ? of[2] : two;
    two = pair == 3 ? of[3] : two;
    const float y = form(__builtin_bit_cast(float, next & 1 ? two & 0xFFFF0000u : two << 16));
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = next == e ? y : v[e];
    todo &= todo - 1;
  }
  return v;
}

// g / (1 + exp(-g)) of a bfloat16 g, within three units in the last place of float32: a power of two whose exponent -g log2(e) is carried in two parts, and a reciprocal.  The denominator is in
// units of 2^16, so that it has a normal reciprocal wherever exp(-g) is finite, and so is g, of which no bit is lost and no product leaves float32.
__device__ __forceinline__ float near_silu(float g) {
  const float x = __builtin_amdgcn_fmed3f(g, -1e4f, 1e4f);
  const float t = x * -1.44269502f;
  const float r = __builtin_fmaf(x, -1.92596303e-8f, __builtin_fmaf(x, -1.44269502f, -t));
  const float d = __builtin_fmaf(__builtin_amdgcn_exp2f(t), __builtin_fmaf(r, 0x1p-16f * 0.693147181f, 0x1p-16f), 0x1p-16f);
  return g * 0x1p-16f * __builtin_amdgcn_rcpf(d);
}

// bf16( bf16(silu(g)) * u ) of eight bfloat16 values each, as e2h_silu_mul forms it
__device__ __forceinline__ u32x4_t gated(u32x4_t g, u32x4_t u) {
  const auto low = [](uint32_t b) { return __builtin_bit_cast(float, b << 16); };
  const auto high = [](uint32_t b) { return __builtin_bit_cast(float, b & 0xFFFF0000u); };
  f32x8_t v;
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = near_silu(e & 1 ? high(g[e >> 1]) : low(g[e >> 1]));
  v = settled(v, g, [](float z) { return z / (1.0f + expf(-z)); });
  u32x4_t out;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t act = f32x2_to_bf16_rne(v[2 * e], v[2 * e + 1]);
    out[e] = f32x2_to_bf16_rne(low(act) * low(u[e]), high(act) * high(u[e]));
  }
  return out;
}
#endif

// The tiles of one plain product, dealt to the XCDs in contiguous runs of equal length: panels of eight column blocks, all row
// blocks of a panel after each other, so that the 32 tiles at work on an XCD share four row blocks and eight column blocks.
// kCols: columns of y per tile, 256, or 128 of a pair of products (two rows of w each).
template <int kCols = kSide>
struct PlainWalk {
  static constexpr bool kHalves = false, kPairs = kCols != kSide;
  static constexpr int kPanel = 8;
  struct Tile {
    int rb, cb;
  };
  const uint16_t *x, *w;
  uint16_t *y;
  int M, N, K, t, end, stride;

  __device__ __forceinline__ PlainWalk(const uint16_t *x_, const uint16_t *w_, uint16_t *y_, int M_, int N_, int K_) : x(x_), w(w_), y(y_), M(M_), N(N_), K(K_) {
    const int64_t total = static_cast<int64_t>((M + 255) / 256) * ((N + kCols - 1) / kCols);
    const int xcd = blockIdx.x & 7;
    stride = static_cast<int>(gridDim.x >> 3);
    end = static_cast<int>(total * (xcd + 1) / 8);
    t = static_cast<int>(total * xcd / 8) + static_cast<int>(blockIdx.x >> 3) - stride;
  }
  __device__ __forceinline__ bool next(Tile &tile) {
    t += stride;
    if (t >= end) return false;
    const int R = (M + 255) / 256, C = (N + kCols - 1) / kCols, panel = t / (kPanel * R), at = t - panel * kPanel * R;
    const int wide = C - panel * kPanel < kPanel ? C - panel * kPanel : kPanel;
    tile.rb = at / wide;
    tile.cb = panel * kPanel + at - tile.rb * wide;
    return true;
  }
  __device__ __forceinline__ bool first(Tile &tile) { return next(tile); }
  __device__ __forceinline__ int chunks() const { return K / 64; }
  __device__ __forceinline__ __amdgpu_buffer_rsrc_t x_rsrc(const Tile &) const { return make_rsrc(x, static_cast<uint32_t>(static_cast<size_t>(M) * K * 2)); }
  __device__ __forceinline__ __amdgpu_buffer_rsrc_t w_rsrc(const Tile &) const { return make_rsrc(w, static_cast<uint32_t>(static_cast<size_t>(N) * K * (kPairs ? 4 : 2))); }
  // a tile's own rows of y: rows past M lie behind the buffer, where stores are dropped
  __device__ __forceinline__ __amdgpu_buffer_rsrc_t y_rsrc(const Tile &tile) const {
    const int rows = M - tile.rb * 256 < 256 ? M - tile.rb * 256 : 256;
    return make_rsrc(y + static_cast<size_t>(tile.rb) * 256 * N, static_cast<uint32_t>(rows) * static_cast<uint32_t>(N) * 2);
  }
  struct Fetch {};
  __device__ __forceinline__ void fetch(const Tile &, int, int, Fetch &) const {}
  __device__ __forceinline__ uint32_t x_at(const Tile &tile, const Fetch &, int, int row) const {
    const int m = tile.rb * 256 + row;
    return static_cast<uint32_t>(m < M ? m : M - 1) * static_cast<uint32_t>(K) * 2;
  }
  // column of y that column `col` (0 .. 255) of the tile's product goes into; the second matrix' rows of a pair stand behind the first one's
  __device__ __forceinline__ int out_col(const Tile &tile, int col) const { return tile.cb * kCols + (kPairs ? (col >> 7) * 64 + (col & 63) : col); }
  __device__ __forceinline__ uint32_t w_at(const Tile &tile, int col) const {
    const int n = out_col(tile, col);
    return (static_cast<uint32_t>(n < N ? n : N - 1) + (kPairs && (col & 64) ? static_cast<uint32_t>(N) : 0u)) * static_cast<uint32_t>(K) * 2;
  }
  __device__ __forceinline__ uint32_t y_at(const Tile &tile, int row, int col) const {
    const int n = out_col(tile, col);
    return n < N ? (static_cast<uint32_t>(row) * static_cast<uint32_t>(N) + static_cast<uint32_t>(n)) * 2 : kNowhere;
  }
};

// Workgroups of a walk over so many tiles: a CU each, an XCD's share alike.
inline unsigned grid_of(int64_t tiles) { return static_cast<unsigned>(8 * (tiles < 256 ? (tiles + 7) / 8 : 32)); }

}  // namespace gemm256
}  // namespace e2h
