// Mixture-of-experts feed-forward: router (e2h_seq_route) and squared-ReLU experts (e2h_seq_experts).
//
// Router: logits on v_mfma_f32_16x16x32_bf16 (products of bfloat16 values, float32 sums), waves split the width; then one wave per
// row picks the largest logits.
// Experts, a "slot" being one (row, choice) pair:
//   few rows    expert_step_kernel: a workgroup per expert in use (and 16 or 32 of its weight rows) finds the expert's slots itself
//               and streams those weights once; waves split K.  The shared expert is part of the same launch.
//   many rows   sort_slots_kernel orders the slots by expert, then expert_tiles_kernel: 256 x 128 outputs per workgroup, operands
//               brought into LDS by direct 16-byte loads (token rows gathered by the loads themselves); from 104 rows per expert on
//               expert_big_tiles_kernel: 256 x 256 outputs (e2h_gemm256.h).
//   otherwise   expert_plain_kernel on the vector units (float32, sizes that are not multiples of 8).
// Matrix products are transposed (weights are the A operand), so a lane holds four neighbouring outputs of one token.
#include "e2h_gemm256.h"
#include "e2h_seq_common.h"

namespace e2h {
namespace {

typedef __attribute__((address_space(3))) void lds_void;

constexpr int kMaxExperts = 1024, kMaxTop = 64;

__device__ __forceinline__ bf16x8_t load_fragment(const bf16_t *p, bool valid) {
  u32x4_t r = {0u, 0u, 0u, 0u};
  if (valid) r = *reinterpret_cast<const u32x4_t *>(p);
  return __builtin_bit_cast(bf16x8_t, r);
}

// ---- router ------------------------------------------------------------------------------------------------------------
// ET x TT tiles of 16 experts x 16 rows per workgroup, kWaves waves along the width.  A decode step has one workgroup per 16
// experts and waits for its loads: sixteen waves hold the loads of 4096 channels in flight at a time, eight half of that (4 rows,
// 64 experts: 7.4 us, with eight 8.1).  With many rows eight waves fill the chip.
template <int ET, int TT, int kWaves>
__global__ __launch_bounds__(64 * kWaves) void router_logits_kernel(const e2h_route_args a, int expert_groups) {
  __shared__ float part[kWaves][ET * TT][16][17];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 15, b4 = lane >> 4;
  const int e0 = (blockIdx.x % expert_groups) * ET * 16;
  const int64_t r0 = static_cast<int64_t>(blockIdx.x / expert_groups) * TT * 16;
  const int W = static_cast<int>(a.width), E = static_cast<int>(a.experts);
  const bf16_t *wp[ET], *xp[TT];
#pragma unroll
  for (int i = 0; i < ET; ++i) {
    const int e = e0 + 16 * i + c;
    wp[i] = static_cast<const bf16_t *>(a.router) + static_cast<size_t>(e < E ? e : E - 1) * W;
  }
#pragma unroll
  for (int j = 0; j < TT; ++j) {
    const int64_t r = r0 + 16 * j + c;
    xp[j] = static_cast<const bf16_t *>(a.x) + (r < a.rows ? r : a.rows - 1) * W;
  }
  f32x4_t acc[ET][TT];
#pragma unroll
  for (int i = 0; i < ET; ++i)
#pragma unroll
    for (int j = 0; j < TT; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  constexpr int U = ET * TT == 1 ? 8 : 4;
  const int steps = (W + 31) / 32;
  for (int s0 = wave * U; s0 < steps; s0 += kWaves * U) {
    bf16x8_t wf[U][ET], xf[U][TT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = 32 * (s0 + u) + 8 * b4;
#pragma unroll
      for (int i = 0; i < ET; ++i) wf[u][i] = load_fragment(wp[i] + k, k < W);
#pragma unroll
      for (int j = 0; j < TT; ++j) xf[u][j] = load_fragment(xp[j] + k, k < W);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int i = 0; i < ET; ++i)
#pragma unroll
        for (int j = 0; j < TT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[u][i], xf[u][j], acc[i][j], 0, 0, 0);
  }
#pragma unroll
  for (int i = 0; i < ET; ++i)
#pragma unroll
    for (int j = 0; j < TT; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) part[wave][i * TT + j][c][4 * b4 + e] = acc[i][j][e];
  __syncthreads();
  for (int n = threadIdx.x; n < ET * TT * 256; n += 64 * kWaves) {
    const int tile = n / 256, row = (n / 16) % 16, e = n % 16;
    const int64_t r = r0 + 16 * (tile % TT) + row;
    const int expert = e0 + 16 * (tile / TT) + e;
    if (r < a.rows && expert < E) {
      float v = a.bias ? a.bias[expert] : 0.f;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) v += part[w][tile][row][e];
      a.logits[r * E + expert] = v;
    }
  }
}

// one wave per (row, expert)
template <typename T>
__global__ __launch_bounds__(256) void router_logits_plain_kernel(const e2h_route_args a) {
  const int lane = threadIdx.x & 63;
  const int64_t item = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (item >= a.rows * a.experts) return;
  const int64_t r = item / a.experts, e = item % a.experts;
  const T *x = static_cast<const T *>(a.x) + r * a.width, *w = static_cast<const T *>(a.router) + e * a.width;
  float v = 0.f;
  for (int64_t k = lane; k < a.width; k += 64) v = __builtin_fmaf(to_f32(x[k]), to_f32(w[k]), v);
  v = wave_add(v);
  if (lane == 0) a.logits[item] = v + (a.bias ? a.bias[e] : 0.f);
}

// At most 64 experts, one wave per row, lane e holds expert e: its place among the row's experts is the number of experts ahead of
// it, which takes one lane read and two compares per expert and no round trips between the lanes.  Lane k ends up with the k-th
// choice, and the weights are summed in the order of the choices.  Picking
// the choices one after another with six exchanges each (the kernel below) took 7.6 us for 4 rows and 8 choices (16.3
// for 8192 rows), this takes 4.2 (9.4).
__global__ __launch_bounds__(256) void router_rank_kernel(const e2h_route_args a) {
  const int lane = threadIdx.x & 63, E = static_cast<int>(a.experts), top = static_cast<int>(a.top);
  const int64_t row = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (row >= a.rows) return;
  float z = lane < E ? a.logits[row * E + lane] : 0.f;
  if (!(z > -3e38f)) z = -3e38f;  // what is no number is chosen last
  int place = 0;
  for (int e = 0; e < E; ++e) {
    const float other = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, z), e));
    place += other > z || (other == z && e < lane);
  }
  if (lane >= E) place = lane;  // the experts hold the places 0 .. E - 1, so the places of all lanes are a permutation
  const int expert = __builtin_amdgcn_ds_permute(4 * place, lane);
  const float v = __builtin_bit_cast(float, __builtin_amdgcn_ds_permute(4 * place, __builtin_bit_cast(int, z)));
  const float largest = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 0));
  const float own = expf(v - largest);
  float sum = 0.f;
  for (int k = 0; k < top; ++k) sum += __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, own), k));
  if (lane < top) {
    a.chosen[row * top + lane] = expert;
    a.weights[row * top + lane] = own / sum;
  }
}

// More experts: one wave per row; lane l holds the logits of experts l, l + 64, ..; lane k ends up with the k-th choice
template <int PER>
__global__ __launch_bounds__(256) void router_choose_kernel(const e2h_route_args a) {
  const int lane = threadIdx.x & 63, E = static_cast<int>(a.experts), top = static_cast<int>(a.top);
  const int64_t row = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (row >= a.rows) return;
  float z[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int e = lane + 64 * i;
    z[i] = e < E ? a.logits[row * E + e] : 0.f;
    if (!(z[i] > -3e38f)) z[i] = -3e38f;  // what is no number is chosen last
  }
  uint32_t open = 0;  // bit i: expert lane + 64 i may still be chosen
#pragma unroll
  for (int i = 0; i < PER; ++i) open |= lane + 64 * i < E ? 1u << i : 0u;
  float mine = 0.f, largest = 0.f, sum = 0.f;
  int my_expert = 0;
  for (int k = 0; k < top; ++k) {
    float v = 0.f;
    int at = INT32_MAX;
#pragma unroll
    for (int i = 0; i < PER; ++i)
      if (((open >> i) & 1u) && (at == INT32_MAX || z[i] > v)) {
        v = z[i];
        at = lane + 64 * i;
      }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const float v2 = __shfl_xor(v, off);
      const int at2 = __shfl_xor(at, off);
      if (at2 != INT32_MAX && (at == INT32_MAX || v2 > v || (v2 == v && at2 < at))) {
        v = v2;
        at = at2;
      }
    }
    if ((at & 63) == lane) open &= ~(1u << (at >> 6));
    if (k == 0) largest = v;
    sum += expf(v - largest);
    if (k == lane) {
      mine = v;
      my_expert = at;
    }
  }
  if (lane < top) {
    a.chosen[row * top + lane] = my_expert;
    a.weights[row * top + lane] = expf(mine - largest) / sum;
  }
}

// ---- slots in the order of their experts --------------------------------------------------------------------------------
// One workgroup per expert: counts the slots of lower experts (where its list starts) and its own, then writes them in order.
__global__ __launch_bounds__(1024) void sort_slots_kernel(const int32_t *chosen, int slots, int experts, int32_t *order, int32_t *offsets) {
  __shared__ int below_of[16], own_of[16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, e = blockIdx.x;
  const int per = (slots + 1023) / 1024 * 64, begin = wave * per, end = begin + per < slots ? begin + per : slots;
  constexpr int kAhead = 8;  // loads in flight per lane
  int below = 0, own = 0;
  for (int i0 = begin + lane; i0 < end; i0 += 64 * kAhead) {
    int id[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) id[u] = i0 + 64 * u < end ? chosen[i0 + 64 * u] : -1;
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      below += id[u] >= 0 && id[u] < e;
      own += id[u] == e;
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    below += __shfl_xor(below, off);
    own += __shfl_xor(own, off);
  }
  if (lane == 0) {
    below_of[wave] = below;
    own_of[wave] = own;
  }
  __syncthreads();
  int base = 0, at = 0, total = 0;
#pragma unroll
  for (int w = 0; w < 16; ++w) {
    base += below_of[w];
    if (w < wave) at += own_of[w];
    total += own_of[w];
  }
  if (threadIdx.x == 0) {
    offsets[e] = base;
    if (e == experts - 1) offsets[experts] = base + total;
  }
  at += base;
  for (int i0 = begin; i0 < end; i0 += 64 * kAhead) {
    int id[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) id[u] = i0 + 64 * u + lane < end ? chosen[i0 + 64 * u + lane] : -1;
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const bool hit = id[u] == e;
      const uint64_t mask = __ballot(hit);
      if (hit) order[at + __popcll(mask & ((1ull << lane) - 1))] = i0 + 64 * u + lane;
      at += __popcll(mask);
    }
  }
}

// A workgroup's place in the list of output tiles, experts in order, all token tiles of a column tile after each other.  offsets NULL:
// one expert with `rows` rows.  Consecutive tiles go to one XCD (workgroups are dealt out to the eight XCDs in turn).
struct Tile {
  int expert, base, count, m, n;  // rows base .. base + count - 1 of the sorted order; tile m of them, column tile n; expert < 0: none
};

// tiles of expert e; all tiles
__device__ __forceinline__ int tiles_of(const int32_t *offsets, int experts, int rows, int tile_rows, int e) {
  if (e >= experts) return 0;
  const int n = offsets ? offsets[e + 1] - offsets[e] : rows;
  return (n + tile_rows - 1) / tile_rows;
}

__device__ __forceinline__ int count_tiles(const int32_t *offsets, int experts, int rows, int tile_rows, int n_tiles) {
  const int lane = threadIdx.x & 63;
  int total = 0;
  for (int e0 = 0; e0 < experts; e0 += 64) {
    int v = tiles_of(offsets, experts, rows, tile_rows, e0 + lane);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    total += v;
  }
  return __builtin_amdgcn_readfirstlane(total) * n_tiles;
}

// tile t, below the total
__device__ __forceinline__ Tile tile_at(const int32_t *offsets, int experts, int rows, int tile_rows, int n_tiles, int t) {
  const int lane = threadIdx.x & 63;
  Tile r = {-1, 0, 0, 0, 0};
  for (int e0 = 0; e0 < experts; e0 += 64) {
    const int mt = tiles_of(offsets, experts, rows, tile_rows, e0 + lane);
    int upto = mt;  // tiles of experts e0 .. e0 + lane
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int o = __shfl_up(upto, off);
      if (lane >= off) upto += o;
    }
    const uint64_t behind = __ballot(upto * n_tiles > t);
    if (behind) {
      const int l = __ffsll(static_cast<unsigned long long>(behind)) - 1;
      const int mine = __shfl(mt, l);
      t -= (__shfl(upto, l) - mine) * n_tiles;
      r.expert = e0 + l;
      r.base = offsets ? offsets[r.expert] : 0;
      r.count = offsets ? offsets[r.expert + 1] - r.base : rows;
      r.m = t % mine;
      r.n = t / mine;
      break;
    }
    t -= __shfl(upto, 63) * n_tiles;
  }
  // the same in all lanes, which the compiler cannot know
  return {__builtin_amdgcn_readfirstlane(r.expert), __builtin_amdgcn_readfirstlane(r.base), __builtin_amdgcn_readfirstlane(r.count),
          __builtin_amdgcn_readfirstlane(r.m), __builtin_amdgcn_readfirstlane(r.n)};
}

__device__ __forceinline__ Tile find_tile(const int32_t *offsets, int experts, int rows, int tile_rows, int n_tiles) {
  const int total = count_tiles(offsets, experts, rows, tile_rows, n_tiles);
  const int chunk = (total + 7) / 8, slot = blockIdx.x >> 3, t = static_cast<int>(blockIdx.x & 7) * chunk + slot;
  if (slot >= chunk || t >= total) return {-1, 0, 0, 0, 0};
  return tile_at(offsets, experts, rows, tile_rows, n_tiles, t);
}

// One matrix product over sorted rows: y[to(p)] = f(weight[e] x[from(p)]).  UP: x row = slot / top, y row = p, f = squared ReLU;
// else x row = p, y row = slot, f = identity.  order NULL: slot = p (the shared expert, top 1).
struct Product {
  const void *x, *weight;
  void *y;
  const int32_t *order, *offsets;
  int experts, rows, top, N, K, n_tiles;
  int64_t x_rows, weight_stride;
};

__device__ __forceinline__ int slot_of(const Product &p, int at) { return p.order ? p.order[at] : at; }

// 256 columns x 128 rows per workgroup, four waves of 128 x 64 (a fragment read from LDS feeds four or eight products: the LDS is what
// limits smaller ones), chunks of 32 along K in three LDS stages: a chunk is loaded two ahead of its use, and two workgroups share a
// CU, so one computes through the other's barriers, first loads and stores.
constexpr int kTileCols = 256, kTileRows = 128;

template <bool UP>
__global__ __launch_bounds__(256, 2) void expert_tiles_kernel(const Product p) {
  constexpr int kRow = 64, kTileW = kTileCols * kRow, kStage = kTileW + kTileRows * kRow;  // bytes: 32 values of a row, the weights, both operands
  constexpr int kLoadsW = 4, kLoadsX = 2;  // per wave and chunk
  __shared__ __attribute__((aligned(1024))) uint8_t lds[3 * kStage];
  const Tile tile = find_tile(p.offsets, p.experts, p.rows, kTileRows, p.n_tiles);
  if (tile.expert < 0) return;  // the whole workgroup, before any barrier
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = lane & 15, b4 = lane >> 4;
  const int wn = wave & 1, wm = wave >> 1;
  const int N = p.N, K = p.K, n0 = tile.n * kTileCols, m0 = tile.m * kTileRows;
  const int chunks = (K + 31) / 32;
  const __amdgpu_buffer_rsrc_t w_rsrc = make_rsrc(static_cast<const bf16_t *>(p.weight) + tile.expert * p.weight_stride,
                                                  static_cast<uint32_t>(static_cast<size_t>(N) * K * 2));
  const __amdgpu_buffer_rsrc_t x_rsrc = make_rsrc(p.x, static_cast<uint32_t>(p.x_rows * K * 2));

  // Wave w loads the 16-row blocks w, w + 4, .. of both operands: lane l row l / 4, to position l % 4 of the row.  The
  // 16-byte piece P of row r stands at position P ^ ((r / 4) % 4): 16 rows then read one piece from 16 different bank groups.
  const int piece = (lane & 3) ^ ((lane >> 4) & 3);
  uint32_t wsrc[kLoadsW], xsrc[kLoadsX];
#pragma unroll
  for (int i = 0; i < kLoadsW; ++i) {
    const int n = n0 + 16 * (wave + 4 * i) + (lane >> 2);
    wsrc[i] = static_cast<uint32_t>((static_cast<size_t>(n < N ? n : N - 1) * K + piece * 8) * 2);
  }
#pragma unroll
  for (int i = 0; i < kLoadsX; ++i) {
    const int m = m0 + 16 * (wave + 4 * i) + (lane >> 2), at = tile.base + (m < tile.count ? m : tile.count - 1);
    xsrc[i] = static_cast<uint32_t>((static_cast<size_t>(UP ? slot_of(p, at) / p.top : at) * K + piece * 8) * 2);
  }
  auto load = [&](int chunk, int stage) {
    const uint32_t back = chunk * 32 + piece * 8 < K ? 0u : static_cast<uint32_t>(piece) * 16;  // a piece beyond the row: its chunk's first one instead
#pragma unroll
    for (int i = 0; i < kLoadsW; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(w_rsrc, (lds_void *)(lds + stage * kStage + (wave + 4 * i) * 1024), 16, wsrc[i] - back,
                                               static_cast<uint32_t>(chunk) * kRow, 0, 0);
#pragma unroll
    for (int i = 0; i < kLoadsX; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(x_rsrc, (lds_void *)(lds + stage * kStage + kTileW + (wave + 4 * i) * 1024), 16, xsrc[i] - back,
                                               static_cast<uint32_t>(chunk) * kRow, 0, 0);
  };
  f32x4_t acc[8][4];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int at = (b4 ^ (c >> 2)) * 16;
  auto compute = [&](int stage, bool zero) {
    const uint8_t *lw = lds + stage * kStage + (128 * wn + c) * kRow + at, *lx = lds + stage * kStage + kTileW + (64 * wm + c) * kRow + at;
    const bf16x8_t none = __builtin_bit_cast(bf16x8_t, u32x4_t{0u, 0u, 0u, 0u});
    bf16x8_t wf[8], xf[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) xf[j] = *reinterpret_cast<const bf16x8_t *>(lx + j * 16 * kRow);
#pragma unroll
    for (int i = 0; i < 8; ++i) wf[i] = *reinterpret_cast<const bf16x8_t *>(lw + i * 16 * kRow);
    if (zero) {  // beyond the row
#pragma unroll
      for (int i = 0; i < 8; ++i) wf[i] = none;
#pragma unroll
      for (int j = 0; j < 4; ++j) xf[j] = none;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[i], xf[j], acc[i][j], 0, 0, 0);
  };
  load(0, 0);
  if (chunks > 1) load(1, 1);
  int stage = 0, next = 2;
  for (int i = 0; i + 1 < chunks; ++i) {
    // this chunk has landed (only the next one's loads may be open), and every wave is done with the stage loaded into below
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kLoadsW + kLoadsX) : "memory");
    if (i + 2 < chunks) load(i + 2, next);
    compute(stage, false);
    stage = stage == 2 ? 0 : stage + 1;
    next = next == 2 ? 0 : next + 1;
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  compute(stage, (chunks - 1) * 32 + 8 * b4 >= K);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int m = m0 + 64 * wm + 16 * j + c;
    if (m >= tile.count) continue;
    const int row = tile.base + m;
    bf16_t *y = static_cast<bf16_t *>(p.y) + static_cast<size_t>(UP ? row : slot_of(p, row)) * N;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int n = n0 + 128 * wn + 16 * i + 4 * b4;
      f32x4_t v = acc[i][j];
      if (UP) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float r = fmaxf(v[e], 0.f);
          v[e] = r * r;
        }
      }
      if (n < N) store4(y + n, v);
    }
  }
}

// The same on tiles of 256 x 256 (e2h_gemm256.h): a workgroup per CU walks its XCD's tiles.  8192 rows x 8 of 64 experts, 4096 x 1024:
// both products 904 us (1216 TFLOP/s), 1301 on the tiles above.  An expert's last tile forms the products of 128 rows where it has no more (both products
// 937 us with whole tiles throughout, a ninth of the products for rows that are not there); the last round of tiles fills half the chip in the up product.
template <bool UP>
struct ExpertWalk {
  typedef e2h::Tile Tile;
  static constexpr bool kHalves = true, kPairs = false;
  const Product &p;
  int t, end, stride;
  int begin, after;  // tiles before the present expert's first, and up to its last
  __amdgpu_buffer_rsrc_t y;

  __device__ __forceinline__ explicit ExpertWalk(const Product &product) : p(product) {
    const int total = count_tiles(p.offsets, p.experts, p.rows, gemm256::kSide, p.n_tiles), xcd = blockIdx.x & 7;
    stride = static_cast<int>(gridDim.x >> 3);
    end = static_cast<int>(static_cast<int64_t>(total) * (xcd + 1) / 8);
    t = static_cast<int>(static_cast<int64_t>(total) * xcd / 8) + static_cast<int>(blockIdx.x >> 3) - stride;
    y = make_rsrc(p.y, static_cast<uint32_t>(static_cast<size_t>(p.rows) * p.N * 2));
  }
  __device__ __forceinline__ int row_tiles(const Tile &tile) const { return (tile.count + gemm256::kSide - 1) / gemm256::kSide; }
  __device__ __forceinline__ bool first(Tile &tile) {
    t += stride;
    if (t >= end) return false;
    tile = tile_at(p.offsets, p.experts, p.rows, gemm256::kSide, p.n_tiles, t);
    const int rows = row_tiles(tile);
    begin = t - tile.n * rows - tile.m;
    after = begin + rows * p.n_tiles;
    return true;
  }
  // The search above would wait for every load and store under way (its own are behind them) and then for a dozen exchanges between
  // lanes.  From tile to tile a workgroup passes few experts: their ends come through the scalar cache.  With that, and the rows of the
  // tile's outputs no longer waited for behind the next tile's first loads, the down product of 18 tiles per CU took 483 us instead
  // of 504, the up product of 4.5 tiles, where it is a tile's 64 chunks that count, 452 instead of 460.
  __device__ __forceinline__ bool next(Tile &tile) {
    typedef const __attribute__((address_space(4))) int32_t *scalar_ints;
    t += stride;
    if (t >= end) return false;
    while (t >= after && tile.expert + 1 < p.experts) {
      ++tile.expert;
      tile.base += tile.count;
      tile.count = reinterpret_cast<scalar_ints>(reinterpret_cast<uintptr_t>(p.offsets))[tile.expert + 1] - tile.base;
      begin = after;
      after += row_tiles(tile) * p.n_tiles;
    }
    const int rows = row_tiles(tile);
    tile.n = (t - begin) / rows;
    tile.m = (t - begin) - tile.n * rows;
    return true;
  }
  __device__ __forceinline__ bool half(const Tile &tile) const { return tile.count - tile.m * gemm256::kSide <= gemm256::kSide / 2; }
  __device__ __forceinline__ int chunks() const { return p.K / 64; }
  __device__ __forceinline__ __amdgpu_buffer_rsrc_t x_rsrc(const Tile &) const { return make_rsrc(p.x, static_cast<uint32_t>(p.x_rows * p.K * 2)); }
  __device__ __forceinline__ __amdgpu_buffer_rsrc_t w_rsrc(const Tile &tile) const {
    return make_rsrc(static_cast<const bf16_t *>(p.weight) + tile.expert * p.weight_stride, static_cast<uint32_t>(static_cast<size_t>(p.N) * p.K * 2));
  }
  __device__ __forceinline__ int sorted_row(const Tile &tile, int row) const {
    const int m = tile.m * gemm256::kSide + row;
    return tile.base + (m < tile.count ? m : tile.count - 1);
  }
  struct Fetch {
    int slot[8];
  };
  __device__ __forceinline__ void fetch(const Tile &tile, int lane, int wave, Fetch &f) const {
    if (!UP) return;
#pragma unroll
    for (int i = 0; i < 8; ++i) f.slot[i] = slot_of(p, sorted_row(tile, 8 * (wave + 4 * i) + (lane >> 3)));
  }
  __device__ __forceinline__ uint32_t x_at(const Tile &tile, const Fetch &f, int i, int row) const {
    const uint32_t at = static_cast<uint32_t>(UP ? f.slot[i] / p.top : sorted_row(tile, row)) * static_cast<uint32_t>(p.K) * 2;
    return tile.m * gemm256::kSide + row < tile.count ? at : gemm256::kNowhere - 256;  // rows that are not there: zeros, from no memory
  }
  __device__ __forceinline__ uint32_t w_at(const Tile &tile, int col) const {
    const int n = tile.n * gemm256::kSide + col;
    return static_cast<uint32_t>(n < p.N ? n : p.N - 1) * static_cast<uint32_t>(p.K) * 2;
  }
  struct Dest {
    int slot[UP ? 1 : 8];
  };
  __device__ __forceinline__ void dest(const Tile &tile, int row, int, Dest &d) const {
    if (UP) return;
#pragma unroll
    for (int j = 0; j < 8; ++j) d.slot[UP ? 0 : j] = slot_of(p, sorted_row(tile, row + 32 * j));
  }
  __device__ __forceinline__ void store(const Tile &tile, const Dest &d, int j, int, int row, int col, float (&v)[8]) const {
    if (UP) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float r = fmaxf(v[e], 0.f);
        v[e] = r * r;
      }
    }
    const int n = tile.n * gemm256::kSide + col, out = UP ? tile.base + tile.m * gemm256::kSide + row : d.slot[UP ? 0 : j];
    const uint32_t at = (static_cast<uint32_t>(out) * static_cast<uint32_t>(p.N) + static_cast<uint32_t>(n)) * 2;
    const bool there = tile.m * gemm256::kSide + row < tile.count && n < p.N;
    __builtin_amdgcn_raw_buffer_store_b128(u32x4_t{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]), pack_bf16(v[4], v[5]), pack_bf16(v[6], v[7])}, y,
                                           there ? at : gemm256::kNowhere, 0, 0);
  }
};

template <bool UP>
__global__ __launch_bounds__(256, 1) void expert_big_tiles_kernel(const Product p) {
#if defined(__HIP_DEVICE_COMPILE__)
  __shared__ __attribute__((aligned(1024))) uint8_t lds[gemm256::kRing];
  ExpertWalk<UP> tiles(p);
  gemm256::walk<false>(tiles, lds);
#endif
}

// 32 rows x 32 columns per workgroup, float32 products
template <typename T, bool UP>
__global__ __launch_bounds__(256) void expert_plain_kernel(const Product p) {
  __shared__ float sx[32][33], sw[32][33];
  const Tile tile = find_tile(p.offsets, p.experts, p.rows, 32, p.n_tiles);
  if (tile.expert < 0) return;
  const int N = p.N, K = p.K, n0 = tile.n * 32, m0 = tile.m * 32, tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  const T *w = static_cast<const T *>(p.weight) + tile.expert * p.weight_stride;
  float acc[2][2] = {{0.f, 0.f}, {0.f, 0.f}};
  for (int k0 = 0; k0 < K; k0 += 32) {
    for (int i = threadIdx.x; i < 1024; i += 256) {
      const int r = i / 32, k = k0 + i % 32;
      float xv = 0.f, wv = 0.f;
      if (k < K) {
        if (m0 + r < tile.count) {
          const int at = tile.base + m0 + r;
          xv = to_f32(static_cast<const T *>(p.x)[static_cast<size_t>(UP ? slot_of(p, at) / p.top : at) * K + k]);
        }
        if (n0 + r < N) wv = to_f32(w[static_cast<size_t>(n0 + r) * K + k]);
      }
      sx[r][i % 32] = xv;
      sw[r][i % 32] = wv;
    }
    __syncthreads();
    for (int k = 0; k < 32; ++k)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_fmaf(sx[ty + 16 * i][k], sw[tx + 16 * j][k], acc[i][j]);
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int m = m0 + ty + 16 * i;
    if (m >= tile.count) continue;
    const int at = tile.base + m;
    T *y = static_cast<T *>(p.y) + static_cast<size_t>(UP ? at : slot_of(p, at)) * N;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int n = n0 + tx + 16 * j;
      float v = acc[i][j];
      if (UP) {
        v = fmaxf(v, 0.f);
        v *= v;
      }
      if (n < N) y[n] = from_f32<T>(v);
    }
  }
}

// ---- few rows --------------------------------------------------------------------------------------------------------------
// Workgroup = one list (an expert, or with by_slot the expert of a slot, if no earlier slot has the same) and 16 RT weight rows; the
// workgroups behind those belong to the shared expert.  hidden [slots, ff], shared_hidden [rows, shared_ff].
constexpr int kStepSlots = 1024;

template <bool UP, int RT>
__global__ __launch_bounds__(256) void expert_step_kernel(const e2h_experts_args a, bf16_t *hidden, bf16_t *shared_hidden, int lists, int tiles, int by_slot) {
  constexpr int U = RT == 1 ? 8 : 4;
  __shared__ int list[kStepSlots], found, leader;
  __shared__ float part[4][RT][16][17];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 15, b4 = lane >> 4;
  const int rows = static_cast<int>(a.rows), top = static_cast<int>(a.top), width = static_cast<int>(a.width);
  const int id = blockIdx.x;
  const bool shared = id >= lists * tiles;
  const int item = shared ? 0 : id / tiles, tile = shared ? id - lists * tiles : id % tiles;
  const int F = static_cast<int>(shared ? a.shared_ff : a.ff);
  int e = item, count = rows;
  if (!shared) {
    if (by_slot) {
      e = a.chosen[item];
      if (e < 0 || e >= a.experts) return;  // the whole workgroup
    }
    if (tid == 0) {
      found = 0;
      leader = INT32_MAX;
    }
    __syncthreads();
    for (int s = tid; s < rows * top; s += 256)
      if (a.chosen[s] == e) {
        list[atomicAdd(&found, 1)] = s;
        atomicMin(&leader, s);
      }
    __syncthreads();
    count = found;
    if (count == 0 || (by_slot && leader != item)) return;
  }
  const int K = UP ? width : F, N = UP ? F : width;
  const bf16_t *weight = static_cast<const bf16_t *>(UP ? (shared ? a.shared_up : a.up) : (shared ? a.shared_down : a.down)) +
                         (shared ? 0 : static_cast<size_t>(e) * N * K);
  const bf16_t *xin = UP ? static_cast<const bf16_t *>(a.x) : shared ? shared_hidden : hidden;
  bf16_t *yout = UP ? (shared ? shared_hidden : hidden) : static_cast<bf16_t *>(shared ? a.shared_out : a.out);
  const int n0 = tile * 16 * RT;
  const bf16_t *wp[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r) wp[r] = weight + static_cast<size_t>(n0 + 16 * r + c < N ? n0 + 16 * r + c : N - 1) * K;
  const int steps = (K + 31) / 32;
  for (int c0 = 0; c0 < count; c0 += 16) {
    const int ti = c0 + c < count ? c0 + c : count - 1, s = shared ? ti : list[ti];
    const bf16_t *xp = xin + static_cast<size_t>(UP && !shared ? s / top : s) * K;
    f32x4_t acc[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) acc[r] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    for (int s0 = wave * U; s0 < steps; s0 += 4 * U) {
      bf16x8_t wf[U][RT], xf[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = 32 * (s0 + u) + 8 * b4;
#pragma unroll
        for (int r = 0; r < RT; ++r) wf[u][r] = load_fragment(wp[r] + k, k < K);
        xf[u] = load_fragment(xp + k, k < K);
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int r = 0; r < RT; ++r) acc[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[u][r], xf[u], acc[r], 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i) part[wave][r][c][4 * b4 + i] = acc[r][i];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      const int t = tid >> 4, n = n0 + 16 * r + (tid & 15);
      if (c0 + t < count && n < N) {
        float v = part[0][r][t][tid & 15] + part[1][r][t][tid & 15] + part[2][r][t][tid & 15] + part[3][r][t][tid & 15];
        if (UP) {
          v = fmaxf(v, 0.f);
          v *= v;
        }
        yout[static_cast<size_t>(shared ? c0 + t : list[c0 + t]) * N + n] = from_f32<bf16_t>(v);
      }
    }
    __syncthreads();
  }
}

// ---- choice of the form, scratch -------------------------------------------------------------------------------------------------
constexpr int kPlain = 1, kStep = 2, kTiles = 3;

int expert_form(const e2h_experts_args &a) {
  const int64_t slots = a.rows * a.top, most = static_cast<int64_t>(UINT32_MAX) / 2;
  bool vec = a.dtype == E2H_SEQ_BF16 && a.width % 8 == 0 && a.ff % 8 == 0 && aligned16(a.x) && aligned16(a.up) && aligned16(a.down) &&
             aligned16(a.out) && aligned16(a.scratch);
  if (a.shared_up) vec = vec && a.shared_ff % 8 == 0 && aligned16(a.shared_up) && aligned16(a.shared_down) && aligned16(a.shared_out);
  const bool tiles = vec && a.rows * a.width <= most && slots * a.ff <= most && a.ff * a.width <= most &&
                     (!a.shared_up || (a.rows * a.shared_ff <= most && a.shared_ff * a.width <= most));
  const bool step = vec && slots <= kStepSlots;
  const int want = seq_options().expert_form;
  if (want == kPlain || (want == kStep && step) || (want == kTiles && tiles)) return want;
  // few rows per expert in use: the launch reads weights, not activations
  if (step && (slots <= 4 * a.experts || slots <= 256)) return kStep;
  return tiles ? kTiles : kPlain;
}

struct Scratch {
  int64_t hidden, shared_hidden, order, offsets, total;
};

Scratch scratch_of(const e2h_experts_args &a) {
  auto up = [](int64_t n) { return (n + 255) / 256 * 256; };
  const int64_t slots = a.rows * a.top, size = a.dtype == E2H_SEQ_BF16 ? 2 : 4;
  Scratch s;
  s.hidden = 0;
  s.shared_hidden = s.hidden + up(slots * a.ff * size);
  s.order = s.shared_hidden + (a.shared_up ? up(a.rows * a.shared_ff * size) : 0);
  s.offsets = s.order + up(slots * 4);
  s.total = s.offsets + up((a.experts + 1) * 4);
  return s;
}

int check_experts(const e2h_experts_args &a) {
  if (a.dtype != E2H_SEQ_BF16 && a.dtype != E2H_SEQ_F32) return E2H_ERR_BAD_SHAPE;
  if (a.rows < 1 || a.width < 1 || a.experts < 1 || a.experts > kMaxExperts || a.top < 1 || a.top > kMaxTop || a.top > a.experts || a.ff < 1 ||
      a.width > INT32_MAX / 8 || a.ff > INT32_MAX / 8)
    return E2H_ERR_BAD_SHAPE;
  if (a.shared_up && (a.shared_ff < 1 || a.shared_ff > INT32_MAX / 8)) return E2H_ERR_BAD_SHAPE;
  const int64_t slots = a.rows * a.top, widest = a.width > a.ff ? a.width : a.ff, most = a.shared_up && a.shared_ff > widest ? a.shared_ff : widest;
  if (slots > INT32_MAX / 2 || (slots / 32 + a.experts + 1) * ((most + 31) / 32) > INT32_MAX / 2) return E2H_ERR_BAD_SHAPE;
  return E2H_OK;
}

// 256-row tiles: from 24 rows per expert on, where rows that are not there cost half a tile at most, and with enough of them for half the CUs, below which two workgroups per CU of the other
// form divide the work better.  Both products, us, tiles of 128 / of 256, the same number of rows for every expert on average: 64 experts, 4096 x 1024, 24 rows each 236 / 233, 64 256 / 252,
// 96 272 / 263, 256 381 / 360; 32 experts, 2048 x 1024, 24 rows 72 / 72, 64 78 / 76, 96 84 / 81.  Rows by Zipf's law, 64 experts: 24 rows on average 313 / 239, 32 314 / 242, but 48 310 / 317,
// 64 325 / 333 and 96 327 / 335; by its square 32 304 / 242, 48 292 / 313, 64 313 / 329, 96 318 / 330, 128 362 / 349.  Below 24 the two are within 2 % where experts have equal shares
// (8 rows 227 / 227, 16 232 / 228; 32 experts, 16 rows 69 / 69), and few uneven ones gain (20 rows by Zipf's law 313 / 234).
bool big_tiles_pay(const Product &p) {
  const int64_t tiles = (static_cast<int64_t>(p.rows) / gemm256::kSide + (p.experts + 1) / 2) * p.n_tiles;
  return p.K % 64 == 0 && p.K >= gemm256::kLeastK && static_cast<int64_t>(p.rows) * p.N <= static_cast<int64_t>(UINT32_MAX) / 2 - 16 && p.rows >= 24LL * p.experts && tiles >= 128;
}

template <bool UP>
void launch_product(Product p, int form, bool bf16, hipStream_t s) {
  const int cols = form == kTiles ? kTileCols : 32, side = form == kTiles ? kTileRows : 32;
  p.n_tiles = (p.N + cols - 1) / cols;
  if (form == kTiles && big_tiles_pay(p)) {
    hipLaunchKernelGGL((expert_big_tiles_kernel<UP>), dim3(256), dim3(256), 0, s, p);
    return;
  }
  const int64_t tiles = (static_cast<int64_t>(p.rows) / side + p.experts) * p.n_tiles;  // at least one per expert and begun block of rows
  const dim3 grid(static_cast<unsigned>((tiles + 7) / 8 * 8)), block(256);
  if (form == kTiles) hipLaunchKernelGGL((expert_tiles_kernel<UP>), grid, block, 0, s, p);
  else if (bf16) hipLaunchKernelGGL((expert_plain_kernel<bf16_t, UP>), grid, block, 0, s, p);
  else hipLaunchKernelGGL((expert_plain_kernel<float, UP>), grid, block, 0, s, p);
}

template <bool UP>
void launch_step(const e2h_experts_args &a, bf16_t *hidden, bf16_t *shared_hidden, hipStream_t s) {
  const int64_t slots = a.rows * a.top, N = UP ? a.ff : a.width, NS = a.shared_up ? (UP ? a.shared_ff : a.width) : 0;
  const int by_slot = slots < a.experts;
  const int lists = static_cast<int>(by_slot ? slots : a.experts);
  // two row tiles per workgroup (they share the token fragments) once that still leaves several workgroups per CU
  const int rt = lists * (N / 32) + NS / 32 >= 2048 ? 2 : 1;
  const int tiles = static_cast<int>((N + 16 * rt - 1) / (16 * rt)), shared_tiles = static_cast<int>((NS + 16 * rt - 1) / (16 * rt));
  const dim3 grid(static_cast<unsigned>(lists * tiles + shared_tiles)), block(256);
  if (rt == 2) hipLaunchKernelGGL((expert_step_kernel<UP, 2>), grid, block, 0, s, a, hidden, shared_hidden, lists, tiles, by_slot);
  else hipLaunchKernelGGL((expert_step_kernel<UP, 1>), grid, block, 0, s, a, hidden, shared_hidden, lists, tiles, by_slot);
}

}  // namespace
}  // namespace e2h

using namespace e2h;

extern "C" int e2h_seq_route(const e2h_route_args *a, void *stream) {
  if (!a || !a->x || !a->router || !a->logits || !a->chosen || !a->weights) return E2H_ERR_NULL_POINTER;
  if (a->dtype != E2H_SEQ_BF16 && a->dtype != E2H_SEQ_F32) return E2H_ERR_BAD_SHAPE;
  if (a->rows < 1 || a->width < 1 || a->width > INT32_MAX / 8 || a->experts < 1 || a->experts > kMaxExperts || a->top < 1 || a->top > kMaxTop ||
      a->top > a->experts || a->rows * a->experts > INT32_MAX / 2)
    return E2H_ERR_BAD_SHAPE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int E = static_cast<int>(a->experts);
  if (a->dtype == E2H_SEQ_BF16 && a->width % 8 == 0 && aligned16(a->x) && aligned16(a->router)) {
    if (a->rows >= 1024) {
      const int groups = (E + 63) / 64;
      hipLaunchKernelGGL((router_logits_kernel<4, 2, 8>), dim3(static_cast<unsigned>((a->rows + 31) / 32 * groups)), dim3(512), 0, s, *a, groups);
    } else {
      const int groups = (E + 15) / 16;
      hipLaunchKernelGGL((router_logits_kernel<1, 1, 16>), dim3(static_cast<unsigned>((a->rows + 15) / 16 * groups)), dim3(1024), 0, s, *a, groups);
    }
  } else {
    const dim3 grid(static_cast<unsigned>((a->rows * E + 3) / 4)), block(256);
    if (a->dtype == E2H_SEQ_BF16) hipLaunchKernelGGL(router_logits_plain_kernel<bf16_t>, grid, block, 0, s, *a);
    else hipLaunchKernelGGL(router_logits_plain_kernel<float>, grid, block, 0, s, *a);
  }
  const dim3 grid(static_cast<unsigned>((a->rows + 3) / 4)), block(256);
  if (E <= 64) hipLaunchKernelGGL(router_rank_kernel, grid, block, 0, s, *a);
  else if (E <= 256) hipLaunchKernelGGL(router_choose_kernel<4>, grid, block, 0, s, *a);
  else hipLaunchKernelGGL(router_choose_kernel<16>, grid, block, 0, s, *a);
  return launch_status();
}

extern "C" int64_t e2h_seq_experts_scratch_bytes(const e2h_experts_args *a) {
  if (!a) return E2H_ERR_NULL_POINTER;
  const int bad = check_experts(*a);
  return bad ? bad : scratch_of(*a).total;
}

extern "C" int e2h_seq_experts(const e2h_experts_args *a, void *stream) {
  if (!a || !a->x || !a->chosen || !a->up || !a->down || !a->out || (a->shared_up && (!a->shared_down || !a->shared_out))) return E2H_ERR_NULL_POINTER;
  const int bad = check_experts(*a);
  if (bad) return bad;
  const Scratch l = scratch_of(*a);
  if (!a->scratch) return E2H_ERR_NULL_POINTER;
  if (a->scratch_bytes < l.total) return E2H_ERR_SCRATCH_TOO_SMALL;
  hipStream_t s = static_cast<hipStream_t>(stream);
  uint8_t *scratch = static_cast<uint8_t *>(a->scratch);
  const int form = expert_form(*a);
  if (form == kStep) {
    bf16_t *hidden = reinterpret_cast<bf16_t *>(scratch + l.hidden), *shared_hidden = reinterpret_cast<bf16_t *>(scratch + l.shared_hidden);
    launch_step<true>(*a, hidden, shared_hidden, s);
    launch_step<false>(*a, hidden, shared_hidden, s);
    return launch_status();
  }
  const bool bf16 = a->dtype == E2H_SEQ_BF16;
  const int slots = static_cast<int>(a->rows * a->top), E = static_cast<int>(a->experts);
  int32_t *order = reinterpret_cast<int32_t *>(scratch + l.order), *offsets = reinterpret_cast<int32_t *>(scratch + l.offsets);
  hipLaunchKernelGGL(sort_slots_kernel, dim3(static_cast<unsigned>(E)), dim3(1024), 0, s, a->chosen, slots, E, order, offsets);
  const int W = static_cast<int>(a->width), F = static_cast<int>(a->ff), top = static_cast<int>(a->top), rows = static_cast<int>(a->rows);
  void *hidden = scratch + l.hidden;
  launch_product<true>({a->x, a->up, hidden, order, offsets, E, slots, top, F, W, 0, a->rows, a->ff * a->width}, form, bf16, s);
  launch_product<false>({hidden, a->down, a->out, order, offsets, E, slots, top, W, F, 0, slots, a->ff * a->width}, form, bf16, s);
  if (a->shared_up) {
    void *sh = scratch + l.shared_hidden;
    const int SF = static_cast<int>(a->shared_ff);
    launch_product<true>({a->x, a->shared_up, sh, nullptr, nullptr, 1, rows, 1, SF, W, 0, a->rows, 0}, form, bf16, s);
    launch_product<false>({sh, a->shared_down, a->shared_out, nullptr, nullptr, 1, rows, 1, W, SF, 0, a->rows, 0}, form, bf16, s);
  }
  return launch_status();
}
