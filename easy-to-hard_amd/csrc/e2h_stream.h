// y = x W^T for up to 64 rows of bfloat16 x and row-major weights of 8 or 16 bits that are streamed from HBM exactly once: the
// decode-batch matmul of int8 linears (e2h_int8_stream.hip) and of bfloat16 ones (e2h_seq_linear.hip).
//
// A workgroup is eight waves that split K and all work on the same T tiles of 16 weight rows, so that a CU streams 16 T rows and
// reads x once.  The split of K over the waves of a workgroup depends on K alone, so with one slice a row's result depends neither on the rows
// beside it nor on N, and every epilogue sees the same sums.  (Slices over several workgroups, which e2h_seq_linear takes for some shapes,
// sum in another order: there a row's result changes by float32 rounding with the choice.)  The waves meet once, at the end: wave w adds and finishes the (column tile, row tile) units w,
// w + 8, .. in k order.
//
// Everything a wave needs passes as units of 2 KB -- 16 rows of x or of a weight tile, 128 bytes each -- through a ring of its own in
// LDS, written by loads that never touch a register.  Eight lanes fetch the 128 bytes of one row, so that every request is a whole
// cache line; operands read straight into registers in matrix order (16 rows x 64 bytes per load) hold a CU to two thirds of
// that rate.  The 16-byte pieces of row r stand at piece ^ (r / 2 mod 8), which makes the operand reads conflict-free.  Waits count
// loads, there is no barrier in the loop.
//
// v_mfma_f32_16x16x32_bf16: lane 16 b + c holds weight row c and activation row c of its tile.  Rows past N and past M and bytes past K
// are sent out of the buffer's range: they return zeros and move no data.
#pragma once

#include <type_traits>

#include "e2h_common.h"

namespace e2h {
namespace stream {

// One row whose RMSNorm is x, formed by every workgroup for itself behind the requests for its first weights, in the round trip that those take as well.
// h = bf16(x + term), term = bf16(sum of the slices) or bf16(bf16(sum) * column scale), or h = x where there are no partial sums; rounding points and orders of sums are those of
// e2h_add_rmsnorm_partials.  Workgroup 0 stores h.  A step of one sequence through four int8 7B layers and the head, nine such products: 281 us with the norms as launches of their
// own (2.8 each), 268.  With two rows what every workgroup reads and does for itself takes as long as the launch (two layers of 7B, 163 us and 164).
struct RowNorm {
  const uint16_t *x;
  const float *partials;       // [slices][K], null: h = x
  const uint16_t *col_scales;  // may be null
  const uint16_t *weight;
  uint16_t *h_out;
  int slices;                  // 1 or 2
  float eps;
};
struct NoNorm {};
constexpr int kNormPieces = 2, kNormPiece = 4096;  // pieces of the row, eight values per thread each; of rows between 2048 and 4096 pieces of 2048 for half of the threads, whose sums run over both,
                                                   // as in the norm's own launch
constexpr int kNormSums = 128, kNormBytes = kNormSums + kNormPieces * kNormPiece * 2;  // LDS: the waves' sums of squares, the row
inline bool norm_fits(int64_t M, int64_t K) { return M == 1 && K >= 128 && K % 128 == 0 && K <= kNormPieces * kNormPiece; }

constexpr int64_t kMaxBytes = int64_t{1} << 31;  // of a buffer: offsets of 2^31 are what is sent out of range
constexpr int kWaves = 8;
constexpr int kMaxUnits = 16;  // (column tile, row tile) pairs of a workgroup: 8 KB of LDS each when the waves meet
constexpr int kUnitBytes = 2048, kRing = 8;  // per wave: 14 KB on their way while 2 KB are in use (18 KB measured the same)

// exact: an int8 value has 8 significant bits, so the high half of its float32 is its bfloat16
__device__ __forceinline__ uint32_t pack_exact(float lo, float hi) {
  return (__builtin_bit_cast(uint32_t, lo) >> 16) | (__builtin_bit_cast(uint32_t, hi) & 0xFFFF0000u);
}

struct Int8Weights {
  static constexpr int kBytes = 1, kXUnits = 2;  // bytes per weight, units of 64 activations per step of 128 bytes of weights
  // operand i of the piece
  static __device__ __forceinline__ bf16x8_t operand(const u32x4_t &w, int i) {
    u32x4_t u;
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      const uint32_t v = w[2 * i + d];
      u[2 * d] = pack_exact(static_cast<float>(static_cast<int8_t>(v)), static_cast<float>(static_cast<int8_t>(v >> 8)));
      u[2 * d + 1] = pack_exact(static_cast<float>(static_cast<int8_t>(v >> 16)), static_cast<float>(static_cast<int8_t>(v >> 24)));
    }
    return __builtin_bit_cast(bf16x8_t, u);
  }
};

struct Bf16Weights {
  static constexpr int kBytes = 2, kXUnits = 1;
  static __device__ __forceinline__ bf16x8_t operand(const u32x4_t &w, int) { return __builtin_bit_cast(bf16x8_t, w); }
};

struct Args {
  const uint16_t *x;  // [M][K]
  const void *w, *w2; // [N][K]; w2: the second matrix of a gated epilogue
  int M, N, K;
};

typedef __attribute__((address_space(3))) void lds_void;

// until at most n (a constant once the loop around the call is unrolled) of this wave's loads are out
__device__ __forceinline__ void wait_loads(int n) {
  switch (n) {
#define E2H_WAIT(N) \
  case N: asm volatile("s_waitcnt vmcnt(" #N ")" ::: "memory"); break;
    E2H_WAIT(7) E2H_WAIT(8) E2H_WAIT(9) E2H_WAIT(10) E2H_WAIT(11) E2H_WAIT(12) E2H_WAIT(13) E2H_WAIT(14)
#undef E2H_WAIT
    default: asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
}

// What a thread holds of the row to be normalised: eight values of every piece, all requested before anything is waited for.
struct NormLoads {
  u32x4_t x[kNormPieces], w[kNormPieces], cs[kNormPieces];
  f32x4_t lo[kNormPieces][2], hi[kNormPieces][2];

  static __device__ __forceinline__ bool halves(int K) { return K > kNormPiece / 2 && K < kNormPiece; }
  static __device__ __forceinline__ int span(int K) { return halves(K) ? kNormPiece / 2 : kNormPiece; }
  // this thread's place in piece p, K where it has none
  static __device__ __forceinline__ int place(int K, int p) {
    const int own = static_cast<int>(threadIdx.x) * 8, i = p * span(K) + own;
    return own < span(K) && i < K ? i : K;
  }

  __device__ __forceinline__ void request(const RowNorm &n, int K) {
#pragma unroll
    for (int p = 0; p < kNormPieces; ++p) {
      const int i = place(K, p), at = i < K ? i : 0;  // past the row: its first piece, not used
      if (K <= p * span(K)) break;
      x[p] = *reinterpret_cast<const u32x4_t *>(n.x + at);
      if (n.partials) {
        const float *const from = n.partials + at, *const other = from + (n.slices > 1 ? K : 0);
        lo[p][0] = *reinterpret_cast<const f32x4_t *>(from);
        hi[p][0] = *reinterpret_cast<const f32x4_t *>(from + 4);
        lo[p][1] = *reinterpret_cast<const f32x4_t *>(other);
        hi[p][1] = *reinterpret_cast<const f32x4_t *>(other + 4);
        if (n.col_scales) cs[p] = *reinterpret_cast<const u32x4_t *>(n.col_scales + at);
      }
      w[p] = *reinterpret_cast<const u32x4_t *>(n.weight + at);
    }
  }

  // the normalised row to lds + kNormSums, the waves' sums of squares in front of it
  __device__ __forceinline__ void finish(const RowNorm &n, int K, uint8_t *lds, bool store) {
    float *const sums = reinterpret_cast<float *>(lds);
    const auto low = [](uint32_t v) { return __builtin_bit_cast(float, v << 16); };
    const auto high = [](uint32_t v) { return __builtin_bit_cast(float, v & 0xFFFF0000u); };
    float ss = 0.f;
#pragma unroll
    for (int p = 0; p < kNormPieces; ++p) {
      const int i = place(K, p);
      float wave = 0.f;
      if (!halves(K)) ss = 0.f;
      if (K > p * span(K)) {
        if (n.partials) {
          f32x4_t a = lo[p][0], b = hi[p][0];
          if (n.slices > 1) a += lo[p][1], b += hi[p][1];
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            float t0 = j < 2 ? a[2 * j] : b[2 * j - 4], t1 = j < 2 ? a[2 * j + 1] : b[2 * j - 3];
            if (n.col_scales) t0 = bf16_round(t0) * low(cs[p][j]), t1 = bf16_round(t1) * high(cs[p][j]);
            x[p][j] = f32x2_to_bf16_rne(low(x[p][j]) + bf16_round(t0), high(x[p][j]) + bf16_round(t1));
          }
          if (store && i < K) *reinterpret_cast<u32x4_t *>(n.h_out + i) = x[p];
        }
        if (i < K) {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float h0 = low(x[p][j]), h1 = high(x[p][j]);
            ss = __builtin_fmaf(h0, h0, ss);
            ss = __builtin_fmaf(h1, h1, ss);
          }
        }
        wave = ss;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) wave += __shfl_xor(wave, off);
      }
      if ((threadIdx.x & 63) == 0) sums[p * kWaves + (threadIdx.x >> 6)] = p == 0 && halves(K) ? 0.f : wave;
    }
    lds_barrier();
    float sum = 0.f;
#pragma unroll
    for (int q = 0; q < kNormPieces * kWaves; ++q) sum += sums[q];
    const float inv = rsqrtf(sum / static_cast<float>(K) + n.eps);
#pragma unroll
    for (int p = 0; p < kNormPieces; ++p) {
      const int i = place(K, p);
      if (i >= K) break;
      u32x4_t o;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t v = f32x2_to_bf16_rne(low(x[p][j]) * inv, high(x[p][j]) * inv);
        o[j] = f32x2_to_bf16_rne(low(v) * low(w[p][j]), high(v) * high(w[p][j]));
      }
      *reinterpret_cast<u32x4_t *>(lds + kNormSums + static_cast<uint32_t>(i) * 2) = o;
    }
    lds_barrier();
  }
};

// whether an epilogue asks for something by its rows, too: load_rows(args, first row, M, column, N)
template <typename Epi, typename = void>
struct WantsRows : std::false_type {};
template <typename Epi>
struct WantsRows<Epi, std::void_t<decltype(&Epi::load_rows)>> : std::true_type {};

// Epi: struct with kGate (two matrices, T / 2 tiles of each), kHalves (acc and acc2 are the sums over the two halves of K), Args, and per
// unit a state: load(args, n, N) issues what it needs early, finish(args, acc, acc2, m0, M, n, N) stores rows m0 .. m0 + 3 of column n.
// XR: rows of x in a tile that can be present (8: M <= 8, one load per unit of x instead of two).
// Norm: NoNorm, or RowNorm, which takes the place of a.x; the normalised row stands behind the rings, and units are weights only.
template <typename W, int MT, int XR, int T, typename Epi, typename Norm>
__global__ __launch_bounds__(64 * kWaves) void stream_mm_kernel(const Args a, const typename Epi::Args ea, const Norm norm) {
  constexpr bool kNorm = std::is_same<Norm, RowNorm>::value;
  static_assert(!kNorm || (MT == 1 && W::kXUnits == 2), "a row in front of 8-bit weights");
  static_assert(T * MT <= kMaxUnits && (!Epi::kGate || T % 2 == 0), "shape");
  constexpr int TC = Epi::kGate ? T / 2 : T;
  constexpr int XN = kNorm ? 0 : MT * W::kXUnits, U = XN + T;  // units of a step: activations first
  constexpr int kAhead = (kRing + U - 1) / U;             // steps that the ring's units reach into, at most
  constexpr int kLate = kAhead * U - kRing;               // units of the last kAhead steps that are issued while those run
  constexpr int kUnits = TC * MT, kPerWave = (kUnits + kWaves - 1) / kWaves;
  constexpr int kRingBytes = kWaves * kRing * kUnitBytes, kRedBytes = kWaves * T * MT * 1024;
  constexpr int kLoopBytes = kRingBytes > kRedBytes ? kRingBytes : kRedBytes;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[kLoopBytes + (kNorm ? kNormBytes : 0)];

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, b = lane >> 4;
  const int n0 = blockIdx.x * (16 * TC);
  const uint32_t row_bytes = static_cast<uint32_t>(a.K) * W::kBytes, x_row_bytes = static_cast<uint32_t>(a.K) * 2u;
  const int all_steps = static_cast<int>((row_bytes + 127) / 128), slice = blockIdx.y, slices = gridDim.y;
  const int slice0 = all_steps * slice / slices, steps = all_steps * (slice + 1) / slices - slice0;
  const int s0 = slice0 + steps * wave / kWaves, nloc = slice0 + steps * (wave + 1) / kWaves - s0;
  const int turn = nloc * wave / kWaves;  // the step a wave begins with; from its last step it goes on with its first

  const int rows = a.N - n0 < 16 * TC ? a.N - n0 : 16 * TC;
  const __amdgpu_buffer_rsrc_t w_rsrc = make_rsrc(static_cast<const uint8_t *>(a.w) + static_cast<size_t>(n0) * row_bytes, rows * row_bytes);
  const __amdgpu_buffer_rsrc_t w2_rsrc =
      make_rsrc(static_cast<const uint8_t *>(Epi::kGate ? a.w2 : a.w) + static_cast<size_t>(n0) * row_bytes, rows * row_bytes);
  const __amdgpu_buffer_rsrc_t x_rsrc = make_rsrc(a.x, static_cast<uint32_t>(a.M) * x_row_bytes);

  // this lane's part of a unit: row lane / 8 (and 8 rows further down in the unit's second load) and one piece of 16 bytes
  const int r8 = lane >> 3;
  const uint32_t piece0 = ((lane & 7) ^ (r8 >> 1)) * 16, piece1 = ((lane & 7) ^ (4 + (r8 >> 1))) * 16;
  uint8_t *const ring = lds + wave * (kRing * kUnitBytes);
  // unit u (static) of step s into the ring at byte `at`
  constexpr int kXLoads = XR / 8;
  // loads of the units behind unit u that may still be out when it is used
  constexpr auto behind = [](int u) {
    int n = 0;
    for (int i = 1; i < kRing; ++i) n += (u + i) % U < XN ? kXLoads : 2;
    return n;
  };
  const auto issue = [&](int u, int s, uint32_t at) {
    const bool is_x = u < XN;
    const int t = is_x ? u / W::kXUnits : u - XN, tile = is_x ? t : t % TC;
    const uint32_t pitch = is_x ? x_row_bytes : row_bytes;
    const int turned = s + turn, step = s0 + (turned < nloc ? turned : turned - nloc);
    const uint32_t at_k = static_cast<uint32_t>(step) * 128u * (is_x ? W::kXUnits : 1) + (is_x ? 128u * (u % W::kXUnits) : 0u);
    const uint32_t left = pitch - at_k;  // bytes of a row from here on; at least 16, and 128 but in the last step
    const uint32_t o0 = (16u * tile + r8) * pitch + piece0, o1 = (16u * tile + 8u + r8) * pitch + piece1;
    const __amdgpu_buffer_rsrc_t rs = is_x ? x_rsrc : (t < TC ? w_rsrc : w2_rsrc);
    // (at_k >= pitch: the second unit of activations of a last step of 64 bytes of weights or less)
    bool in0 = at_k < pitch && piece0 < left, in1 = at_k < pitch && piece1 < left;
    if (kNorm) in0 &= s < nloc, in1 &= s < nloc;  // (issued without a branch at the start, so that the waits for the row can count them)
    if (is_x) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void *)(ring + at), 16, in0 ? o0 : 0x80000000u, at_k, 0, 0);
      if (kXLoads == 2) __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void *)(ring + at + 1024), 16, in1 ? o1 : 0x80000000u, at_k, 0, 0);
    } else {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void *)(ring + at), 16, in0 ? o0 : 0x80000000u, at_k, 0, 2);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void *)(ring + at + 1024), 16, in1 ? o1 : 0x80000000u, at_k, 0, 2);
    }
  };

  f32x4_t acc[T][MT];
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[t][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  bf16x8_t xf[MT][2 * W::kXUnits];
  const uint32_t row_at = c * 128u, swz = (c >> 1) & 7;
  // unit u, which has landed at byte `at` of the ring: 16-bit weights take operand o from pieces 4 o + b, 8-bit ones two operands from each
  // piece 4 h + b of 16 weights, and x follows
  const auto use = [&](int u, uint32_t at) {
    const uint8_t *p = ring + at + row_at;
    if (u < XN) {
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const uint32_t piece = W::kXUnits == 1 ? 4u * e + b : 2u * b + e;
        xf[u / W::kXUnits][2 * (u % W::kXUnits) + e] = *reinterpret_cast<const bf16x8_t *>(p + ((piece ^ swz) * 16));
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read before the unit's place is given away (weights: used up by then)
    } else {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const u32x4_t w = *reinterpret_cast<const u32x4_t *>(p + (((4u * h + b) ^ swz) * 16));
#pragma unroll
        for (int o = 0; o < W::kXUnits; ++o) {
          const bf16x8_t wf = W::operand(w, o);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
            acc[u - XN][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[mt][W::kXUnits * h + o], wf, acc[u - XN][mt], 0, 0, 0);
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  const auto next = [](uint32_t at) { return at == (kRing - 1) * kUnitBytes ? 0u : at + kUnitBytes; };

  [[maybe_unused]] NormLoads row_in;
  if constexpr (kNorm) row_in.request(norm, a.K);
#pragma unroll
  for (int q = 0; q < kRing; ++q)
    if (kNorm || q / U < nloc) issue(q % U, q / U, q * kUnitBytes);
  if constexpr (kNorm) {
    __builtin_amdgcn_sched_barrier(0);
    row_in.finish(norm, a.K, lds + kLoopBytes, blockIdx.x == 0 && blockIdx.y == 0);
  }
  // the activations of step s, where they stand behind the rings
  const auto take_x = [&](int s) {
    if constexpr (kNorm) {
      const int turned = s + turn, step = s0 + (turned < nloc ? turned : turned - nloc);
      const uint32_t row = kLoopBytes + kNormSums, at_k = static_cast<uint32_t>(step) * 256u;
#pragma unroll
      for (int i = 0; i < 4; ++i)  // every lane column holds it; what the others give is not stored
        xf[0][i] = *reinterpret_cast<const bf16x8_t *>(lds + row + at_k + 128u * (i >> 1) + (2u * b + (i & 1)) * 16u);
    }
  };
  Epi epi[kPerWave];
#pragma unroll
  for (int i = 0; i < kPerWave; ++i) {
    const int u = wave + kWaves * i;
    if (u < kUnits) epi[i].load(ea, n0 + 16 * (u / MT) + c, a.N);
    if constexpr (WantsRows<Epi>::value) {
      if (u < kUnits) epi[i].load_rows(ea, 16 * (u % MT) + 4 * b, a.M, n0 + 16 * (u / MT) + c, a.N);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  uint32_t at = 0;
  int s = 0;
#pragma unroll 1
  for (; s < nloc - kAhead; ++s) {
    take_x(s);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      wait_loads(behind(u));  // (loads of the epilogue only make it wait longer)
      use(u, at);
      issue((u + kRing) % U, s + (u + kRing) / U, at);
      at = next(at);
    }
  }
  // the last steps: what is left to issue, then nothing more is on its way than what they need
  if (s < nloc && nloc >= kAhead) {
    take_x(s);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (u < kLate) wait_loads(behind(u));
      if (u == kLate) wait_loads(0);
      use(u, at);
      if (u < kLate) issue((u + kRing) % U, s + (u + kRing) / U, at);
      at = next(at);
    }
    ++s;
  } else {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
#pragma unroll 1
  for (; s < nloc; ++s) {
    take_x(s);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      use(u, at);
      at = next(at);
    }
  }

  lds_barrier();  // the rings become the meeting place
  f32x4_t *const red = reinterpret_cast<f32x4_t *>(lds);
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) red[(wave * (T * MT) + t * MT + mt) * 64 + lane] = acc[t][mt];
  lds_barrier();
#pragma unroll
  for (int i = 0; i < kPerWave; ++i) {
    const int u = wave + kWaves * i;
    if (u >= kUnits) break;
    // the lower half of K, the upper half, and their sum
    const auto half = [&](int unit, int k0) {
      f32x4_t sum = red[(k0 * (T * MT) + unit) * 64 + lane];
#pragma unroll
      for (int k = 1; k < kWaves / 2; ++k) sum += red[((k0 + k) * (T * MT) + unit) * 64 + lane];
      return sum;
    };
    const f32x4_t lo = half(u, 0), hi = half(u, kWaves / 2);
    const int m0 = 16 * (u % MT) + 4 * b, n = n0 + 16 * (u / MT) + c;
    if constexpr (Epi::kGate) epi[i].finish(ea, lo + hi, half(u + kUnits, 0) + half(u + kUnits, kWaves / 2), m0, a.M, n, a.N);
    else if constexpr (Epi::kHalves) epi[i].finish(ea, lo, hi, m0, a.M, n, a.N);
    else epi[i].finish(ea, lo + hi, lo, m0, a.M, n, a.N);
  }
}

// weight tiles per workgroup: the rounds of workgroups over the CUs, each a workgroup's weights plus the activations it reads from its L2
// (a quarter of a weight byte's cost) plus a fixed part
template <typename W, bool GATE>
inline int pick_tiles(int M, int N, int K, int slices = 1) {
  const int mt = (M + 15) / 16, cap = kMaxUnits / (mt <= 1 ? 1 : mt <= 2 ? 2 : 4);
  const int tiles = (N + 15) / 16;
  int best = 0;
  double best_cost = 0;
  for (int t : {1, 2, 3, 4, 6, 8}) {
    if (t > cap || (GATE && t % 2)) continue;
    const int tc = GATE ? t / 2 : t;
    if (int64_t{16} * tc * K * W::kBytes >= kMaxBytes) continue;
    const int rounds = ((tiles + tc - 1) / tc * slices + 255) / 256;
    const double cost = rounds * (16.0 * t * W::kBytes + 0.25 * 2 * M + 16384.0 / K);
    if (!best || cost < best_cost) best = t, best_cost = cost;
  }
  return best;
}

template <typename W, typename Epi, int MT, int XR, int T, typename Norm>
int launch(const Args &a, const typename Epi::Args &ea, int slices, hipStream_t stream, const Norm &norm) {
  if constexpr (T * MT > kMaxUnits || (Epi::kGate && T % 2)) {
    return E2H_ERR_BAD_SHAPE;
  } else {
    constexpr int TC = Epi::kGate ? T / 2 : T;
    const int tiles = (a.N + 15) / 16;
    hipLaunchKernelGGL((stream_mm_kernel<W, MT, XR, T, Epi, Norm>), dim3((tiles + TC - 1) / TC, slices), dim3(64 * kWaves), 0, stream, a, ea, norm);
    return launch_status();
  }
}

template <typename W, typename Epi, int MT, int XR, typename Norm = NoNorm>
int launch_rows(const Args &a, const typename Epi::Args &ea, int t, int slices, hipStream_t stream, const Norm &norm = Norm{}) {
  switch (t) {
    case 1: return launch<W, Epi, MT, XR, 1>(a, ea, slices, stream, norm);
    case 2: return launch<W, Epi, MT, XR, 2>(a, ea, slices, stream, norm);
    case 3: return launch<W, Epi, MT, XR, 3>(a, ea, slices, stream, norm);
    case 4: return launch<W, Epi, MT, XR, 4>(a, ea, slices, stream, norm);
    case 6: return launch<W, Epi, MT, XR, 6>(a, ea, slices, stream, norm);
    case 8: return launch<W, Epi, MT, XR, 8>(a, ea, slices, stream, norm);
    default: return E2H_ERR_BAD_SHAPE;
  }
}

// rows in pieces of 16 bytes, whole row tiles of x and a tile of weights below 2^31 bytes; x and w 16-byte aligned
inline bool takes(int64_t M, int64_t N, int64_t K, int bytes) {
  const int64_t x_rows = M <= 16 ? 16 : M <= 32 ? 32 : 64;
  return M >= 1 && M <= 64 && N >= 1 && N < (int64_t{1} << 31) - 128 && K >= 1 && K < (int64_t{1} << 30) && K * bytes % 16 == 0 &&
         x_rows * K * 2 < kMaxBytes && 16 * K * bytes < kMaxBytes;
}

// slices > 1: workgroups split K too, and the epilogue stores its slice's sums (blockIdx.y)
template <typename W, typename Epi>
int run(const Args &a, const typename Epi::Args &ea, hipStream_t stream, int slices = 1) {
  const int t = pick_tiles<W, Epi::kGate>(a.M, a.N, a.K, slices);
  if (a.M <= 8) return launch_rows<W, Epi, 1, 8>(a, ea, t, slices, stream);
  if (a.M <= 16) return launch_rows<W, Epi, 1, 16>(a, ea, t, slices, stream);
  if (a.M <= 32) return launch_rows<W, Epi, 2, 16>(a, ea, t, slices, stream);
  return launch_rows<W, Epi, 4, 16>(a, ea, t, slices, stream);
}

// the same over a row that a norm forms first (norm_fits)
template <typename W, typename Epi>
int run_norm(const Args &a, const typename Epi::Args &ea, const RowNorm &norm, hipStream_t stream) {
  return launch_rows<W, Epi, 1, 8>(a, ea, pick_tiles<W, Epi::kGate>(a.M, a.N, a.K), 1, stream, norm);
}

}  // namespace stream
}  // namespace e2h
