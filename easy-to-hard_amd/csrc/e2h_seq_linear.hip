// bfloat16 linears of decode batches (e2h_seq_linear): up to 64 rows over weights that are read once, e2h_stream.h.
//
// Measured on one MI355X, graph replay over rotating weights (vendor matmul in brackets): 22528 x 4096 at 1 / 32 rows 31.7 / 33.3 us
// (50.4 / 45.2), 16384 x 4096 24.7 / 25.1 (33.5 / 33.4), 4096 x 16384 29.2 / 30 (31.0 / 35.3), 4096 x 8192 12.9 / 18.6 (16.3 /
// 19.1), 4096 x 4096 7.7 / 11.6 (15.3 / 13.8), 32000 x 4096 44.4 / 45.8 (59.7 / 55.1): 4.2 to 6 TB/s of weights.
#include "e2h_gemm256.h"
#include "e2h_seq_common.h"
#include "e2h_stream.h"

namespace e2h {
namespace {

enum Act { kNone = 0, kSquare = 1, kCap = 2 };
constexpr int kSlices = 4;

// act(bf16(acc)), rounded: the linear's own output is rounded first, as when the activation is a launch of its own
template <int ACT>
__device__ __forceinline__ bf16_t activated(float acc, float cap) {
  const bf16_t y = from_f32<bf16_t>(acc);
  if (ACT == kSquare) {
    const float p = fmaxf(to_f32(y), 0.f);
    return from_f32<bf16_t>(p * p);
  }
  return ACT == kCap ? from_f32<bf16_t>(cap * tanhf(to_f32(y) / cap)) : y;
}

template <int ACT>
struct Linear {
  static constexpr bool kGate = false, kHalves = false;
  struct Args {
    bf16_t *y;
    float cap;
  };
  __device__ __forceinline__ void load(const Args &, int, int) {}
  __device__ __forceinline__ void finish(const Args &a, f32x4_t acc, f32x4_t, int m0, int M, int n, int N) const {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (n < N && m0 + r < M) a.y[static_cast<size_t>(m0 + r) * N + n] = activated<ACT>(acc[r], a.cap);
  }
};

// gelu(bf16(acc)) * table[tokens[row], column + n], as e2h_seq_gelu_gate_rows forms it from the linear's output.  In a step of two layers at 32 rows the two launches of that cost
// 2.7 us; with the rows asked for in `finish`, tokens first, half of it was lost again.
struct GeluGate {
  static constexpr bool kGate = false, kHalves = false;
  struct Args {
    bf16_t *y;
    const bf16_t *table;
    const int64_t *tokens;
    int64_t ld, column, table_rows;
  };
  bf16_t row[4];  // of the table: on their way under the product
  bool there[4];
  __device__ __forceinline__ void load(const Args &, int, int) {}
  __device__ __forceinline__ void load_rows(const Args &a, int m0, int M, int n, int N) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t token = a.tokens[m0 + r < M ? m0 + r : M - 1];
      there[r] = token >= 0 && token < a.table_rows && n < N;
      row[r] = a.table[there[r] ? token * a.ld + a.column + n : a.column];
    }
  }
  __device__ __forceinline__ void finish(const Args &a, f32x4_t acc, f32x4_t, int m0, int M, int n, int N) const {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (n < N && m0 + r < M) a.y[static_cast<size_t>(m0 + r) * N + n] = from_f32<bf16_t>(gelu_tanh_f32(to_f32(from_f32<bf16_t>(acc[r]))) * (there[r] ? to_f32(row[r]) : 0.f));
  }
};

// float32 sums of a K slice, [slices][M][N]
struct Slice {
  static constexpr bool kGate = false, kHalves = false;
  struct Args {
    float *out;
  };
  __device__ __forceinline__ void load(const Args &, int, int) {}
  __device__ __forceinline__ void finish(const Args &a, f32x4_t acc, f32x4_t, int m0, int M, int n, int N) const {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (n < N && m0 + r < M) a.out[(static_cast<size_t>(blockIdx.y) * M + m0 + r) * N + n] = acc[r];
  }
};

template <int ACT>
__global__ __launch_bounds__(256) void add_slices_kernel(const float *s, bf16_t *y, int n, float cap) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  float v[kSlices];
#pragma unroll
  for (int k = 0; k < kSlices; ++k) v[k] = s[static_cast<size_t>(k) * n + i];
#pragma unroll
  for (int k = 1; k < kSlices; ++k) v[0] += v[k];
  y[i] = activated<ACT>(v[0], cap);
}

// Narrow matrices with many rows: one tile of 16 weight rows per CU reads all of x beside it, twice its weights at 32 rows.  K over four
// workgroups instead, each with four times the tiles, and a launch that adds them (32 rows, both launches; one launch; vendor matmul):
// 4096 x 16384 30 us, 39.5, 35.3; 4096 x 8192 18.6, 19.9, 19.1; 2048 x 8192 12, 16.  At 4096 x 4096 the second launch costs what the
// first gains (11.6 in one launch, 13.8 vendor), and up to 16 rows x is the smaller part.
bool sliced(int64_t rows, int64_t n, int64_t k) { return rows > 16 && n <= 16 * 256 && k >= 8192; }

template <int ACT>
int run_linear(const stream::Args &a, bf16_t *y, float cap, float *scratch, hipStream_t s) {
  if (!sliced(a.M, a.N, a.K)) return stream::run<stream::Bf16Weights, Linear<ACT>>(a, {y, cap}, s);
  if (int rc = stream::run<stream::Bf16Weights, Slice>(a, {scratch}, s, kSlices)) return rc;
  const int n = a.M * a.N;
  hipLaunchKernelGGL(add_slices_kernel<ACT>, dim3((n + 255) / 256), dim3(256), 0, s, scratch, y, n, cap);
  return launch_status();
}

// ---- many rows: the activation behind a tile of products (e2h_gemm256.h) ---------------------------------------------------------------
// cap tanh(y / cap): with z = y y it is y (1 + z Q(z)) up to |y| = 0.75 cap, Q by the Remez algorithm (3.3e-8 of tanh, half a unit in the last place of float32) in powers of 1 / cap^2, else
// cap (1 - 2 / (1 + exp(2 y / cap))); what either could round otherwise to bfloat16 than e2h_seq_softcap does is formed as there (gemm256::settled).  A tile's store forms the first for all of
// its values, and the second too where a wave's 512 values have one that needs it: ten instructions a value with the look at its rounding, where tanhf and the division take 45, which would
// take as long as the pass over memory that is saved (128 values per lane and wave with nothing beside them).
struct Cap {
  float cap, limit, q[5], twice;  // limit: 0.75 cap; twice: 2 / cap in units of log 2
};
Cap cap_of(float cap) {
  const double u = 1.0 / (static_cast<double>(cap) * cap);
  const double q[5] = {-0.3333306838118954, 0.1332652117591573, -0.05339025879171665, 0.01966491390244702, -0.004769490464846426};
  Cap c = {cap, 0.75f * cap, {}, static_cast<float>(2 * 1.4426950408889634 / cap)};
  double power = u;
  for (int j = 0; j < 5; ++j, power *= u) c.q[j] = static_cast<float>(q[j] * power);
  return c;
}
// where cap^-10 and the squares of what lies below cap are far from the ends of float32
bool cap_fits(float cap) { return cap >= 0x1p-6f && cap <= 0x1p10f; }

template <int ACT>
struct RowsWalk : gemm256::PlainWalk<> {
  Cap c;
  __device__ __forceinline__ RowsWalk(const uint16_t *x_, const uint16_t *w_, uint16_t *y_, const Cap &c_, int M_, int N_, int K_) : PlainWalk(x_, w_, y_, M_, N_, K_), c(c_) {}
  struct Dest {};
  __device__ __forceinline__ void dest(const Tile &, int, int, Dest &) const {}
  __device__ __forceinline__ float capped(float y) const {
    const float z = y * y;
    float q = c.q[4];
#pragma unroll
    for (int j = 3; j >= 0; --j) q = __builtin_fmaf(q, z, c.q[j]);
    return y * __builtin_fmaf(z, q, 1.0f);  // (-0 stays that)
  }
  __device__ __forceinline__ float capped_far(float y, float near) const {
    const float far = c.cap * __builtin_fmaf(-2.0f, __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(y * c.twice)), 1.0f);
    return __builtin_fabsf(y) > c.limit ? far : near;  // (what is no number stays none)
  }
  __device__ __forceinline__ void store(const Tile &tile, const Dest &, int, int, int row, int col, float (&v)[8]) const {
    const auto low = [](uint32_t b) { return __builtin_bit_cast(float, b << 16); };
    const auto high = [](uint32_t b) { return __builtin_bit_cast(float, b & 0xFFFF0000u); };
    u32x4_t out;
#pragma unroll
    for (int e = 0; e < 4; ++e) out[e] = pack_bf16(v[2 * e], v[2 * e + 1]);  // the linear's own output is rounded first
    if (ACT == kSquare) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float lo = fmaxf(low(out[e]), 0.f), hi = fmaxf(high(out[e]), 0.f);
        out[e] = pack_bf16(lo * lo, hi * hi);
      }
    }
    if (ACT == kCap) {
      gemm256::f32x8_t near;
      float y[8], top = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        y[e] = e & 1 ? high(out[e >> 1]) : low(out[e >> 1]);
        near[e] = capped(y[e]);
        top = __builtin_fmaxf(top, __builtin_fabsf(y[e]));
      }
      if (__builtin_amdgcn_ballot_w64(top > c.limit)) {
#pragma unroll
        for (int e = 0; e < 8; ++e) near[e] = capped_far(y[e], near[e]);
      }
      const float cap = c.cap;
      near = gemm256::settled(near, out, [cap](float z) { return cap * tanhf(z / cap); });
#pragma unroll
      for (int e = 0; e < 4; ++e) out[e] = pack_bf16(near[2 * e], near[2 * e + 1]);
    }
    __builtin_amdgcn_raw_buffer_store_b128(out, y_rsrc(tile), y_at(tile, row, col), 0, 0);
  }
};

template <int ACT>
__global__ __launch_bounds__(256, 1) void linear_rows_kernel(const uint16_t *x, const uint16_t *w, uint16_t *y, const Cap cap, int M, int N, int K) {
#if defined(__HIP_DEVICE_COMPILE__)
  __shared__ __attribute__((aligned(1024))) uint8_t lds[gemm256::kRing];
  RowsWalk<ACT> tiles(x, w, y, cap, M, N, K);
  gemm256::walk<false>(tiles, lds);
#endif
}

bool rows_fit(int64_t m, int64_t n, int64_t k) {
  return m >= 1 && n >= 8 && n % 8 == 0 && k % 64 == 0 && k >= gemm256::kLeastK && m <= INT32_MAX / 2 && n <= INT32_MAX / 2 && k <= INT32_MAX / 2 &&
         m * k * 2 < (int64_t{1} << 32) && n * k * 2 < (int64_t{1} << 32) && 256 * n * 2 < (int64_t{1} << 32);
}

}  // namespace
}  // namespace e2h

using namespace e2h;

// 1 where the product with its activation is expected to be faster here than the library's product and a pass over its result.  Measured, us, that / here: 16384 x 4096 1000 rows 114 / 96,
// 8192 rows 817 / 743; 8192 x 2048 2048 rows 68 / 51; 2048 x 4096 8192 rows 112 / 95; 16384 x 4096 512 rows 70 / 76: not taken.  Without an activation the library's product is
// 2 % the faster one where it fills the chip (16384 x 4096 8192 rows 725 / 742).  With a soft cap 32000 x 4096 8192 rows 1425 + 229 / 1504.
// us, as for the quantized linears on the same loop (a last round that is not full runs at a higher clock), against the library's product at what it reaches where it fills the chip, 1.5
// PFLOP/s, and a pass over the result of its own.
extern "C" int e2h_seq_linear_rows_pays(int64_t rows, int64_t n, int64_t k, int act, float cap) {
  if (rows <= 64 || (act != kSquare && (act != kCap || !cap_fits(cap))) || !rows_fit(rows, n, k)) return 0;
  const int64_t tiles = (rows + 255) / 256 * ((n + 255) / 256), full = tiles / 256, rest = tiles % 256;
  const double rounds = static_cast<double>(full) + (rest == 0 ? 0. : full == 0 ? 1. : 0.6 + 0.4 * static_cast<double>(rest) / 256);
  const double outputs = static_cast<double>(rows) * static_cast<double>(n);
  return 4 + rounds * (static_cast<double>(k) / 64 * 1.36 + (act == kCap ? 9 : 5)) < outputs * static_cast<double>(k) * 2 / 1.5e9 + outputs * 4 / 6e6 + 12 ? 1 : 0;
}

extern "C" int e2h_seq_linear_rows(const void *x, const void *w, void *y, int64_t rows, int64_t n, int64_t k, int act, float cap, void *stream) {
  if (!x || !w || !y) return E2H_ERR_NULL_POINTER;
  if (!rows_fit(rows, n, k) || act < kNone || act > kCap || (act == kCap && !cap_fits(cap))) return E2H_ERR_BAD_SHAPE;
  if (!aligned16(x) || !aligned16(w) || !aligned16(y)) return E2H_ERR_MISALIGNED;
  const dim3 grid(gemm256::grid_of((rows + 255) / 256 * ((n + 255) / 256)));
  const auto *xs = static_cast<const uint16_t *>(x), *ws = static_cast<const uint16_t *>(w);
  auto *ys = static_cast<uint16_t *>(y);
  const int M = static_cast<int>(rows), N = static_cast<int>(n), K = static_cast<int>(k);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const Cap c = act == kCap ? cap_of(cap) : Cap{};
  if (act == kSquare) hipLaunchKernelGGL(linear_rows_kernel<kSquare>, grid, dim3(256), 0, s, xs, ws, ys, c, M, N, K);
  else if (act == kCap) hipLaunchKernelGGL(linear_rows_kernel<kCap>, grid, dim3(256), 0, s, xs, ws, ys, c, M, N, K);
  else hipLaunchKernelGGL(linear_rows_kernel<kNone>, grid, dim3(256), 0, s, xs, ws, ys, c, M, N, K);
  return launch_status();
}

extern "C" int64_t e2h_seq_linear_scratch_bytes(int64_t rows, int64_t n, int64_t k) {
  if (!stream::takes(rows, n, k, 2)) return E2H_ERR_BAD_SHAPE;
  return sliced(rows, n, k) ? kSlices * rows * n * 4 : 0;
}

extern "C" int e2h_seq_linear(const void *x, const void *w, void *y, int64_t rows, int64_t n, int64_t k, int act, float cap, void *scratch,
                              int64_t scratch_bytes, void *stream) {
  if (!x || !w || !y) return E2H_ERR_NULL_POINTER;
  if (!stream::takes(rows, n, k, 2) || act < kNone || act > kCap || (act == kCap && !(cap > 0.f))) return E2H_ERR_BAD_SHAPE;
  if (sliced(rows, n, k) && (!scratch || scratch_bytes < kSlices * rows * n * 4)) return E2H_ERR_SCRATCH_TOO_SMALL;
  if (!aligned16(x) || !aligned16(w) || (reinterpret_cast<uintptr_t>(y) & 1u) || (reinterpret_cast<uintptr_t>(scratch) & 3u)) return E2H_ERR_MISALIGNED;
  const stream::Args a{static_cast<const uint16_t *>(x), w, w, static_cast<int>(rows), static_cast<int>(n), static_cast<int>(k)};
  hipStream_t s = static_cast<hipStream_t>(stream);
  bf16_t *out = static_cast<bf16_t *>(y);
  float *f = static_cast<float *>(scratch);
  if (act == kSquare) return run_linear<kSquare>(a, out, 0.f, f, s);
  if (act == kCap) return run_linear<kCap>(a, out, cap, f, s);
  return run_linear<kNone>(a, out, 0.f, f, s);
}

extern "C" int e2h_seq_linear_gelu_gate(const void *x, const void *w, const void *table, const int64_t *tokens, void *y, int64_t rows, int64_t n, int64_t k, int64_t ld, int64_t column,
                                        int64_t table_rows, void *stream) {
  if (!x || !w || !table || !tokens || !y) return E2H_ERR_NULL_POINTER;
  if (!stream::takes(rows, n, k, 2) || sliced(rows, n, k) || column < 0 || column + n > ld || table_rows < 1) return E2H_ERR_BAD_SHAPE;
  if (!aligned16(x) || !aligned16(w) || (reinterpret_cast<uintptr_t>(y) & 1u) || (reinterpret_cast<uintptr_t>(table) & 1u) || (reinterpret_cast<uintptr_t>(tokens) & 7u)) return E2H_ERR_MISALIGNED;
  const stream::Args a{static_cast<const uint16_t *>(x), w, w, static_cast<int>(rows), static_cast<int>(n), static_cast<int>(k)};
  return stream::run<stream::Bf16Weights, GeluGate>(a, {static_cast<bf16_t *>(y), static_cast<const bf16_t *>(table), tokens, ld, column, table_rows}, static_cast<hipStream_t>(stream));
}

extern "C" int e2h_seq_linear_sums(const void *x, const void *w, float *sums, int64_t rows, int64_t n, int64_t k, void *stream) {
  if (!x || !w || !sums) return E2H_ERR_NULL_POINTER;
  if (!stream::takes(rows, n, k, 2) || !sliced(rows, n, k)) return E2H_ERR_BAD_SHAPE;
  if (!aligned16(x) || !aligned16(w) || !aligned16(sums)) return E2H_ERR_MISALIGNED;
  const stream::Args a{static_cast<const uint16_t *>(x), w, w, static_cast<int>(rows), static_cast<int>(n), static_cast<int>(k)};
  return stream::run<stream::Bf16Weights, Slice>(a, {sums}, static_cast<hipStream_t>(stream), kSlices);
}
