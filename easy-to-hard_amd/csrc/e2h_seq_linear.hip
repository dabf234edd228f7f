// bfloat16 linears of decode batches (e2h_seq_linear): up to 64 rows over weights that are read once, e2h_stream.h.
//
// Measured on one MI355X, graph replay over rotating weights (vendor matmul in brackets): 22528 x 4096 at 1 / 32 rows 31.7 / 33.3 us
// (50.4 / 45.2), 16384 x 4096 24.7 / 25.1 (33.5 / 33.4), 4096 x 16384 29.2 / 30 (31.0 / 35.3), 4096 x 8192 12.9 / 18.6 (16.3 /
// 19.1), 4096 x 4096 7.7 / 11.6 (15.3 / 13.8), 32000 x 4096 44.4 / 45.8 (59.7 / 55.1): 4.2 to 6 TB/s of weights.
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

}  // namespace
}  // namespace e2h

using namespace e2h;

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
