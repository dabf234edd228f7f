// Quantized linears over thousands of rows: the weights are unpacked to 16-bit values in scratch memory once per call, then multiplied
// by the loop of e2h_gemm256.h.
//
// int8: y = bf16( bf16( x @ q^T ) * scales ).  A code has at most eight significant bits, so its bfloat16 value is exact and the result is that
// of the kernels which convert on the way into the matrix cores (e2h_int8_gemm.hip).  Those are bound by the energy and the LDS traffic of 64-byte rows and
// by conversions beside the products.
#include <algorithm>

#include "e2h_common.h"
#include "e2h_gemm256.h"
#include "e2h_unpacked_gemm.h"

namespace e2h {
namespace {

__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, bf16x2));
}

// 16 codes per thread.  Bound by memory: 12288 x 4096 (151 MB moved) 31 us.
__global__ __launch_bounds__(256) void unpack_int8_kernel(const int8_t *__restrict__ q, uint16_t *__restrict__ w, int64_t pieces) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= pieces) return;
  const u32x4_t c = reinterpret_cast<const u32x4_t *>(q)[i];
  u32x4_t out[2];
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const uint32_t t = c[d];
    const float f0 = static_cast<float>(static_cast<int8_t>(t & 0xFFu)), f1 = static_cast<float>(static_cast<int8_t>((t >> 8) & 0xFFu));
    const float f2 = static_cast<float>(static_cast<int8_t>((t >> 16) & 0xFFu)), f3 = static_cast<float>(static_cast<int8_t>(t >> 24));
    out[d >> 1][2 * (d & 1)] = pack_bf16(f0, f1);
    out[d >> 1][2 * (d & 1) + 1] = pack_bf16(f2, f3);
  }
  reinterpret_cast<u32x4_t *>(w)[2 * i] = out[0];
  reinterpret_cast<u32x4_t *>(w)[2 * i + 1] = out[1];
}

// The tiles of one plain product, dealt to the XCDs in contiguous runs of equal length: panels of eight column blocks, all row
// blocks of a panel after each other, so that the 32 tiles at work on an XCD share four row blocks and eight column blocks.
struct PlainWalk {
  static constexpr int kPanel = 8;
  struct Tile {
    int rb, cb;
  };
  const uint16_t *x, *w;
  uint16_t *y;
  int M, N, K, t, end, stride;

  __device__ __forceinline__ PlainWalk(const uint16_t *x_, const uint16_t *w_, uint16_t *y_, int M_, int N_, int K_) : x(x_), w(w_), y(y_), M(M_), N(N_), K(K_) {
    const int64_t total = static_cast<int64_t>((M + 255) / 256) * ((N + 255) / 256);
    const int xcd = blockIdx.x & 7;
    stride = static_cast<int>(gridDim.x >> 3);
    end = static_cast<int>(total * (xcd + 1) / 8);
    t = static_cast<int>(total * xcd / 8) + static_cast<int>(blockIdx.x >> 3) - stride;
  }
  __device__ __forceinline__ bool next(Tile &tile) {
    t += stride;
    if (t >= end) return false;
    const int R = (M + 255) / 256, C = (N + 255) / 256, panel = t / (kPanel * R), at = t - panel * kPanel * R;
    const int wide = C - panel * kPanel < kPanel ? C - panel * kPanel : kPanel;
    tile.rb = at / wide;
    tile.cb = panel * kPanel + at - tile.rb * wide;
    return true;
  }
  __device__ __forceinline__ bool first(Tile &tile) { return next(tile); }
  __device__ __forceinline__ int chunks() const { return K / 64; }
  __device__ __forceinline__ __amdgpu_buffer_rsrc_t x_rsrc(const Tile &) const { return make_rsrc(x, static_cast<uint32_t>(static_cast<size_t>(M) * K * 2)); }
  __device__ __forceinline__ __amdgpu_buffer_rsrc_t w_rsrc(const Tile &) const { return make_rsrc(w, static_cast<uint32_t>(static_cast<size_t>(N) * K * 2)); }
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
  __device__ __forceinline__ uint32_t w_at(const Tile &tile, int col) const {
    const int n = tile.cb * 256 + col;
    return static_cast<uint32_t>(n < N ? n : N - 1) * static_cast<uint32_t>(K) * 2;
  }
  __device__ __forceinline__ uint32_t y_at(const Tile &tile, int row, int col) const {
    const int n = tile.cb * 256 + col;
    return n < N ? (static_cast<uint32_t>(row) * static_cast<uint32_t>(N) + static_cast<uint32_t>(n)) * 2 : gemm256::kNowhere;
  }
};

struct Int8Walk : PlainWalk {
  const uint16_t *scales;
  __device__ __forceinline__ Int8Walk(const uint16_t *x_, const uint16_t *w_, const uint16_t *scales_, uint16_t *y_, int M_, int N_, int K_)
      : PlainWalk(x_, w_, y_, M_, N_, K_), scales(scales_) {}
  struct Dest {
    u32x4_t scale[4];  // of the eight columns of each store of a row
  };
  __device__ __forceinline__ void dest(const Tile &tile, int, int col, Dest &d) const {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int n = tile.cb * 256 + col + 32 * q;
      d.scale[q] = *reinterpret_cast<const u32x4_t *>(scales + (n < N ? n : N - 8));
    }
  }
  __device__ __forceinline__ void store(const Tile &tile, const Dest &d, int, int q, int row, int col, float (&v)[8]) const {
    u32x4_t out;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t t = pack_bf16(v[2 * e], v[2 * e + 1]), s = d.scale[q][e];  // the linear's output, then its product with the scale, as in the reference
      out[e] = pack_bf16(__builtin_bit_cast(float, t << 16) * __builtin_bit_cast(float, s << 16),
                         __builtin_bit_cast(float, t & 0xFFFF0000u) * __builtin_bit_cast(float, s & 0xFFFF0000u));
    }
    __builtin_amdgcn_raw_buffer_store_b128(out, y_rsrc(tile), y_at(tile, row, col), 0, 0);
  }
};

__global__ __launch_bounds__(256, 1) void int8_unpacked_gemm_kernel(const uint16_t *x, const uint16_t *w, const uint16_t *scales, uint16_t *y, int M, int N, int K) {
#if defined(__HIP_DEVICE_COMPILE__)
  __shared__ __attribute__((aligned(1024))) uint8_t lds[gemm256::kRing];
  Int8Walk tiles(x, w, scales, y, M, N, K);
  gemm256::walk<false>(tiles, lds);
#endif
}

unsigned grid_of(int64_t M, int64_t N) {
  const int64_t tiles = ((M + 255) / 256) * ((N + 255) / 256);
  return static_cast<unsigned>(8 * std::min<int64_t>(32, (tiles + 7) / 8));
}

}  // namespace

// Microseconds of a product with the unpacked weights, within 10 % of 48 measured shapes of 1024 .. 8192 rows: 1.36 per chunk of 64 k and 5 per round of 256 tiles; a last
// round that is not full runs at a higher clock.
double unpacked_cost(int64_t M, int64_t N, int64_t K, double unpack) {
  const int64_t tiles = ((M + 255) / 256) * ((N + 255) / 256), full = tiles / 256, rest = tiles % 256;
  const double rounds = static_cast<double>(full) + (rest == 0 ? 0. : full == 0 ? 1. : 0.6 + 0.4 * static_cast<double>(rest) / 256);
  return unpack + 4 + rounds * (static_cast<double>(K) / 64 * 1.36 + 5);
}

// The same of int8_gemm32 (e2h_int8_gemm.hip), by its own rule: 256-row tiles dealt to the XCDs by whole column blocks, 1.52 per chunk, or
// rounds of 128-row ones, 1.03 per chunk.
double int8_gemm32_cost(int64_t M, int64_t N, int64_t K) {
  const int64_t cols = (N + 255) / 256, rounds256 = (((M + 255) / 256) * cols + 255) / 256, rounds128 = (((M + 127) / 128) * cols + 255) / 256;
  const double chunks = static_cast<double>(K) / 64;
  if (rounds256 * 20 <= rounds128 * 11) return static_cast<double>(((cols + 7) / 8 * ((M + 255) / 256) + 31) / 32) * (chunks * 1.52 + 5);
  return static_cast<double>(rounds128) * (chunks * 1.03 + 5);
}

// Taken where it is the cheaper one, the unpacking (three bytes a weight at 4.8 TB/s) included: 8192 rows 12288 x 4096 571 us (611 converting in the loop),
// 11008 x 4096 542 (591), 5120 x 13824 875 (1250: 20 column blocks on 8 XCDs); 2048 rows 4096 x 11008 209 (177), left to the other form.
int64_t int8_unpacked_bytes(int64_t M, int64_t N, int64_t K) {
  if (M < 1 || N < 8 || N % 8 != 0 || K % 128 != 0 || K < 256 || N > INT32_MAX || K > INT32_MAX || N * K * 2 >= (int64_t{1} << 32)) return 0;
  const Options &o = options();
  if (o.int4_no_gemm32 || o.int8_force_generic || o.int8_gemm_tile || o.int8_gemm_waves || o.int8_gemm_wave_cols || o.int8_rows_per_wave) return 0;  // another form is asked for
  return unpacked_cost(M, N, K, static_cast<double>(N) * static_cast<double>(K) * 3 / 4.8e6) < int8_gemm32_cost(M, N, K) ? N * K * 2 : 0;
}

int int8_unpacked_gemm(const uint16_t *x, const int8_t *q, const uint16_t *scales, uint16_t *y, int M, int N, int K, uint16_t *w, hipStream_t stream) {
  const int64_t pieces = static_cast<int64_t>(N) * K / 16;
  hipLaunchKernelGGL(unpack_int8_kernel, dim3(static_cast<unsigned>((pieces + 255) / 256)), dim3(256), 0, stream, q, w, pieces);
  // rows in slices that a 32-bit offset reaches
  int64_t most = ((int64_t{1} << 32) - 1) / (2 * static_cast<int64_t>(K));
  most -= most % 256;
  for (int64_t m0 = 0; m0 < M; m0 += most) {
    const int rows = static_cast<int>(M - m0 < most ? M - m0 : most);
    hipLaunchKernelGGL(int8_unpacked_gemm_kernel, dim3(grid_of(rows, N)), dim3(256), 0, stream, x + m0 * K, w, scales, y + m0 * N, rows, N, K);
  }
  return launch_status();
}

}  // namespace e2h

extern "C" int64_t e2h_int8_mm_scratch_bytes(int64_t m, int64_t n, int64_t k) { return e2h::int8_unpacked_bytes(m, n, k); }

extern "C" int e2h_int8_mm_scratch(const uint16_t *x, const int8_t *q, const uint16_t *scales, uint16_t *y, int64_t m, int64_t n, int64_t k, void *scratch,
                                   int64_t scratch_bytes, void *stream) {
  using namespace e2h;
  if (!x || !q || !scales || !y) return E2H_ERR_NULL_POINTER;
  const int64_t need = m > INT32_MAX ? 0 : int8_unpacked_bytes(m, n, k);
  if (!scratch || need == 0 || scratch_bytes < need || !aligned16(x) || !aligned16(q) || !aligned16(scales) || !aligned16(y) || !aligned16(scratch))
    return e2h_int8_mm(x, q, scales, y, m, n, k, nullptr, 0, stream);
  return int8_unpacked_gemm(x, q, scales, y, static_cast<int>(m), static_cast<int>(n), static_cast<int>(k), static_cast<uint16_t *>(scratch),
                            static_cast<hipStream_t>(stream));
}
