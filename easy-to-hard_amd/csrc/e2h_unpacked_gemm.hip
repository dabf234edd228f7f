// Quantized linears over thousands of rows: the weights are unpacked to 16-bit values in scratch memory once per call, then multiplied
// by the loop of e2h_gemm256.h.
//
// int8: y = bf16( bf16( x @ q^T ) * scales ).  A code has at most eight significant bits, so its bfloat16 value is exact and the result is that
// of the kernels which convert on the way into the matrix cores (e2h_int8_gemm.hip).  Those are bound by the energy and the LDS traffic of 64-byte rows and
// by conversions beside the products.
//
// int4: y = bf16( sum_g sum_{k in g} x[m,k] (s[g,n] (q[n,k] - 8)) + sum_g z[g,n] X[m,g] ), X[m,g] = sum_{k in g} x[m,k].
// s (q - 8) is an eight-bit significand times a three-bit integer (or eight): it fits the eleven bits of a float16, and x (eight bits) does too.  So both become
// float16 without rounding, a row of x and a column of weights each in units of a power of two of its own that puts its largest value near the
// type's end; products are exact and sums float32, as in the kernel that multiplies codes (e2h_int4_gemm.hip: 1.1 - 1.2 PFLOP/s, bound by unpacking and rescaling
// beside the products).  The zero-point term is three more columns per group: X as g p0 + p1 + p2 of float16 values, against g z, z and z.  K grows by 2.4 % at
// group size 128.
// A value of x below about 2^-30 of its row's largest can have bits that its float16 does not hold, and so can the sum of a group of such values.  What is lacking
// stands in a list of the row's, and the store adds its products in float32 before the rounding (ordinary activations have such a value in one row of ten thousand).
// What does not fit is multiplied by that other kernel: the passes that unpack raise a flag at a scale or zero that is not finite, would be rounded
// (a scale below about 2^-28, a zero below 2^-31 of the larger of its column's 8 s and g z) or whose column's largest such value lies outside 2^-46 .. 2^45, at a value
// or group sum of x that is not finite, and at a row of x with more lacking values than its list holds.  With a flag of the weights the product's workgroups end at once and the
// other kernel does the call; with flags of rows it does these rows behind the product (the row blocks that hold one, of which it stores those rows), so that a row's result
// does not depend on what stands in others; without flags its workgroups end at once.  8192 x 12288 x 4096, group size 128: 660 us; a flag in the weights 735,
// one row 715, every row 767, where the other kernel alone takes 690.
#include <algorithm>

#include "e2h_common.h"
#include "e2h_gemm256.h"
#include "e2h_int4_unpack.h"

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

struct Int8Walk : gemm256::PlainWalk<> {
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
  __device__ __forceinline__ u32x4_t outputs(const Dest &d, int q, const float (&v)[8]) const {
    u32x4_t out;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t t = pack_bf16(v[2 * e], v[2 * e + 1]), s = d.scale[q][e];  // the linear's output, then its product with the scale, as in the reference
      out[e] = pack_bf16(__builtin_bit_cast(float, t << 16) * __builtin_bit_cast(float, s << 16),
                         __builtin_bit_cast(float, t & 0xFFFF0000u) * __builtin_bit_cast(float, s & 0xFFFF0000u));
    }
    return out;
  }
  __device__ __forceinline__ void store(const Tile &tile, const Dest &d, int, int q, int row, int col, float (&v)[8]) const {
    __builtin_amdgcn_raw_buffer_store_b128(outputs(d, q, v), y_rsrc(tile), y_at(tile, row, col), 0, 0);
  }
};

// Both matrices of silu(x w1) * (x w3): a lane ends up with the two products of its outputs.
struct Int8GateWalk : gemm256::PlainWalk<128> {
  const uint16_t *scales, *scales2;
  __device__ __forceinline__ Int8GateWalk(const uint16_t *x_, const uint16_t *w_, const uint16_t *scales_, const uint16_t *scales2_, uint16_t *y_, int M_, int N_, int K_)
      : PlainWalk(x_, w_, y_, M_, N_, K_), scales(scales_), scales2(scales2_) {}
  struct Dest {
    u32x4_t scale[2], scale2[2];
  };
  __device__ __forceinline__ void dest(const Tile &tile, int, int col, Dest &d) const {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int n = out_col(tile, col + 32 * q), at = n < N ? n : N - 8;
      d.scale[q] = *reinterpret_cast<const u32x4_t *>(scales + at);
      d.scale2[q] = *reinterpret_cast<const u32x4_t *>(scales2 + at);
    }
  }
  __device__ __forceinline__ void store(const Tile &tile, const Dest &d, int, int q, int row, int col, float (&v)[8], float (&u)[8]) const {
    const auto low = [](uint32_t b) { return __builtin_bit_cast(float, b << 16); };
    const auto high = [](uint32_t b) { return __builtin_bit_cast(float, b & 0xFFFF0000u); };
    u32x4_t g, up;
#pragma unroll
    for (int e = 0; e < 4; ++e) {  // the rounding points of the two linears
      const uint32_t a = pack_bf16(v[2 * e], v[2 * e + 1]), b = pack_bf16(u[2 * e], u[2 * e + 1]), sa = d.scale[q][e], sb = d.scale2[q][e];
      g[e] = pack_bf16(low(a) * low(sa), high(a) * high(sa));
      up[e] = pack_bf16(low(b) * low(sb), high(b) * high(sb));
    }
    __builtin_amdgcn_raw_buffer_store_b128(gemm256::gated(g, up), y_rsrc(tile), y_at(tile, row, col), 0, 0);
  }
};

__global__ __launch_bounds__(256, 1) void int8_unpacked_gate_kernel(const uint16_t *x, const uint16_t *w, const uint16_t *scales, const uint16_t *scales2, uint16_t *y, int M,
                                                                    int N, int K) {
#if defined(__HIP_DEVICE_COMPILE__)
  __shared__ __attribute__((aligned(1024))) uint8_t lds[gemm256::kRing];
  Int8GateWalk tiles(x, w, scales, scales2, y, M, N, K);
  gemm256::walk<false>(tiles, lds);
#endif
}

__global__ __launch_bounds__(256, 1) void int8_unpacked_gemm_kernel(const uint16_t *x, const uint16_t *w, const uint16_t *scales, uint16_t *y, int M, int N, int K) {
#if defined(__HIP_DEVICE_COMPILE__)
  __shared__ __attribute__((aligned(1024))) uint8_t lds[gemm256::kRing];
  Int8Walk tiles(x, w, scales, y, M, N, K);
  gemm256::walk<false>(tiles, lds);
#endif
}

// What a fused q | k | v product of B sequences of T tokens (row b T + t) leaves behind: q [B][H][T][D] and k, v [B][Hkv][S][D], q and k rotated by the angles of the tokens'
// positions.
struct RopeRows {
  const uint16_t *freqs;  // [freq_rows][D / 2][2]
  uint16_t *q, *k, *v;
  const int64_t *pos;     // [T]
  int B, T, H, Hkv, S, D, freq_rows, by_token;  // by_token: k and v of token t are row t, else row pos[t]
};

// Stores of a walk over such a product.  A wave's 128 columns belong to one of the three.  The angles of a row of its outputs (a 16-byte load beside each store) come
// kAhead - 1 rows ahead of their use, in registers that hold fragments in the main loop.
struct RopeStore {
  static constexpr int kAhead = 3;
  struct Dest {
    int pos[8];                   // of the lane's rows
    int b, t;                     // sequence and token of the row being stored
    u32x4_t cos_sin[kAhead][4];
  };
  const RopeRows &r;
  int row_base;  // of the walk's first row

  __device__ __forceinline__ void place(int row, Dest &d) const {
    const int m = row_base + row;
    d.b = m / r.T;
    d.t = m - d.b * r.T;
  }
  __device__ __forceinline__ void step(Dest &d) const {  // 16 rows on; T is no less
    d.t += 16;
    if (d.t >= r.T) {
      d.t -= r.T;
      ++d.b;
    }
  }
  __device__ __forceinline__ void dest(int row, Dest &d) const {
    place(row, d);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      d.pos[j] = static_cast<int>(reinterpret_cast<const uint32_t *>(r.pos)[2 * d.t]);
      step(d);
    }
  }
  __device__ __forceinline__ void request(Dest &d, int j, int col, bool rotated) const {
    const __amdgpu_buffer_rsrc_t f = make_rsrc(r.freqs, static_cast<uint32_t>(r.freq_rows) * static_cast<uint32_t>(r.D) * 2);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t at = static_cast<uint32_t>(d.pos[j]) * static_cast<uint32_t>(r.D) * 2 + static_cast<uint32_t>((col + 32 * q) & (r.D - 1)) * 2;
      d.cos_sin[j % kAhead][q] = __builtin_amdgcn_raw_buffer_load_b128(f, rotated && d.pos[j] >= 0 && d.pos[j] < r.freq_rows ? at : gemm256::kNowhere, 0, 0);
    }
  }
  // own: the outputs (row, n .. n + 7) of the product
  __device__ __forceinline__ void store(Dest &d, int j, int q, int row, int rows, int n, u32x4_t own) const {
    const auto low = [](uint32_t b) { return __builtin_bit_cast(float, b << 16); };
    const auto high = [](uint32_t b) { return __builtin_bit_cast(float, b & 0xFFFF0000u); };
    const int HD = r.H * r.D, KD = r.Hkv * r.D, wave_n = __builtin_amdgcn_readfirstlane(n) & ~127;
    const bool is_q = wave_n < HD, rotated = wave_n < HD + KD;
    if (q == 0) {
      if (j == 0) {
        place(row, d);
#pragma unroll
        for (int a = 0; a + 1 < kAhead; ++a) request(d, a, n, rotated);
      } else {
        step(d);
      }
      if (j + kAhead - 1 < 8) request(d, j + kAhead - 1, n, rotated);
    }
    u32x4_t out;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t x = own[e], f = d.cos_sin[j % kAhead][q][e];
      const float r0 = low(x) * low(f) - high(x) * high(f), r1 = high(x) * low(f) + low(x) * high(f);  // two rounded products, then their sum, as torch forms it
      out[e] = rotated ? pack_bf16(r0, r1) : x;
    }
    const int pos = d.pos[j], slot = r.by_token ? d.t : pos, at = n - (is_q ? 0 : rotated ? HD : HD + KD);
    const int heads = is_q ? r.H : r.Hkv, length = is_q ? r.T : r.S, log_d = r.D == 128 ? 7 : 6;
    const uint32_t line = static_cast<uint32_t>(d.b * heads + (at >> log_d)) * static_cast<uint32_t>(length) + static_cast<uint32_t>(is_q ? d.t : slot);
    const uint32_t to = ((line << log_d) + static_cast<uint32_t>(at & (r.D - 1))) * 2;
    const bool there = row < rows && pos >= 0 && slot >= 0 && slot < r.S && wave_n < HD + 2 * KD;
    const __amdgpu_buffer_rsrc_t y = make_rsrc(is_q ? r.q : rotated ? r.k : r.v, static_cast<uint32_t>(r.B * heads) * static_cast<uint32_t>(length) * static_cast<uint32_t>(r.D) * 2);
    __builtin_amdgcn_raw_buffer_store_b128(out, y, there ? to : gemm256::kNowhere, 0, 0);
  }
};

struct Int8RopeWalk : Int8Walk {
  RopeStore rope;
  __device__ __forceinline__ Int8RopeWalk(const uint16_t *x_, const uint16_t *w_, const uint16_t *scales_, const RopeRows &r, int row_base, int M_, int N_, int K_)
      : Int8Walk(x_, w_, scales_, nullptr, M_, N_, K_), rope{r, row_base} {}
  struct Dest {
    Int8Walk::Dest product;
    RopeStore::Dest rope;
  };
  __device__ __forceinline__ void dest(const Tile &tile, int row, int col, Dest &d) const {
    Int8Walk::dest(tile, row, col, d.product);
    rope.dest(tile.rb * 256 + row, d.rope);
  }
  __device__ __forceinline__ void store(const Tile &tile, Dest &d, int j, int q, int row, int col, float (&v)[8]) const {
    rope.store(d.rope, j, q, tile.rb * 256 + row, M, out_col(tile, col), outputs(d.product, q, v));
  }
};

__global__ __launch_bounds__(256, 1) void int8_unpacked_rope_kernel(const uint16_t *x, const uint16_t *w, const uint16_t *scales, const RopeRows r, int row_base, int M, int N, int K) {
#if defined(__HIP_DEVICE_COMPILE__)
  __shared__ __attribute__((aligned(1024))) uint8_t lds[gemm256::kRing];
  Int8RopeWalk tiles(x, w, scales, r, row_base, M, N, K);
  gemm256::walk<false>(tiles, lds);
#endif
}

// ---- int4 ------------------------------------------------------------------------------------------------------------------------
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t pack_f16(float lo, float hi) {  // round to nearest even; most callers' values are exact
  return __builtin_bit_cast(uint32_t, f16x2_t{static_cast<_Float16>(lo), static_cast<_Float16>(hi)});
}

constexpr int kTopX = 13, kTopW = 15;  // largest value of a row of x: 2^kTopX .. 2^(kTopX + 1); of a column: below 2^kTopW
constexpr float kWhole = 0x1p-17f;     // eight bits from here on fit a float16

struct Lacking {
  int at;    // column of the extended K
  float by;  // value of x, or sum of a group, less what its float16 values hold
};
constexpr int kMostLacking = 16;

struct Int4Scratch {
  int *flag;         // [1] what the other kernel does of this call: 1 everything, 2 the rows with row_flag, 0 nothing
  int *row_exp;      // [M] low half: x is multiplied by 2^that; high half: entries of the row's list
  int *row_flag;     // [M] 1: the other kernel's
  int *skip;         // [M / 256] all rows of the block are
  Lacking *lacking;  // [M][kMostLacking]
  float *col_unit;   // [N] what one step of a column's sums is worth
  float *xsum;       // [K / G][stride] group sums, for the other kernel
  uint16_t *x, *w;   // [M][KE], [N][KE]
  int64_t bytes;
};
int extended(int K, int G) { return (K + 3 * (K / G) + 63) / 64 * 64; }  // G: 32, 64 or 128
int sum_stride(int64_t M) { return static_cast<int>((M + 63) / 64 * 64); }

Int4Scratch int4_scratch(uint8_t *base, int64_t M, int64_t N, int64_t K, int groupsize) {
  const int G = groupsize == 256 ? 128 : groupsize;
  int64_t at = 0;
  const auto take = [&](int64_t n) {
    uint8_t *p = base + at;
    at += (n + 255) / 256 * 256;
    return p;
  };
  Int4Scratch s;
  const int64_t KE = extended(static_cast<int>(K), G);
  s.flag = reinterpret_cast<int *>(take(4));
  s.row_exp = reinterpret_cast<int *>(take(M * 4));
  s.row_flag = reinterpret_cast<int *>(take(M * 4));
  s.skip = reinterpret_cast<int *>(take((M + 255) / 256 * 4));
  s.lacking = reinterpret_cast<Lacking *>(take(M * kMostLacking * static_cast<int64_t>(sizeof(Lacking))));
  s.col_unit = reinterpret_cast<float *>(take(N * 4));
  s.xsum = reinterpret_cast<float *>(take(K / G * sum_stride(M) * 4));
  s.x = reinterpret_cast<uint16_t *>(take(M * KE * 2));
  s.w = reinterpret_cast<uint16_t *>(take(N * KE * 2));
  s.bytes = at;
  return s;
}

__device__ __forceinline__ int exponent_of(float v) { return static_cast<int>((__builtin_bit_cast(uint32_t, v) >> 23) & 0xFFu) - 127; }

// One wave per row, two passes over it (the second from the cache): largest value, then float16 values, group sums and their parts.
// Bound by memory: 8192 x 4096 (133 MB moved) 36 us.
template <int G>
__global__ __launch_bounds__(256) void int4_unpack_x_kernel(const uint16_t *__restrict__ x, int M, int K, int KE, Int4Scratch s, int stride) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *s.flag = 0;  // raised by the next launch
  const int lane = threadIdx.x & 63, m = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (m >= M) return;
  const u32x4_t *row = reinterpret_cast<const u32x4_t *>(x + static_cast<size_t>(m) * K);
  const int pieces = K / 8;  // a multiple of 16
  uint32_t top = 0;
#pragma unroll 4
  for (int p = lane; p < pieces; p += 64) {
    const u32x4_t v = row[p];
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const uint32_t lo = v[d] & 0x7FFFu, hi = (v[d] >> 16) & 0x7FFFu;
      top = top > lo ? top : lo;
      top = top > hi ? top : hi;
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const uint32_t o = static_cast<uint32_t>(__shfl_xor(static_cast<int>(top), off));
    top = top > o ? top : o;
  }
  const bool finite = top < 0x7F80u;
  const int up = top == 0 || !finite ? 0 : kTopX - exponent_of(bf16_to_f32(static_cast<uint16_t>(top)));
  uint16_t *out = s.x + static_cast<size_t>(m) * KE;
  Lacking *list = s.lacking + static_cast<size_t>(m) * kMostLacking;
  int lacking = 0;  // entries so far, in lane 0, which takes part in every round
  bool endless = !finite;
  const auto enter = [&](int at, float by) {  // of the lanes here, those whose `by` is not zero
    const uint64_t all = __builtin_amdgcn_ballot_w64(by != 0.f);
    const int i = lacking + __builtin_popcountll(all & ((uint64_t{1} << lane) - 1));
    if (by != 0.f && i < kMostLacking) list[i] = Lacking{at, by};
    lacking += __builtin_popcountll(all);
  };
#pragma unroll 2
  for (int p = lane; p < pieces; p += 64) {
    const u32x4_t v = row[p];
    u32x4_t h;
    float sum[4];
    bool small = false;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const float a = __builtin_bit_cast(float, v[d] << 16), b = __builtin_bit_cast(float, v[d] & 0xFFFF0000u);
      sum[d] = a + b;
      const float as = __builtin_ldexpf(a, up), bs = __builtin_ldexpf(b, up);
      small |= (a != 0.f && __builtin_fabsf(as) < kWhole) || (b != 0.f && __builtin_fabsf(bs) < kWhole);
      h[d] = pack_f16(as, bs);
    }
    reinterpret_cast<u32x4_t *>(out)[p] = h;
    if (__builtin_amdgcn_ballot_w64(small)) {  // hardly ever
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const uint32_t pair = h[d];  // (a bit cast of the element itself reads the vector's first one)
        const f16x2_t held = __builtin_bit_cast(f16x2_t, pair);
        enter(8 * p + 2 * d, __builtin_bit_cast(float, v[d] << 16) - __builtin_ldexpf(static_cast<float>(held[0]), -up));
        enter(8 * p + 2 * d + 1, __builtin_bit_cast(float, v[d] & 0xFFFF0000u) - __builtin_ldexpf(static_cast<float>(held[1]), -up));
      }
    }
    float t = (sum[0] + sum[1]) + (sum[2] + sum[3]);
#pragma unroll
    for (int off = 1; off < G / 8; off <<= 1) t += __shfl_xor(t, off);  // the lanes of a group are all here or none
    const int g = p / (G / 8);
    const float ts = __builtin_ldexpf(t, up);
    const _Float16 p0 = static_cast<_Float16>(ts * (1.0f / G));
    const float r = ts - static_cast<float>(p0) * G;
    const _Float16 p1 = static_cast<_Float16>(r), p2 = static_cast<_Float16>(r - static_cast<float>(p1));
    endless |= !__builtin_isfinite(t);
    float by = 0.f;
    if (lane % (G / 8) == 0) {
      s.xsum[static_cast<size_t>(g) * stride + m] = t;
      out[K + 3 * g] = __builtin_bit_cast(uint16_t, p0);
      out[K + 3 * g + 1] = __builtin_bit_cast(uint16_t, p1);
      out[K + 3 * g + 2] = __builtin_bit_cast(uint16_t, p2);
      by = t - __builtin_ldexpf((static_cast<float>(p0) * G + static_cast<float>(p1)) + static_cast<float>(p2), -up);
    }
    if (__builtin_amdgcn_ballot_w64(by != 0.f)) enter(K + 3 * g + 1, by);
  }
  for (int k = K + 3 * (K / G) + lane; k < KE; k += 64) out[k] = 0;
  const bool odd = __builtin_amdgcn_ballot_w64(endless) != 0 || lacking > kMostLacking;
  if (lane == 0) {
    s.row_exp[m] = (up & 0xFFFF) | (odd ? 0 : lacking << 16);
    s.row_flag[m] = odd;
  }
}

// Sixteen columns and a share of K per workgroup: the columns' units first (every share finds them for itself), then a lane per 16-byte piece
// of the result.  Bound by memory: 12288 x 4096 (130 MB moved) 36 us.
template <int G>
__global__ __launch_bounds__(256) void int4_unpack_w_kernel(const uint32_t *__restrict__ wp, const uint32_t *__restrict__ sz, int twice, int M, int N, int K, int KE,
                                                            Int4Scratch s) {
  __shared__ float top_of[16][17];
  __shared__ int raised;
  const int groups = K / G, tid = threadIdx.x, col0 = blockIdx.x * 16;
  if (tid == 0) raised = 0;
  __syncthreads();
  // every row's flag, shared among all workgroups
  int odd = 0;
  for (int64_t m0 = (static_cast<int64_t>(blockIdx.y) * gridDim.x + blockIdx.x) * 256; m0 < M; m0 += static_cast<int64_t>(gridDim.x) * gridDim.y * 256) {
    const bool there = m0 + tid < M;
    const int flag = there ? s.row_flag[m0 + tid] : 1, all = __syncthreads_and(flag);
    if (there) odd |= flag << 1;
    if (tid == 0) s.skip[m0 >> 8] = all;
  }
  const int c1 = tid & 15, g1 = tid >> 4;
  const bool live1 = col0 + c1 < N;
  float top = 0.f;
  if (live1)
    for (int g = g1; g < groups; g += 16) {
      const uint32_t pair = sz[static_cast<size_t>(g >> twice) * N + col0 + c1];
      const float scale = __builtin_bit_cast(float, pair << 16), zero = __builtin_bit_cast(float, pair & 0xFFFF0000u);
      odd |= !__builtin_isfinite(scale) || !__builtin_isfinite(zero);
      top = fmaxf(top, fmaxf(8.f * __builtin_fabsf(scale), static_cast<float>(G) * __builtin_fabsf(zero)));
    }
  top_of[c1][g1] = top;
  __syncthreads();
  const auto unit_of = [&](int c) {  // the power of two that the column is multiplied by
    float t = 0.f;
#pragma unroll
    for (int g = 0; g < 16; ++g) t = fmaxf(t, top_of[c][g]);
    return t == 0.f ? 0 : kTopW - 1 - exponent_of(t);
  };
  const int up1 = unit_of(c1);
  odd |= live1 && (up1 < -30 || up1 > 60);
  if (live1)
    for (int g = g1; g < groups; g += 16) {
      const uint32_t pair = sz[static_cast<size_t>(g >> twice) * N + col0 + c1];
      const float scale = __builtin_bit_cast(float, pair << 16), zero = __builtin_bit_cast(float, pair & 0xFFFF0000u);
      const float a = __builtin_fabsf(__builtin_ldexpf(scale, up1)), z = __builtin_ldexpf(zero, up1);
      odd |= (scale != 0.f && a < kWhole) || (zero != 0.f && __builtin_fabsf(z) < kWhole);
      if (blockIdx.y == 0) {
        uint16_t *ext = s.w + static_cast<size_t>(col0 + c1) * KE + K + 3 * g;
        ext[0] = __builtin_bit_cast(uint16_t, static_cast<_Float16>(z * static_cast<float>(G)));
        ext[1] = ext[2] = __builtin_bit_cast(uint16_t, static_cast<_Float16>(z));
      }
    }
  if (blockIdx.y == 0 && live1) {
    for (int k = K + 3 * groups + g1; k < KE; k += 16) s.w[static_cast<size_t>(col0 + c1) * KE + k] = 0;
    if (g1 == 0) s.col_unit[col0 + c1] = __builtin_ldexpf(1.f, -up1);
  }
  if (odd) atomicOr(&raised, odd);
  __syncthreads();
  if (tid == 0 && raised) atomicOr(s.flag, raised);

  // piece (span p, part i) of column c: codes k = 128 b + 32 p + 8 i + 2 j + {0, 1} in nibbles i and i + 4 of word [j][p]
  const int c = tid >> 4, p = (tid >> 2) & 3, i = tid & 3, col = col0 + c, KT = K >> 7;
  if (col >= N) return;
  const int up = unit_of(c);
  const uint32_t *words = wp + static_cast<size_t>(col >> 3) * KT * 128 + (col & 7) * 16 + p;
  uint16_t *out = s.w + static_cast<size_t>(col) * KE + 32 * p + 8 * i;
  const int b1 = static_cast<int>(static_cast<int64_t>(KT) * (blockIdx.y + 1) / gridDim.y);
#pragma unroll 4
  for (int b = static_cast<int>(static_cast<int64_t>(KT) * blockIdx.y / gridDim.y); b < b1; ++b) {
    const int g = (128 * b + 32 * p + 8 * i) / G;
    const float scale = __builtin_ldexpf(__builtin_bit_cast(float, sz[static_cast<size_t>(g >> twice) * N + col] << 16), up);
    u32x4_t h;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t w = words[static_cast<size_t>(b) * 128 + 4 * j];
      const float q0 = static_cast<float>((w >> (4 * i)) & 15u), q1 = static_cast<float>((w >> (4 * i + 16)) & 15u);
      h[j] = pack_f16(__builtin_fmaf(q0, scale, -8.f * scale), __builtin_fmaf(q1, scale, -8.f * scale));
    }
    *reinterpret_cast<u32x4_t *>(out + static_cast<size_t>(b) * 128) = h;
  }
}

// Eight sums of a row and the columns n .. n + 7 (rows n + first .. of w), back in the operands' units and with what the row's float16 values lack.  up: the row's row_exp.
template <class Walk>
__device__ __forceinline__ void finish_int4(const Walk &walk, const typename Walk::Tile &tile, int up, const f32x4_t (&unit)[2], int row, int n, int first, float (&v)[8]) {
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = __builtin_ldexpf(v[e] * unit[e >> 2][e & 3], -static_cast<int>(static_cast<int16_t>(up)));
  if (__builtin_expect(up >= 1 << 16, 0)) {
    const int m = tile.rb * 256 + row;
    const Lacking *list = walk.lacking + static_cast<size_t>(m < walk.M ? m : walk.M - 1) * kMostLacking;
    const __amdgpu_buffer_rsrc_t wr = walk.w_rsrc(tile);
#pragma unroll 1
    for (int i = 0; i < up >> 16; ++i) {
      const Lacking l = list[i];
#pragma unroll
      for (int e = 0; e < 8; ++e) {  // (columns past N: of column 0, not stored)
        const uint32_t at = (static_cast<uint32_t>(first + (n < walk.N ? n + e : 0)) * static_cast<uint32_t>(walk.K) + static_cast<uint32_t>(l.at)) * 2;
        const float w = static_cast<float>(__builtin_bit_cast(_Float16, __builtin_amdgcn_raw_buffer_load_b16(wr, at, 0, 0)));
        v[e] = __builtin_fmaf(l.by, w * unit[e >> 2][e & 3], v[e]);
      }
    }
  }
}

struct Int4Walk : gemm256::PlainWalk<> {
  const float *col_unit;
  const int *row_exp, *skip;
  const Lacking *lacking;
  __device__ __forceinline__ Int4Walk(const Int4Scratch &s, uint16_t *y_, int M_, int N_, int KE)
      : PlainWalk(s.x, s.w, y_, M_, N_, KE), col_unit(s.col_unit), row_exp(s.row_exp), skip(s.skip), lacking(s.lacking) {}
  __device__ __forceinline__ bool next(Tile &tile) {
    while (PlainWalk::next(tile))
      if (!skip[tile.rb]) return true;
    return false;
  }
  __device__ __forceinline__ bool first(Tile &tile) { return next(tile); }
  struct Dest {
    f32x4_t unit[4][2];  // of the eight columns of each store of a row
    int up[8];           // row_exp of the rows
  };
  __device__ __forceinline__ void dest(const Tile &tile, int row, int col, Dest &d) const {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int n = tile.cb * 256 + col + 32 * q;
      const f32x4_t *u = reinterpret_cast<const f32x4_t *>(col_unit + (n < N ? n : N - 8));
      d.unit[q][0] = u[0];
      d.unit[q][1] = u[1];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int m = tile.rb * 256 + row + 16 * j;
      d.up[j] = row_exp[m < M ? m : M - 1];
    }
  }
  __device__ __forceinline__ u32x4_t outputs(const Tile &tile, const Dest &d, int j, int q, int row, int col, float (&v)[8]) const {
    u32x4_t out;
    finish_int4(*this, tile, d.up[j], d.unit[q], row, out_col(tile, col), 0, v);
#pragma unroll
    for (int e = 0; e < 4; ++e) out[e] = pack_bf16(v[2 * e], v[2 * e + 1]);
    return out;
  }
  __device__ __forceinline__ void store(const Tile &tile, const Dest &d, int j, int q, int row, int col, float (&v)[8]) const {
    __builtin_amdgcn_raw_buffer_store_b128(outputs(tile, d, j, q, row, col, v), y_rsrc(tile), y_at(tile, row, col), 0, 0);
  }
};

struct Int4RopeWalk : Int4Walk {
  RopeStore rope;
  __device__ __forceinline__ Int4RopeWalk(const Int4Scratch &s, const RopeRows &r, int M_, int N_, int KE) : Int4Walk(s, nullptr, M_, N_, KE), rope{r, 0} {}
  struct Dest {
    Int4Walk::Dest product;
    RopeStore::Dest rope;
  };
  __device__ __forceinline__ void dest(const Tile &tile, int row, int col, Dest &d) const {
    Int4Walk::dest(tile, row, col, d.product);
    rope.dest(tile.rb * 256 + row, d.rope);
  }
  __device__ __forceinline__ void store(const Tile &tile, Dest &d, int j, int q, int row, int col, float (&v)[8]) const {
    rope.store(d.rope, j, q, tile.rb * 256 + row, M, out_col(tile, col), outputs(tile, d.product, j, q, row, col, v));
  }
};

// Both matrices of silu(x w1) * (x w3), the second one's rows and units behind the first one's.
struct Int4GateWalk : gemm256::PlainWalk<128> {
  const float *col_unit;
  const int *row_exp, *skip;
  const Lacking *lacking;
  __device__ __forceinline__ Int4GateWalk(const Int4Scratch &s, uint16_t *y_, int M_, int N_, int KE)
      : PlainWalk(s.x, s.w, y_, M_, N_, KE), col_unit(s.col_unit), row_exp(s.row_exp), skip(s.skip), lacking(s.lacking) {}
  __device__ __forceinline__ bool next(Tile &tile) {
    while (PlainWalk::next(tile))
      if (!skip[tile.rb]) return true;
    return false;
  }
  __device__ __forceinline__ bool first(Tile &tile) { return next(tile); }
  struct Dest {
    f32x4_t unit[2][2][2];  // of the eight columns of each store of a row, in both matrices
    int up[8];
  };
  __device__ __forceinline__ void dest(const Tile &tile, int row, int col, Dest &d) const {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int n = out_col(tile, col + 32 * q), at = n < N ? n : N - 8;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const f32x4_t *u = reinterpret_cast<const f32x4_t *>(col_unit + h * N + at);
        d.unit[q][h][0] = u[0];
        d.unit[q][h][1] = u[1];
      }
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int m = tile.rb * 256 + row + 16 * j;
      d.up[j] = row_exp[m < M ? m : M - 1];
    }
  }
  __device__ __forceinline__ void store(const Tile &tile, const Dest &d, int j, int q, int row, int col, float (&v)[8], float (&u)[8]) const {
    const int n = out_col(tile, col);
    finish_int4(*this, tile, d.up[j], d.unit[q][0], row, n, 0, v);
    finish_int4(*this, tile, d.up[j], d.unit[q][1], row, n, N, u);
    u32x4_t g, up;
#pragma unroll
    for (int e = 0; e < 4; ++e) g[e] = pack_bf16(v[2 * e], v[2 * e + 1]), up[e] = pack_bf16(u[2 * e], u[2 * e + 1]);
    __builtin_amdgcn_raw_buffer_store_b128(gemm256::gated(g, up), y_rsrc(tile), y_at(tile, row, col), 0, 0);
  }
};

__global__ __launch_bounds__(256, 1) void int4_unpacked_gemm_kernel(const Int4Scratch s, uint16_t *y, int M, int N, int KE) {
#if defined(__HIP_DEVICE_COMPILE__)
  if (*s.flag & 1) return;  // the whole grid
  __shared__ __attribute__((aligned(1024))) uint8_t lds[gemm256::kRing];
  Int4Walk tiles(s, y, M, N, KE);
  gemm256::walk<true>(tiles, lds);
#endif
}

__global__ __launch_bounds__(256, 1) void int4_unpacked_gate_kernel(const Int4Scratch s, uint16_t *y, int M, int N, int KE) {
#if defined(__HIP_DEVICE_COMPILE__)
  if (*s.flag & 1) return;  // the whole grid
  __shared__ __attribute__((aligned(1024))) uint8_t lds[gemm256::kRing];
  Int4GateWalk tiles(s, y, M, N, KE);
  gemm256::walk<true>(tiles, lds);
#endif
}

__global__ __launch_bounds__(256, 1) void int4_unpacked_rope_kernel(const Int4Scratch s, const RopeRows r, int M, int N, int KE) {
#if defined(__HIP_DEVICE_COMPILE__)
  if (*s.flag & 1) return;  // the whole grid
  __shared__ __attribute__((aligned(1024))) uint8_t lds[gemm256::kRing];
  Int4RopeWalk tiles(s, r, M, N, KE);
  gemm256::walk<true>(tiles, lds);
#endif
}

// What RopeStore does, for the rows that the other kernel left in y: those with row_flag, or all.  A wave per row.
__global__ __launch_bounds__(256) void rope_flagged_rows_kernel(const uint16_t *__restrict__ y, const Int4Scratch s, const RopeRows r) {
  const int asked = *s.flag;
  if (asked == 0) return;
  const int lane = threadIdx.x & 63, HD = r.H * r.D, KD = r.Hkv * r.D, N = HD + 2 * KD, M = r.B * r.T;
  for (int m = blockIdx.x * 4 + (threadIdx.x >> 6); m < M; m += gridDim.x * 4) {
    if (!(asked & 1) && !s.row_flag[m]) continue;
    const int b = m / r.T, t = m - b * r.T, pos = static_cast<int>(r.pos[t]), slot = r.by_token ? t : pos;
    if (pos < 0 || slot < 0 || slot >= r.S) continue;
    for (int n = 2 * lane; n < N; n += 128) {
      const bool is_q = n < HD, rotated = n < HD + KD;
      const int at = n - (is_q ? 0 : rotated ? HD : HD + KD), head = at / r.D, d = at - head * r.D;
      uint32_t pair = *reinterpret_cast<const uint32_t *>(y + static_cast<size_t>(m) * N + n);
      if (rotated) {
        const uint32_t f = pos < r.freq_rows ? *reinterpret_cast<const uint32_t *>(r.freqs + static_cast<size_t>(pos) * r.D + d) : 0u;
        const float x0 = __builtin_bit_cast(float, pair << 16), x1 = __builtin_bit_cast(float, pair & 0xFFFF0000u);
        const float cs = __builtin_bit_cast(float, f << 16), sn = __builtin_bit_cast(float, f & 0xFFFF0000u);
        pair = pack_bf16(x0 * cs - x1 * sn, x1 * cs + x0 * sn);
      }
      uint16_t *out = is_q ? r.q + ((static_cast<size_t>(b) * r.H + head) * r.T + t) * r.D : (rotated ? r.k : r.v) + ((static_cast<size_t>(b) * r.Hkv + head) * r.S + slot) * r.D;
      *reinterpret_cast<uint32_t *>(out + d) = pair;
    }
  }
}

template <int G>
void launch_unpack(const uint16_t *x, const uint32_t *wp, const uint32_t *sz, const Int4Scratch &s, int twice, int M, int N, int K, int KE, hipStream_t stream) {
  if (x) hipLaunchKernelGGL(int4_unpack_x_kernel<G>, dim3(static_cast<unsigned>((M + 3) / 4)), dim3(256), 0, stream, x, M, K, KE, s, sum_stride(M));
  const int cols = (N + 15) / 16, shares = std::max(1, std::min(K / 512, (4096 + cols - 1) / cols));  // at least four blocks of 128 k each
  hipLaunchKernelGGL(int4_unpack_w_kernel<G>, dim3(static_cast<unsigned>(cols), static_cast<unsigned>(shares)), dim3(256), 0, stream, wp, sz, twice, M, N, K, KE, s);
}

// x null: it is unpacked already
void unpack(const uint16_t *x, const int32_t *packed, const uint16_t *scales_and_zeros, const Int4Scratch &s, int groupsize, int M, int N, int K, hipStream_t stream) {
  const int twice = groupsize == 256, G = twice ? 128 : groupsize, KE = extended(K, G);
  const uint32_t *wp = reinterpret_cast<const uint32_t *>(packed), *sz = reinterpret_cast<const uint32_t *>(scales_and_zeros);
  switch (G) {
    case 32: launch_unpack<32>(x, wp, sz, s, twice, M, N, K, KE, stream); break;
    case 64: launch_unpack<64>(x, wp, sz, s, twice, M, N, K, KE, stream); break;
    default: launch_unpack<128>(x, wp, sz, s, twice, M, N, K, KE, stream); break;
  }
}

unsigned grid_of(int64_t M, int64_t N, int64_t cols = gemm256::kSide) { return gemm256::grid_of((M + 255) / 256 * ((N + cols - 1) / cols)); }

}  // namespace

// Microseconds of a product with the unpacked weights, within 10 % of 48 measured shapes of 1024 .. 8192 rows: 1.36 per chunk of 64 k and 5 per round of 256 tiles; a last
// round that is not full runs at a higher clock.
double unpacked_cost(int64_t M, int64_t N, int64_t K, double unpack) {
  const int64_t tiles = ((M + 255) / 256) * ((N + 255) / 256), full = tiles / 256, rest = tiles % 256;
  const double rounds = static_cast<double>(full) + (rest == 0 ? 0. : full == 0 ? 1. : 0.6 + 0.4 * static_cast<double>(rest) / 256);
  return unpack + 4 + rounds * (static_cast<double>(K) / 64 * 1.36 + 5);
}

// The same of the kernel that multiplies codes (e2h_int4_gemm.hip) with a thousand rows and more and one K slice: the cost that int4_gemm_shape picks its rows per workgroup by, which holds
// for chips full of matrix work (its expected time is fitted to fewer rows), and what more of the rescaling group sizes 32 and 64 cost there.
double int4_codes_cost(int64_t M, int64_t N, int64_t K, int groupsize) {
  constexpr double kOne[] = {1.2, 1.47, 1.85}, kTwo[] = {1.95, 2.42, 3.3};
  double best = -1;
  for (int i = 0; i < (groupsize == 32 ? 1 : 3); ++i) {
    const int64_t rows = 64 + 32 * i, per_cu = ((M + rows - 1) / rows * (((N + 255) / 256 + 7) / 8) + 31) / 32;
    const double cost = (static_cast<double>(per_cu / 2) * kTwo[i] + (per_cu & 1 ? kOne[i] : 0)) * static_cast<double>(K / 128) + 3;
    if (best < 0 || cost < best) best = cost;
  }
  return groupsize == 32 ? 1.3 * best : groupsize == 64 ? 1.15 * best : best;
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
// Known to be off over a short K, where a last round that is not full takes as long as a full one: 1280 rows 16384 x 1024 66 us, 57 in the other form.
int64_t int8_unpacked_bytes(int64_t M, int64_t N, int64_t K) {
  if (M < 1 || N < 8 || N % 8 != 0 || K % 128 != 0 || K < 256 || N > INT32_MAX || K > INT32_MAX || N * K * 2 >= (int64_t{1} << 32)) return 0;
  const Options &o = options();
  if (o.int4_no_gemm32 || o.int8_force_generic || o.int8_gemm_tile || o.int8_gemm_waves || o.int8_gemm_wave_cols || o.int8_rows_per_wave) return 0;  // another form is asked for
  return unpacked_cost(M, N, K, static_cast<double>(N) * static_cast<double>(K) * 3 / 4.8e6) < int8_gemm32_cost(M, N, K) ? N * K * 2 : 0;
}

// rows in slices that a 32-bit offset reaches
int64_t rows_at_once(int64_t K) { return ((int64_t{1} << 32) - 1) / (2 * K) / 256 * 256; }

int int8_unpacked_gemm(const uint16_t *x, const int8_t *q, const uint16_t *scales, uint16_t *y, int M, int N, int K, uint16_t *w, hipStream_t stream) {
  const int64_t pieces = static_cast<int64_t>(N) * K / 16;
  hipLaunchKernelGGL(unpack_int8_kernel, dim3(static_cast<unsigned>((pieces + 255) / 256)), dim3(256), 0, stream, q, w, pieces);
  const int64_t most = rows_at_once(K);
  for (int64_t m0 = 0; m0 < M; m0 += most) {
    const int rows = static_cast<int>(M - m0 < most ? M - m0 : most);
    hipLaunchKernelGGL(int8_unpacked_gemm_kernel, dim3(grid_of(rows, N)), dim3(256), 0, stream, x + m0 * K, w, scales, y + m0 * N, rows, N, K);
  }
  return launch_status();
}

// Taken where it is the cheaper one, the unpacking (two and a half bytes a weight, four a value of x, at 4.8 TB/s; 8 us of launches) included.  Measured, us, here (codes multiplied
// in the loop): 8192 rows 12288 x 4096 g128 647 (695), 32000 x 4096 1664 (1793), 12288 x 4096 g32 699 (1056), g64 656 (765), g256 644; 3000 rows 32000 x 4096 g64 685 (804), 2048 rows 12288 x 4096 g128 230
// (204), left to the other form.
int64_t int4_unpacked_bytes(int64_t M, int64_t N, int64_t K, int groupsize, int inner_k_tiles) {
  if (inner_k_tiles != 8 || (groupsize != 32 && groupsize != 64 && groupsize != 128 && groupsize != 256)) return 0;
  const int G = groupsize == 256 ? 128 : groupsize;
  if (M <= 64 || N < 8 || N % 8 != 0 || K < 256 || K % 128 != 0 || K % groupsize != 0 || M > INT32_MAX / 64 || N > INT32_MAX / 64 || K > INT32_MAX / 64) return 0;
  const Options &o = options();
  if (o.int4_no_gemm32 || o.int4_gemm_tile || o.int4_gemm32_min_rows || o.int4_no_xsum || o.int4_k_slices || o.int4_rows_per_wave || o.row_tiles) return 0;  // another form is asked for
  const int64_t KE = extended(static_cast<int>(K), G);
  if (M * KE * 2 >= (int64_t{1} << 32) || N * KE * 2 >= (int64_t{1} << 32) || K / G * sum_stride(M) * 4 >= (int64_t{1} << 32)) return 0;
  const int64_t bytes = int4_scratch(nullptr, M, N, K, groupsize).bytes;
  const double unpack = (static_cast<double>(N) * static_cast<double>(K) * 2.5 + static_cast<double>(M) * static_cast<double>(K) * 4) / 4.8e6 + 8;
  return unpacked_cost(M, N, KE, unpack) < int4_codes_cost(M, N, K, G) ? bytes : 0;
}

int int4_unpacked_gemm(const uint16_t *x, const int32_t *packed, const uint16_t *scales_and_zeros, uint16_t *y, int M, int N, int K, int groupsize, void *scratch,
                       hipStream_t stream) {
  const Int4Scratch s = int4_scratch(static_cast<uint8_t *>(scratch), M, N, K, groupsize);
  const int G = groupsize == 256 ? 128 : groupsize, KE = extended(K, G);
  unpack(x, packed, scales_and_zeros, s, groupsize, M, N, K, stream);
  hipLaunchKernelGGL(int4_unpacked_gemm_kernel, dim3(grid_of(M, N)), dim3(256), 0, stream, s, y, M, N, KE);
  return int4_gemm(x, packed, scales_and_zeros, y, s.xsum, sum_stride(M), nullptr, int4_gemm_shape(M, N, K, G, 0), M, N, K, groupsize, stream, s.flag, s.row_flag);
}

// A pass over the results of two calls, which gates them: six bytes an output.
double gate_pass_cost(int64_t M, int64_t N) { return 3 + static_cast<double>(M) * static_cast<double>(N) * 6 / 5e6; }

// Scratch of a gated call on unpacked operands, or 0 where it is not taken: where it is not expected to be 3 % faster than two calls, whichever form those have, and that pass, or, int4, than
// the gated launch on codes.  Measured, us, two calls and the pass / here: int8 2 x 11008 x 4096 1500 rows 385 / 303, 8192 rows 1166 / 1044, 2 x 22016 x 8192 3000 rows 1911 / 1770,
// 1200 rows 774 / 870: not taken; int4 2 x 11008 x 4096 g128 8192 rows 1327 / 1159, g64 2048 rows 446 / 378, g32 1200 rows 319 / 304.
int64_t int8_gate_unpacked_bytes(int64_t M, int64_t N, int64_t K) {
  if (M < 1024 || N < 8 || N > INT32_MAX / 2 || N % 8 != 0) return 0;
  const int64_t bytes = int8_unpacked_bytes(M, 2 * N, K);
  if (bytes == 0) return 0;
  const double unpack = static_cast<double>(N) * static_cast<double>(K) * 3 / 4.8e6;
  const double call = std::min(unpacked_cost(M, N, K, unpack), int8_gemm32_cost(M, N, K));
  return 1.03 * unpacked_cost(M, 2 * N, K, 2 * unpack) < 2 * call + gate_pass_cost(M, N) ? bytes : 0;
}

int64_t int4_gate_unpacked_bytes(int64_t M, int64_t N, int64_t K, int groupsize, int inner_k_tiles) {
  if (M < 1024 || N < 8 || N > INT32_MAX / 2 || N % 8 != 0) return 0;
  const int64_t bytes = int4_unpacked_bytes(M, 2 * N, K, groupsize, inner_k_tiles);
  if (bytes == 0) return 0;
  const int G = groupsize == 256 ? 128 : groupsize;
  const int64_t KE = extended(static_cast<int>(K), G);
  const double w = static_cast<double>(N) * static_cast<double>(K) * 2.5 / 4.8e6, rows = static_cast<double>(M) * static_cast<double>(K) * 4 / 4.8e6 + 8;
  const double call = std::min(unpacked_cost(M, N, KE, w + rows), int4_codes_cost(M, N, K, G));
  return 1.03 * unpacked_cost(M, 2 * N, KE, 2 * w + rows) < std::min(2 * call + gate_pass_cost(M, N), int4_codes_cost(M, 2 * N, K, G)) ? bytes : 0;
}

// y = bf16( bf16(silu(bf16(x w1))) * bf16(x w3) ), scratch of int4_unpacked_bytes for both matrices' columns: x is unpacked once, the tiles of both products fill the chip
// together, and the gate costs a tile what its lanes compute.  8192 x 2 x 11008 x 4096, group size 128: 1327 us in two calls and a pass over their results, 1159.
int int4_unpacked_gate(const uint16_t *x, const int32_t *packed, const uint16_t *sz, const int32_t *packed2, const uint16_t *sz2, uint16_t *y, int M, int N, int K, int groupsize,
                       void *scratch, hipStream_t stream) {
  const Int4Scratch s = int4_scratch(static_cast<uint8_t *>(scratch), M, 2 * static_cast<int64_t>(N), K, groupsize);
  const int G = groupsize == 256 ? 128 : groupsize, KE = extended(K, G);
  Int4Scratch second = s;
  second.w += static_cast<int64_t>(N) * KE;
  second.col_unit += N;
  unpack(x, packed, sz, s, groupsize, M, N, K, stream);
  unpack(nullptr, packed2, sz2, second, groupsize, M, N, K, stream);
  hipLaunchKernelGGL(int4_unpacked_gate_kernel, dim3(grid_of(M, N, 128)), dim3(256), 0, stream, s, y, M, N, KE);
  return int4_gemm_gate(x, packed, sz, packed2, sz2, y, s.xsum, sum_stride(M), int4_gemm_shape(M, 2 * N, K, G, 0), M, N, K, groupsize, stream, s.flag, s.row_flag);
}

// The same of int8 linears, scratch of int8_unpacked_bytes for both matrices' rows.  8192 x 2 x 11008 x 4096: 1166 us, 1044.
int int8_unpacked_gate(const uint16_t *x, const int8_t *q, const uint16_t *scales, const int8_t *q2, const uint16_t *scales2, uint16_t *y, int M, int N, int K, uint16_t *w,
                       hipStream_t stream) {
  const int64_t pieces = static_cast<int64_t>(N) * K / 16;
  const dim3 grid(static_cast<unsigned>((pieces + 255) / 256));
  hipLaunchKernelGGL(unpack_int8_kernel, grid, dim3(256), 0, stream, q, w, pieces);
  hipLaunchKernelGGL(unpack_int8_kernel, grid, dim3(256), 0, stream, q2, w + static_cast<int64_t>(N) * K, pieces);
  const int64_t most = rows_at_once(K);
  for (int64_t m0 = 0; m0 < M; m0 += most) {
    const int rows = static_cast<int>(M - m0 < most ? M - m0 : most);
    hipLaunchKernelGGL(int8_unpacked_gate_kernel, dim3(grid_of(rows, N, 128)), dim3(256), 0, stream, x + m0 * K, w, scales, scales2, y + m0 * N, rows, N, K);
  }
  return launch_status();
}

// Scratch of a fused q | k | v product whose tiles rotate, transpose and write the caches themselves, or 0 where it is not taken.  Where the product alone runs on unpacked
// weights this is it and no pass over its results behind it (four bytes an output at 5.9 TB/s), for 3 us a round of tiles: 49152 x 12288 x 4096 and the pass 3290 + 413 us, here 3420.
bool rope_rows_fit(int64_t batch, int64_t seqlen, int64_t n_head, int64_t n_kv_head, int64_t cache_len, int64_t head_dim) {
  constexpr int64_t kMost = (int64_t{1} << 32) - 512;  // bytes that a 32-bit offset reaches
  if (batch < 1 || seqlen < 16 || n_head < 1 || n_kv_head < 1 || cache_len < 1 || (head_dim != 64 && head_dim != 128)) return false;
  if (batch > INT32_MAX / 2 / seqlen || n_head > INT32_MAX / 1024 || n_kv_head > INT32_MAX / 1024 || cache_len > INT32_MAX / 2 / head_dim) return false;
  const int64_t q = n_head * head_dim, kv = n_kv_head * head_dim;
  return q % 128 == 0 && kv % 128 == 0 && q <= kMost / 2 / (batch * seqlen) && kv <= kMost / 2 / batch / cache_len;
}
int64_t int8_unpacked_rope_bytes(int64_t batch, int64_t seqlen, int64_t n_head, int64_t n_kv_head, int64_t cache_len, int64_t head_dim, int64_t K) {
  return rope_rows_fit(batch, seqlen, n_head, n_kv_head, cache_len, head_dim) ? int8_unpacked_bytes(batch * seqlen, (n_head + 2 * n_kv_head) * head_dim, K) : 0;
}
// The same of int4 linears, with room for the rows that the other kernel forms, which a small pass rotates behind it (5 us where there are none).  32 prompts of 256 tokens through two int4
// 7B layers: 7495 us with the pass over all results, 7405.
int64_t int4_unpacked_rope_bytes(int64_t batch, int64_t seqlen, int64_t n_head, int64_t n_kv_head, int64_t cache_len, int64_t head_dim, int64_t K, int groupsize, int inner_k_tiles) {
  if (!rope_rows_fit(batch, seqlen, n_head, n_kv_head, cache_len, head_dim) || batch * seqlen < 1024) return 0;
  const int64_t M = batch * seqlen, N = (n_head + 2 * n_kv_head) * head_dim, bytes = int4_unpacked_bytes(M, N, K, groupsize, inner_k_tiles);
  return bytes == 0 ? 0 : bytes + M * N * 2;
}

int int4_unpacked_rope(const uint16_t *x, const int32_t *packed, const uint16_t *sz, const RopeRows &r, int K, int groupsize, void *scratch, hipStream_t stream) {
  const int N = (r.H + 2 * r.Hkv) * r.D, M = r.B * r.T;
  const Int4Scratch s = int4_scratch(static_cast<uint8_t *>(scratch), M, N, K, groupsize);
  const int G = groupsize == 256 ? 128 : groupsize, KE = extended(K, G);
  uint16_t *y = reinterpret_cast<uint16_t *>(static_cast<uint8_t *>(scratch) + s.bytes);
  unpack(x, packed, sz, s, groupsize, M, N, K, stream);
  hipLaunchKernelGGL(int4_unpacked_rope_kernel, dim3(grid_of(M, N)), dim3(256), 0, stream, s, r, M, N, KE);
  const int rc = int4_gemm(x, packed, sz, y, s.xsum, sum_stride(M), nullptr, int4_gemm_shape(M, N, K, G, 0), M, N, K, groupsize, stream, s.flag, s.row_flag);
  if (rc != E2H_OK) return rc;
  hipLaunchKernelGGL(rope_flagged_rows_kernel, dim3(1024), dim3(256), 0, stream, y, s, r);
  return launch_status();
}

int int8_unpacked_rope(const uint16_t *x, const int8_t *q, const uint16_t *scales, const RopeRows &r, int K, uint16_t *w, hipStream_t stream) {
  const int N = (r.H + 2 * r.Hkv) * r.D, M = r.B * r.T;
  const int64_t pieces = static_cast<int64_t>(N) * K / 16;
  hipLaunchKernelGGL(unpack_int8_kernel, dim3(static_cast<unsigned>((pieces + 255) / 256)), dim3(256), 0, stream, q, w, pieces);
  const int64_t most = rows_at_once(K);
  for (int64_t m0 = 0; m0 < M; m0 += most) {
    const int rows = static_cast<int>(M - m0 < most ? M - m0 : most);
    hipLaunchKernelGGL(int8_unpacked_rope_kernel, dim3(grid_of(rows, N)), dim3(256), 0, stream, x + m0 * K, w, scales, r, static_cast<int>(m0), rows, N, K);
  }
  return launch_status();
}

}  // namespace e2h

extern "C" int64_t e2h_int8_mm_rope_kv_rows_scratch_bytes(int64_t batch, int64_t seqlen, int64_t n_head, int64_t n_kv_head, int64_t cache_len, int64_t head_dim, int64_t k) {
  return e2h::int8_unpacked_rope_bytes(batch, seqlen, n_head, n_kv_head, cache_len, head_dim, k);
}

extern "C" int e2h_int8_mm_rope_kv_rows(const uint16_t *x, const int8_t *q, const uint16_t *scales, const uint16_t *freqs_cis, int64_t freq_rows, uint16_t *q_out, uint16_t *k_cache,
                                        uint16_t *v_cache, const int64_t *input_pos, int64_t batch, int64_t seqlen, int64_t n_head, int64_t n_kv_head, int64_t cache_len,
                                        int64_t head_dim, int64_t k, int rows_by_token, void *scratch, int64_t scratch_bytes, void *stream) {
  using namespace e2h;
  if (!x || !q || !scales || !freqs_cis || !q_out || !k_cache || !v_cache || !input_pos || !scratch) return E2H_ERR_NULL_POINTER;
  const int64_t need = int8_unpacked_rope_bytes(batch, seqlen, n_head, n_kv_head, cache_len, head_dim, k);
  if (need == 0 || freq_rows < 1 || freq_rows > INT32_MAX / 2 / head_dim) return E2H_ERR_BAD_SHAPE;
  if (scratch_bytes < need) return E2H_ERR_SCRATCH_TOO_SMALL;
  if (!aligned16(x) || !aligned16(q) || !aligned16(scales) || !aligned16(freqs_cis) || !aligned16(q_out) || !aligned16(k_cache) || !aligned16(v_cache) || !aligned16(scratch) ||
      (reinterpret_cast<uintptr_t>(input_pos) & 7u))
    return E2H_ERR_MISALIGNED;
  const RopeRows r = {freqs_cis, q_out, k_cache, v_cache, input_pos, static_cast<int>(batch), static_cast<int>(seqlen), static_cast<int>(n_head), static_cast<int>(n_kv_head),
                      static_cast<int>(cache_len), static_cast<int>(head_dim), static_cast<int>(freq_rows), rows_by_token ? 1 : 0};
  return int8_unpacked_rope(x, q, scales, r, static_cast<int>(k), static_cast<uint16_t *>(scratch), static_cast<hipStream_t>(stream));
}

extern "C" int64_t e2h_int4_mm_rope_kv_rows_scratch_bytes(int64_t batch, int64_t seqlen, int64_t n_head, int64_t n_kv_head, int64_t cache_len, int64_t head_dim, int64_t k, int groupsize,
                                                          int inner_k_tiles) {
  return e2h::int4_unpacked_rope_bytes(batch, seqlen, n_head, n_kv_head, cache_len, head_dim, k, groupsize, inner_k_tiles);
}

extern "C" int e2h_int4_mm_rope_kv_rows(const uint16_t *x, const int32_t *packed, const uint16_t *scales_and_zeros, const uint16_t *freqs_cis, int64_t freq_rows, uint16_t *q_out,
                                        uint16_t *k_cache, uint16_t *v_cache, const int64_t *input_pos, int64_t batch, int64_t seqlen, int64_t n_head, int64_t n_kv_head,
                                        int64_t cache_len, int64_t head_dim, int64_t k, int groupsize, int inner_k_tiles, int rows_by_token, void *scratch, int64_t scratch_bytes,
                                        void *stream) {
  using namespace e2h;
  if (!x || !packed || !scales_and_zeros || !freqs_cis || !q_out || !k_cache || !v_cache || !input_pos || !scratch) return E2H_ERR_NULL_POINTER;
  const int64_t need = int4_unpacked_rope_bytes(batch, seqlen, n_head, n_kv_head, cache_len, head_dim, k, groupsize, inner_k_tiles);
  if (need == 0 || freq_rows < 1 || freq_rows > INT32_MAX / 2 / head_dim) return E2H_ERR_BAD_SHAPE;
  const int64_t n = (n_head + 2 * n_kv_head) * head_dim;
  if (n * k / 2 >= (int64_t{1} << 32) || (k / groupsize) * n * 4 >= (int64_t{1} << 32)) return E2H_ERR_BAD_SHAPE;
  if (scratch_bytes < need) return E2H_ERR_SCRATCH_TOO_SMALL;
  if (!aligned16(x) || !aligned16(packed) || !aligned16(scales_and_zeros) || !aligned16(freqs_cis) || !aligned16(q_out) || !aligned16(k_cache) || !aligned16(v_cache) ||
      !aligned16(scratch) || (reinterpret_cast<uintptr_t>(input_pos) & 7u))
    return E2H_ERR_MISALIGNED;
  const RopeRows r = {freqs_cis, q_out, k_cache, v_cache, input_pos, static_cast<int>(batch), static_cast<int>(seqlen), static_cast<int>(n_head), static_cast<int>(n_kv_head),
                      static_cast<int>(cache_len), static_cast<int>(head_dim), static_cast<int>(freq_rows), rows_by_token ? 1 : 0};
  return int4_unpacked_rope(x, packed, scales_and_zeros, r, static_cast<int>(k), groupsize, scratch, static_cast<hipStream_t>(stream));
}

extern "C" int64_t e2h_int8_mm_silu_gate_rows_scratch_bytes(int64_t m, int64_t n, int64_t k) {
  return m <= INT32_MAX ? e2h::int8_gate_unpacked_bytes(m, n, k) : 0;
}

extern "C" int e2h_int8_mm_silu_gate_rows(const uint16_t *x, const int8_t *q_gate, const uint16_t *scales_gate, const int8_t *q_up, const uint16_t *scales_up, uint16_t *y, int64_t m,
                                          int64_t n, int64_t k, void *scratch, int64_t scratch_bytes, void *stream) {
  using namespace e2h;
  if (!x || !q_gate || !scales_gate || !q_up || !scales_up || !y || !scratch) return E2H_ERR_NULL_POINTER;
  const int64_t need = e2h_int8_mm_silu_gate_rows_scratch_bytes(m, n, k);
  if (need == 0) return E2H_ERR_BAD_SHAPE;
  if (scratch_bytes < need) return E2H_ERR_SCRATCH_TOO_SMALL;
  if (!aligned16(x) || !aligned16(q_gate) || !aligned16(q_up) || !aligned16(scales_gate) || !aligned16(scales_up) || !aligned16(y) || !aligned16(scratch)) return E2H_ERR_MISALIGNED;
  return int8_unpacked_gate(x, q_gate, scales_gate, q_up, scales_up, y, static_cast<int>(m), static_cast<int>(n), static_cast<int>(k), static_cast<uint16_t *>(scratch),
                            static_cast<hipStream_t>(stream));
}

extern "C" int64_t e2h_int4_mm_scratch_bytes(int64_t m, int64_t n, int64_t k, int groupsize, int inner_k_tiles) {
  return e2h::int4_unpacked_bytes(m, n, k, groupsize, inner_k_tiles);
}

extern "C" int e2h_int4_mm_scratch(const uint16_t *x, const int32_t *packed, const uint16_t *scales_and_zeros, uint16_t *y, int64_t m, int64_t n, int64_t k, int groupsize,
                                   int inner_k_tiles, void *workspace, int64_t workspace_bytes, void *scratch, int64_t scratch_bytes, void *stream) {
  using namespace e2h;
  if (!x || !packed || !scales_and_zeros || !y) return E2H_ERR_NULL_POINTER;
  const int64_t need = int4_unpacked_bytes(m, n, k, groupsize, inner_k_tiles);
  if (!scratch || need == 0 || scratch_bytes < need || !aligned16(x) || !aligned16(packed) || !aligned16(scales_and_zeros) || !aligned16(y) || !aligned16(scratch) ||
      (workspace && !aligned16(workspace)) || n * k / 2 >= (int64_t{1} << 32) || (k / groupsize) * n * 4 >= (int64_t{1} << 32))
    return e2h_int4_mm(x, packed, scales_and_zeros, y, m, n, k, groupsize, inner_k_tiles, workspace, workspace_bytes, stream);
  return int4_unpacked_gemm(x, packed, scales_and_zeros, y, static_cast<int>(m), static_cast<int>(n), static_cast<int>(k), groupsize, scratch, static_cast<hipStream_t>(stream));
}

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
