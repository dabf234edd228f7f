// Quantization, packing and dequantization kernels (one pass over a weight matrix each; HBM-bound,
// run once per checkpoint or once per on-the-fly conversion).
//
// Bit-exactness contract: the int8 path is IEEE float32 (true division, round-half-even); the int4
// path reproduces torch's bfloat16 elementwise semantics, i.e. every op of the reference is computed
// in float32 and rounded to bfloat16 before the next op.  This file must be compiled without fast-math
// and without FMA contraction.
#include "e2h_common.h"

namespace e2h {
namespace {

// ------------------------------------------------------------------------------------------------
// int8 per-channel (reference models/quantize.py:39-71)
// ------------------------------------------------------------------------------------------------

template <bool BF16>
__device__ __forceinline__ float load_w(const void *w, size_t i) {
  if constexpr (BF16) {
    return bf16_to_f32(static_cast<const uint16_t *>(w)[i]);
  } else {
    return static_cast<const float *>(w)[i];
  }
}

// One code: rintf(w / scale), clamped.  The quotient from the reciprocal is a few units in the last place off, which matters only
// next to a rounding boundary n + 1/2; there (and for anything not finite) the true division decides.
__device__ __forceinline__ int int8_code(float w, float scale, float rcp) {
  float v = w * rcp;
  const float near = v - floorf(v) - 0.5f;
  if (!(fabsf(near) > 1e-3f)) v = w / scale;   // :66  true division
  return static_cast<int>(fminf(fmaxf(rintf(v), -128.f), 127.f));  // :67 half to even, :69
}

// One row per workgroup, bound by HBM.  VEC: eight values per load and lane (rows a multiple of eight values, 16-byte aligned); rows
// up to kHeld * 2048 values stay in registers between the two passes, which otherwise read the row again.
template <bool BF16, bool VEC>
__global__ __launch_bounds__(256) void int8_quantize_rows_kernel(const void *__restrict__ w, int8_t *__restrict__ q,
                                                                 float *__restrict__ scales_f32,
                                                                 uint16_t *__restrict__ scales_bf16, int64_t K) {
  constexpr int kHeld = 6;
  const int64_t row = blockIdx.x;
  const size_t base = static_cast<size_t>(row) * K;
  const auto load8 = [&](int64_t k, float (&v)[8]) {
    if constexpr (BF16) {
      const u32x4_t raw = *reinterpret_cast<const u32x4_t *>(static_cast<const uint16_t *>(w) + base + k);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        v[2 * i] = __builtin_bit_cast(float, raw[i] << 16);
        v[2 * i + 1] = __builtin_bit_cast(float, raw[i] & 0xFFFF0000u);
      }
    } else {
      const f32x4_t *p = reinterpret_cast<const f32x4_t *>(static_cast<const float *>(w) + base + k);
      const f32x4_t lo = p[0], hi = p[1];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        v[i] = lo[i];
        v[4 + i] = hi[i];
      }
    }
  };
  // max(-min(min_val, 0), max(max_val, 0)) == max |x| over the row  (:49-58)
  float amax = 0.f, held[kHeld][8];
  if constexpr (VEC) {
#pragma unroll
    for (int i = 0; i < kHeld; ++i) {
      const int64_t k = (i * 256 + threadIdx.x) * int64_t{8};
      if (k < K) load8(k, held[i]);
    }
#pragma unroll
    for (int i = 0; i < kHeld; ++i)
      if ((i * 256 + threadIdx.x) * int64_t{8} < K)
#pragma unroll
        for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(held[i][j]));
    for (int64_t k = (kHeld * 256 + threadIdx.x) * int64_t{8}; k < K; k += 2048) {
      float v[8];
      load8(k, v);
#pragma unroll
      for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(v[j]));
    }
  } else {
    for (int64_t k = threadIdx.x; k < K; k += blockDim.x) amax = fmaxf(amax, fabsf(load_w<BF16>(w, base + k)));
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off));
  __shared__ float wave_max[4];
  if ((threadIdx.x & 63) == 0) wave_max[threadIdx.x >> 6] = amax;
  __syncthreads();
  amax = fmaxf(fmaxf(wave_max[0], wave_max[1]), fmaxf(wave_max[2], wave_max[3]));
  float scale = amax / 127.5f;             // :59  float(quant_max - quant_min) / 2
  scale = fmaxf(scale, 1.1920928955078125e-07f);  // :61  clamp(min=float32 eps)
  if (threadIdx.x == 0) {
    if (scales_f32) scales_f32[row] = scale;
    if (scales_bf16) scales_bf16[row] = f32_to_bf16_rne(scale);
  }
  const float rcp = __builtin_amdgcn_rcpf(scale);
  if constexpr (VEC) {
    const auto store8 = [&](int64_t k, const float (&v)[8]) {
      u32x2_t o = {0u, 0u};
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j >> 2] |= (static_cast<uint32_t>(int8_code(v[j], scale, rcp)) & 255u) << (8 * (j & 3));
      *reinterpret_cast<u32x2_t *>(q + base + k) = o;
    };
#pragma unroll
    for (int i = 0; i < kHeld; ++i) {
      const int64_t k = (i * 256 + threadIdx.x) * int64_t{8};
      if (k < K) store8(k, held[i]);
    }
    for (int64_t k = (kHeld * 256 + threadIdx.x) * int64_t{8}; k < K; k += 2048) {
      float v[8];
      load8(k, v);
      store8(k, v);
    }
  } else {
    for (int64_t k = threadIdx.x; k < K; k += blockDim.x) q[base + k] = static_cast<int8_t>(int8_code(load_w<BF16>(w, base + k), scale, rcp));
  }
}

// ------------------------------------------------------------------------------------------------
// int4 group-wise (reference models/quantize.py:74-92, :118-144), bfloat16 arithmetic
// ------------------------------------------------------------------------------------------------

struct GroupQParams {
  float scale, zero;  // bfloat16-exact values
};

__device__ __forceinline__ GroupQParams qparams_from_minmax(float mn, float mx) {
  float r = bf16_round(mx - mn);                  // :88  max_val - min_val
  r = fmaxf(r, bf16_to_f32(0x3586));              // :88  .clamp(min=1e-6); bfloat16(1e-6) = 0x3586
  const float scale = bf16_round(r / 15.0f);      // :88  / max_int
  const float half = bf16_round(scale * 8.0f);    // :89  scales * 2**(n_bit-1)
  const float zero = bf16_round(mn + half);       // :89
  return {scale, zero};
}

__device__ __forceinline__ int quantize_one(float w, float scale, float min_val) {
  float t = bf16_round(w - min_val);  // :136 .sub(min_val)
  t = bf16_round(t / scale);          // :137 .div(scales)
  t = rintf(t);                       // :138 .round()
  t = fminf(fmaxf(t, 0.f), 15.f);     // :139 .clamp_(0, 15)
  return static_cast<int>(t);
}

__device__ __forceinline__ float requant_min(float scale, float zero) {
  return bf16_round(zero - bf16_round(scale * 8.0f));  // :132
}

enum : int { kModeQParams = 0, kModeCodes = 1, kModeFromQParams = 2 };

// One lane handles 8 consecutive k (one 16-byte load); a group is G/8 adjacent lanes of a wave.
// MODE kModeQParams:     writes scales/zeros [N][K/G].
// MODE kModeCodes:       writes codes [N][K] int32 and scales_and_zeros [K/G][N][2].
// MODE kModeFromQParams: reads scales/zeros [N][K/G], writes codes.
template <int G, int MODE>
__global__ __launch_bounds__(256) void int4_group_kernel(const uint16_t *__restrict__ w, uint16_t *__restrict__ scales,
                                                         uint16_t *__restrict__ zeros, int32_t *__restrict__ codes,
                                                         uint16_t *__restrict__ sz, int64_t N, int64_t K) {
  constexpr int LPG = G / 8;
  const int64_t total8 = N * K / 8;
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const bool live = idx < total8;
  const int64_t e0 = (live ? idx : total8 - 1) * 8;
  const int64_t n = e0 / K;
  const int64_t k = e0 - n * K;
  const int64_t groups_per_row = K / G;
  const int64_t g = k / G;

  const u32x4_t raw = *reinterpret_cast<const u32x4_t *>(w + e0);
  float v[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[2 * i] = __builtin_bit_cast(float, raw[i] << 16);
    v[2 * i + 1] = __builtin_bit_cast(float, raw[i] & 0xFFFF0000u);
  }
  float scale, zero;
  if constexpr (MODE == kModeFromQParams) {
    scale = bf16_to_f32(scales[n * groups_per_row + g]);
    zero = bf16_to_f32(zeros[n * groups_per_row + g]);
  } else {
    float mn = v[0], mx = v[0];
#pragma unroll
    for (int i = 1; i < 8; ++i) {
      mn = fminf(mn, v[i]);
      mx = fmaxf(mx, v[i]);
    }
#pragma unroll
    for (int off = 1; off < LPG; off <<= 1) {
      mn = fminf(mn, __shfl_xor(mn, off));
      mx = fmaxf(mx, __shfl_xor(mx, off));
    }
    const GroupQParams qp = qparams_from_minmax(mn, mx);
    scale = qp.scale;
    zero = qp.zero;
  }
  if (!live) return;
  if constexpr (MODE == kModeQParams) {
    if ((k % G) == 0) {
      scales[n * groups_per_row + g] = f32_to_bf16_rne(scale);
      zeros[n * groups_per_row + g] = f32_to_bf16_rne(zero);
    }
  } else {
    const float min_val = requant_min(scale, zero);
    int32_t out[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) out[i] = quantize_one(v[i], scale, min_val);
    int4 *dst = reinterpret_cast<int4 *>(codes + e0);
    dst[0] = make_int4(out[0], out[1], out[2], out[3]);
    dst[1] = make_int4(out[4], out[5], out[6], out[7]);
    if constexpr (MODE == kModeCodes) {
      if ((k % G) == 0) {
        const uint32_t pair = static_cast<uint32_t>(f32_to_bf16_rne(scale)) | (static_cast<uint32_t>(f32_to_bf16_rne(zero)) << 16);
        reinterpret_cast<uint32_t *>(sz)[g * N + n] = pair;  // [K/G][N][2]
      }
    }
  }
}

// Generic group size (any g >= 2 dividing K): one thread per group, serial over the group.
template <int MODE>
__global__ __launch_bounds__(256) void int4_group_generic_kernel(const uint16_t *__restrict__ w, uint16_t *__restrict__ scales,
                                                                 uint16_t *__restrict__ zeros, int32_t *__restrict__ codes,
                                                                 uint16_t *__restrict__ sz, int64_t N, int64_t K, int G) {
  const int64_t groups_per_row = K / G;
  const int64_t gid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (gid >= N * groups_per_row) return;
  const int64_t n = gid / groups_per_row, g = gid - n * groups_per_row;
  const uint16_t *src = w + n * K + g * G;
  float scale, zero;
  if constexpr (MODE == kModeFromQParams) {
    scale = bf16_to_f32(scales[gid]);
    zero = bf16_to_f32(zeros[gid]);
  } else {
    float mn = bf16_to_f32(src[0]), mx = mn;
    for (int i = 1; i < G; ++i) {
      const float v = bf16_to_f32(src[i]);
      mn = fminf(mn, v);
      mx = fmaxf(mx, v);
    }
    const GroupQParams qp = qparams_from_minmax(mn, mx);
    scale = qp.scale;
    zero = qp.zero;
  }
  if constexpr (MODE == kModeQParams) {
    scales[gid] = f32_to_bf16_rne(scale);
    zeros[gid] = f32_to_bf16_rne(zero);
  } else {
    const float min_val = requant_min(scale, zero);
    for (int i = 0; i < G; ++i) codes[n * K + g * G + i] = quantize_one(bf16_to_f32(src[i]), scale, min_val);
    if constexpr (MODE == kModeCodes) {
      const uint32_t pair = static_cast<uint32_t>(f32_to_bf16_rne(scale)) | (static_cast<uint32_t>(f32_to_bf16_rne(zero)) << 16);
      reinterpret_cast<uint32_t *>(sz)[g * N + n] = pair;
    }
  }
}

// ------------------------------------------------------------------------------------------------
// tile packing (torch.ops.aten._convert_weight_to_int4pack, PyTorch 2.2.0 CUDA nibble order)
// ------------------------------------------------------------------------------------------------

// k offsets (relative to the 32-wide span of a packed word) of nibbles 0..7 for j = t % 4
__device__ __forceinline__ int nibble_k(int i, int j) {
  // nibble i holds v[s], s = {0,2,4,6,1,3,5,7}[i]; v[s] sits at 16*(s>>2) + 8*((s>>1)&1) + (s&1) + 2j
  const int s = (i < 4) ? 2 * i : 2 * (i - 4) + 1;
  return 16 * (s >> 2) + 8 * ((s >> 1) & 1) + (s & 1) + 2 * j;
}

// word index -> (row n, first k of its 32-wide span, j)
struct WordCoord {
  int64_t n, k0;
  int j;
};

__device__ __forceinline__ WordCoord word_coord(int64_t widx, int64_t K, int ikt) {
  const int words = ikt / 2;
  const int64_t kt = K / (16 * ikt);
  const int p = static_cast<int>(widx % words);
  int64_t r = widx / words;
  const int t = static_cast<int>(r % 32);
  r /= 32;
  const int64_t k_outer = r % kt;
  const int64_t n_tile = r / kt;
  return {n_tile * 8 + (t >> 2), (k_outer * ikt + 2 * p) * 16, t & 3};
}

__global__ __launch_bounds__(256) void int4_pack_kernel(const int32_t *__restrict__ codes, uint32_t *__restrict__ packed,
                                                        int64_t N, int64_t K, int ikt) {
  const int64_t widx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (widx >= N * K / 8) return;
  const WordCoord wc = word_coord(widx, K, ikt);
  const int32_t *row = codes + wc.n * K + wc.k0;
  uint32_t word = 0;
#pragma unroll
  for (int i = 0; i < 8; ++i) word |= (static_cast<uint32_t>(row[nibble_k(i, wc.j)]) & 15u) << (4 * i);
  packed[widx] = word;
}

__global__ __launch_bounds__(256) void int4_unpack_kernel(const uint32_t *__restrict__ packed, int32_t *__restrict__ codes,
                                                          int64_t N, int64_t K, int ikt) {
  const int64_t widx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (widx >= N * K / 8) return;
  const WordCoord wc = word_coord(widx, K, ikt);
  int32_t *row = codes + wc.n * K + wc.k0;
  const uint32_t word = packed[widx];
#pragma unroll
  for (int i = 0; i < 8; ++i) row[nibble_k(i, wc.j)] = static_cast<int32_t>((word >> (4 * i)) & 15u);
}

// group_dequantize_tensor_from_qparams (:154-171) on the packed weight: bf16(bf16((q-8)*s) + z)
__global__ __launch_bounds__(256) void int4_dequantize_kernel(const uint32_t *__restrict__ packed, const uint16_t *__restrict__ sz,
                                                              uint16_t *__restrict__ w_out, int64_t N, int64_t K, int G, int ikt) {
  const int64_t widx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (widx >= N * K / 8) return;
  const WordCoord wc = word_coord(widx, K, ikt);
  const uint32_t word = packed[widx];
  const int64_t g = wc.k0 / G;  // a 32-wide span never straddles a group (G >= 32)
  const float scale = bf16_to_f32(sz[(g * N + wc.n) * 2]);
  const float zero = bf16_to_f32(sz[(g * N + wc.n) * 2 + 1]);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float qv = static_cast<float>(static_cast<int>((word >> (4 * i)) & 15u) - 8);
    const float t = bf16_round(qv * scale);
    w_out[wc.n * K + wc.k0 + nibble_k(i, wc.j)] = f32_to_bf16_rne(t + zero);
  }
}


// group_dequantize_tensor_from_qparams (:154-171) on plain int32 codes [N][K] with qparams [N][K/G]
__global__ __launch_bounds__(256) void int4_dequantize_codes_kernel(const int32_t *__restrict__ codes, const uint16_t *__restrict__ scales,
                                                                    const uint16_t *__restrict__ zeros, uint16_t *__restrict__ w_out,
                                                                    int64_t N, int64_t K, int G) {
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (idx >= N * K) return;
  const int64_t n = idx / K, k = idx - n * K;
  const int64_t gi = n * (K / G) + k / G;
  const float t = bf16_round(static_cast<float>(codes[idx] - 8) * bf16_to_f32(scales[gi]));  // :169 .sub(8).mul(scales)
  w_out[idx] = f32_to_bf16_rne(t + bf16_to_f32(zeros[gi]));                                   // :169 .add(zeros)
}

// ---- fused quantize + pack ----------------------------------------------------------------------------
// Lane layout as int4_group_kernel (8 consecutive k per lane, 32 lanes per row, a workgroup 8 rows x 256 k).  Four neighbouring
// lanes hold the 32 codes of four packed words: word j takes from lane h of the quad code 2 j as nibble h and code 2 j + 1 as
// nibble 4 + h, so the words form by two ORs across the quad, without LDS, and lane j stores word j.

__device__ __forceinline__ float float_of(uint32_t u) { return __builtin_bit_cast(float, u); }

// nearest bfloat16 by the conversion instruction (no NaN here), as float32
__device__ __forceinline__ float to_bf16(float v) {
  return float_of(static_cast<uint32_t>(__builtin_bit_cast(uint16_t, static_cast<__bf16>(v))) << 16);
}

// value of the lane whose number differs by XOR (1, 2: any; 7, 15: within its row of 16)
template <int XOR>
__device__ __forceinline__ uint32_t lane_xor(uint32_t v) {
  constexpr int kCtrl = XOR == 1 ? 0xB1 : XOR == 2 ? 0x4E : XOR == 7 ? 0x141 : 0x140;  // quad_perm, row_half_mirror, row_mirror
  return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), kCtrl, 0xF, 0xF, true));
}

// minimum and maximum over LPG neighbouring lanes
template <int LPG>
__device__ __forceinline__ void group_minmax(float &mn, float &mx) {
  const auto step = [&](auto other) {
    const float a = float_of(other(__builtin_bit_cast(uint32_t, mn))), b = float_of(other(__builtin_bit_cast(uint32_t, mx)));
    mn = fminf(mn, a);
    mx = fmaxf(mx, b);
  };
  step([](uint32_t v) { return lane_xor<1>(v); });
  step([](uint32_t v) { return lane_xor<2>(v); });
  if constexpr (LPG >= 8) step([](uint32_t v) { return lane_xor<7>(v); });    // a quad's lanes agree by now
  if constexpr (LPG >= 16) step([](uint32_t v) { return lane_xor<15>(v); });  // so do eight
  if constexpr (LPG >= 32) step([](uint32_t v) { return static_cast<uint32_t>(__shfl_xor(static_cast<int>(v), 16)); });
}

// quantize_one for two values at once and a finite scale >= 1e-6 / 15.  w - min_val and the scale are bfloat16 values, so their quotient
// Q is exactly a rounding boundary (of bfloat16, or of the integers) or a relative 2^-17 away from one.  q0 = a rcp(s) is within 2^-22 of
// Q, its residual e = a - q0 s is exact in float32, and q0 + e rcp(s) is Q to 2^-45 before its one rounding: on a boundary it is
// that value, elsewhere on Q's side.  Adding 1.5 * 2^23 rounds to the integer, ties to even, and leaves it in the low bits.
__device__ __forceinline__ void quantize_two(float w0, float w1, float scale, float rcp, float min_val, uint32_t &c0, uint32_t &c1) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  const uint32_t a = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{w0 - min_val, w1 - min_val}, bf16x2));
  const float a0 = float_of(a << 16), a1 = float_of(a & 0xFFFF0000u);
  const float q0 = a0 * rcp, q1 = a1 * rcp;
  const float r0 = __builtin_fmaf(__builtin_fmaf(-q0, scale, a0), rcp, q0), r1 = __builtin_fmaf(__builtin_fmaf(-q1, scale, a1), rcp, q1);
  const uint32_t t = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{r0, r1}, bf16x2));
  c0 = __builtin_bit_cast(uint32_t, fminf(fmaxf(float_of(t << 16), 0.f), 15.f) + 12582912.f) & 15u;
  c1 = __builtin_bit_cast(uint32_t, fminf(fmaxf(float_of(t & 0xFFFF0000u), 0.f), 15.f) + 12582912.f) & 15u;
}

// U: spans of 256 k per workgroup, all loaded before the first is worked on.  The bound is HBM once a weight costs about 20 vector
// instructions: 11008 x 4096 at g128 (112 MB in and out) takes 31 us, 3.6 TB/s beside 4.8 for a large copy.  With IEEE divisions (ten
// instructions each), software rounding with its NaN branch, shuffles through LDS and 64-bit index divisions it took 67 us.
// U = 2 measured 30.7 us, 1: 31.5, 4: 31.8, 8: 33.5.
template <int G, int U>
__global__ __launch_bounds__(256) void int4_quantize_pack_kernel(const uint16_t *__restrict__ w, uint32_t *__restrict__ packed,
                                                                 uint16_t *__restrict__ sz, int64_t N, int64_t K, unsigned spans, int ikt_log2) {
  constexpr int LPG = G / 8;
  constexpr int SPAN = 256;
  const unsigned n_tile = blockIdx.x / spans, span0 = (blockIdx.x - n_tile * spans) * U;
  const int r = threadIdx.x >> 5;         // row within the tile
  const int kl = (threadIdx.x & 31) * 8;  // k within a span
  const int h = threadIdx.x & 3;
  const int64_t n = static_cast<int64_t>(n_tile) * 8 + r;
  const int64_t k0 = static_cast<int64_t>(span0) * SPAN;
  const uint16_t *const src = w + n * K + k0 + kl;
  u32x4_t raw[U];
#pragma unroll
  for (int u = 0; u < U; ++u) raw[u] = *reinterpret_cast<const u32x4_t *>(src + u * SPAN);
  // word (row, h) of the 32-wide piece p of k block k_outer sits at ((n_tile * k blocks + k_outer) * 32 + 4 r + h) * ikt / 2 + p
  const int kblk_log2 = ikt_log2 + 4, words_log2 = ikt_log2 - 1;
  uint32_t *const dst = packed + (((static_cast<int64_t>(n_tile) * (K >> kblk_log2) + (k0 >> kblk_log2) + (kl >> kblk_log2)) * 32 + 4 * r + h) << words_log2) +
                        ((kl >> 5) & ((1 << words_log2) - 1));
  uint32_t *const sz_dst = reinterpret_cast<uint32_t *>(sz) + ((k0 + kl) / G) * N + n;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    float v[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = float_of(raw[u][i] << 16);
      v[2 * i + 1] = float_of(raw[u][i] & 0xFFFF0000u);
    }
    float mn = v[0], mx = v[0];
#pragma unroll
    for (int i = 1; i < 8; ++i) {
      mn = fminf(mn, v[i]);
      mx = fmaxf(mx, v[i]);
    }
    group_minmax<LPG>(mn, mx);
    uint32_t c[8], pair;
    if (__builtin_expect(mx - mn < 1e37f, 1)) {
      // qparams_from_minmax and requant_min, the division by 15 as quantize_two divides; scale * 8 is exact
      const float range = fmaxf(to_bf16(mx - mn), bf16_to_f32(0x3586));
      const float over = range * (1.0f / 15.0f);
      const float scale = to_bf16(__builtin_fmaf(__builtin_fmaf(-over, 15.0f, range), 1.0f / 15.0f, over));
      const float zero = to_bf16(mn + scale * 8.0f), min_val = to_bf16(zero - scale * 8.0f), rcp = __builtin_amdgcn_rcpf(scale);
      pair = __builtin_bit_cast(uint32_t, scale) >> 16 | __builtin_bit_cast(uint32_t, zero);
#pragma unroll
      for (int i = 0; i < 4; ++i) quantize_two(v[2 * i], v[2 * i + 1], scale, rcp, min_val, c[2 * i], c[2 * i + 1]);
    } else {  // infinities or nearly so
      const GroupQParams qp = qparams_from_minmax(mn, mx);
      const float min_val = requant_min(qp.scale, qp.zero);
      pair = static_cast<uint32_t>(f32_to_bf16_rne(qp.scale)) | (static_cast<uint32_t>(f32_to_bf16_rne(qp.zero)) << 16);
#pragma unroll
      for (int i = 0; i < 8; ++i) c[i] = static_cast<uint32_t>(quantize_one(v[i], qp.scale, min_val));
    }
    if ((kl % G) == 0) sz_dst[u * (SPAN / G) * N] = pair;
    uint32_t word = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint32_t t = (c[2 * j] | c[2 * j + 1] << 16) << (4 * h);
      t |= lane_xor<1>(t);
      t |= lane_xor<2>(t);
      word = h == j ? t : word;
    }
    dst[u * SPAN] = word;  // a span of 8 rows is 256 words
  }
}

template <int G>
void launch_quantize_pack(const uint16_t *w, uint32_t *packed, uint16_t *sz, int64_t n, int64_t k, int ikt, hipStream_t s) {
  const unsigned spans = static_cast<unsigned>(k / 256);
  const int ikt_log2 = ikt == 8 ? 3 : ikt == 4 ? 2 : 1;
  const unsigned tiles = static_cast<unsigned>(n / 8);
  if (spans % 2 == 0)
    hipLaunchKernelGGL((int4_quantize_pack_kernel<G, 2>), dim3(tiles * (spans / 2)), dim3(256), 0, s, w, packed, sz, n, k, spans / 2, ikt_log2);
  else
    hipLaunchKernelGGL((int4_quantize_pack_kernel<G, 1>), dim3(tiles * spans), dim3(256), 0, s, w, packed, sz, n, k, spans, ikt_log2);
}

inline unsigned blocks_for(int64_t items, int per_block) { return static_cast<unsigned>((items + per_block - 1) / per_block); }

int check_int4_quant_args(const void *w, int64_t n, int64_t k, int g) {
  if (!w) return E2H_ERR_NULL_POINTER;
  if (n < 1 || k < 1 || n * k > (int64_t{1} << 40)) return E2H_ERR_BAD_SHAPE;
  if (g < 2 || k % g != 0) return E2H_ERR_BAD_GROUPSIZE;
  return E2H_OK;
}

bool fast_group(int g) { return g == 32 || g == 64 || g == 128 || g == 256; }

template <int MODE>
int launch_group_kernel(const uint16_t *w, uint16_t *scales, uint16_t *zeros, int32_t *codes, uint16_t *sz, int64_t n,
                        int64_t k, int g, hipStream_t s) {
  if (fast_group(g) && aligned16(w) && (MODE == kModeQParams || aligned16(codes))) {
    const unsigned blocks = blocks_for(n * k / 8, 256);
    switch (g) {
      case 32: hipLaunchKernelGGL((int4_group_kernel<32, MODE>), dim3(blocks), dim3(256), 0, s, w, scales, zeros, codes, sz, n, k); break;
      case 64: hipLaunchKernelGGL((int4_group_kernel<64, MODE>), dim3(blocks), dim3(256), 0, s, w, scales, zeros, codes, sz, n, k); break;
      case 128: hipLaunchKernelGGL((int4_group_kernel<128, MODE>), dim3(blocks), dim3(256), 0, s, w, scales, zeros, codes, sz, n, k); break;
      default: hipLaunchKernelGGL((int4_group_kernel<256, MODE>), dim3(blocks), dim3(256), 0, s, w, scales, zeros, codes, sz, n, k); break;
    }
  } else {
    const unsigned blocks = blocks_for(n * (k / g), 256);
    hipLaunchKernelGGL((int4_group_generic_kernel<MODE>), dim3(blocks), dim3(256), 0, s, w, scales, zeros, codes, sz, n, k, g);
  }
  return launch_status();
}

}  // namespace
}  // namespace e2h

using namespace e2h;

extern "C" int e2h_int8_quantize_per_channel(const void *w, int w_is_bf16, int8_t *q, float *scales_f32,
                                             uint16_t *scales_bf16, int64_t n, int64_t k, void *stream) {
  if (!w || !q) return E2H_ERR_NULL_POINTER;
  if (n < 1 || k < 1 || n > INT32_MAX) return E2H_ERR_BAD_SHAPE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool vec = (k % 8) == 0 && aligned16(w) && (reinterpret_cast<uintptr_t>(q) & 7u) == 0;
  const auto kernel = w_is_bf16 ? (vec ? int8_quantize_rows_kernel<true, true> : int8_quantize_rows_kernel<true, false>)
                                : (vec ? int8_quantize_rows_kernel<false, true> : int8_quantize_rows_kernel<false, false>);
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(n)), dim3(256), 0, s, w, q, scales_f32, scales_bf16, k);
  return launch_status();
}

extern "C" int e2h_int4_group_qparams(const uint16_t *w, uint16_t *scales, uint16_t *zeros, int64_t n, int64_t k,
                                      int groupsize, void *stream) {
  if (int rc = check_int4_quant_args(w, n, k, groupsize)) return rc;
  if (!scales || !zeros) return E2H_ERR_NULL_POINTER;
  return launch_group_kernel<kModeQParams>(w, scales, zeros, nullptr, nullptr, n, k, groupsize, static_cast<hipStream_t>(stream));
}

extern "C" int e2h_int4_quantize_from_qparams(const uint16_t *w, const uint16_t *scales, const uint16_t *zeros,
                                              int32_t *codes, int64_t n, int64_t k, int groupsize, void *stream) {
  if (int rc = check_int4_quant_args(w, n, k, groupsize)) return rc;
  if (!scales || !zeros || !codes) return E2H_ERR_NULL_POINTER;
  return launch_group_kernel<kModeFromQParams>(w, const_cast<uint16_t *>(scales), const_cast<uint16_t *>(zeros), codes, nullptr, n, k,
                                               groupsize, static_cast<hipStream_t>(stream));
}

extern "C" int e2h_int4_group_quantize(const uint16_t *w, int32_t *codes, uint16_t *scales_and_zeros, int64_t n,
                                       int64_t k, int groupsize, void *stream) {
  if (int rc = check_int4_quant_args(w, n, k, groupsize)) return rc;
  if (!codes || !scales_and_zeros) return E2H_ERR_NULL_POINTER;
  if (reinterpret_cast<uintptr_t>(scales_and_zeros) & 3u) return E2H_ERR_MISALIGNED;
  return launch_group_kernel<kModeCodes>(w, nullptr, nullptr, codes, scales_and_zeros, n, k, groupsize, static_cast<hipStream_t>(stream));
}

static int check_pack_args(const void *a, const void *b, int64_t n, int64_t k, int ikt) {
  if (!a || !b) return E2H_ERR_NULL_POINTER;
  if (ikt != 2 && ikt != 4 && ikt != 8) return E2H_ERR_BAD_INNER_K_TILES;
  if (n < 8 || k < 1 || (n % 8) != 0 || n * k > (int64_t{1} << 40)) return E2H_ERR_BAD_SHAPE;
  if (k % (16 * ikt) != 0) return E2H_ERR_BAD_INNER_K_TILES;
  return E2H_OK;
}

extern "C" int e2h_int4_pack(const int32_t *codes, int32_t *packed, int64_t n, int64_t k, int inner_k_tiles, void *stream) {
  if (int rc = check_pack_args(codes, packed, n, k, inner_k_tiles)) return rc;
  hipLaunchKernelGGL(int4_pack_kernel, dim3(blocks_for(n * k / 8, 256)), dim3(256), 0, static_cast<hipStream_t>(stream), codes,
                     reinterpret_cast<uint32_t *>(packed), n, k, inner_k_tiles);
  return launch_status();
}

extern "C" int e2h_int4_unpack(const int32_t *packed, int32_t *codes, int64_t n, int64_t k, int inner_k_tiles, void *stream) {
  if (int rc = check_pack_args(packed, codes, n, k, inner_k_tiles)) return rc;
  hipLaunchKernelGGL(int4_unpack_kernel, dim3(blocks_for(n * k / 8, 256)), dim3(256), 0, static_cast<hipStream_t>(stream),
                     reinterpret_cast<const uint32_t *>(packed), codes, n, k, inner_k_tiles);
  return launch_status();
}

extern "C" int e2h_int4_dequantize(const int32_t *packed, const uint16_t *scales_and_zeros, uint16_t *w_out, int64_t n,
                                   int64_t k, int groupsize, int inner_k_tiles, void *stream) {
  if (int rc = check_pack_args(packed, w_out, n, k, inner_k_tiles)) return rc;
  if (!scales_and_zeros) return E2H_ERR_NULL_POINTER;
  if (!fast_group(groupsize) || k % groupsize != 0) return E2H_ERR_BAD_GROUPSIZE;
  hipLaunchKernelGGL(int4_dequantize_kernel, dim3(blocks_for(n * k / 8, 256)), dim3(256), 0, static_cast<hipStream_t>(stream),
                     reinterpret_cast<const uint32_t *>(packed), scales_and_zeros, w_out, n, k, groupsize, inner_k_tiles);
  return launch_status();
}

extern "C" int e2h_int4_dequantize_codes(const int32_t *codes, const uint16_t *scales, const uint16_t *zeros, uint16_t *w_out,
                                         int64_t n, int64_t k, int groupsize, void *stream) {
  if (!codes || !scales || !zeros || !w_out) return E2H_ERR_NULL_POINTER;
  if (n < 1 || k < 1 || n * k > (int64_t{1} << 40)) return E2H_ERR_BAD_SHAPE;
  if (groupsize < 2 || k % groupsize != 0) return E2H_ERR_BAD_GROUPSIZE;
  hipLaunchKernelGGL(int4_dequantize_codes_kernel, dim3(blocks_for(n * k, 256)), dim3(256), 0, static_cast<hipStream_t>(stream), codes,
                     scales, zeros, w_out, n, k, groupsize);
  return launch_status();
}

extern "C" int e2h_int4_quantize_pack(const uint16_t *w, int32_t *packed, uint16_t *scales_and_zeros, int64_t n, int64_t k,
                                      int groupsize, int inner_k_tiles, void *stream) {
  if (int rc = check_pack_args(w, packed, n, k, inner_k_tiles)) return rc;
  if (!scales_and_zeros) return E2H_ERR_NULL_POINTER;
  if (!fast_group(groupsize) || k % groupsize != 0) return E2H_ERR_BAD_GROUPSIZE;
  if (!aligned16(w) || (reinterpret_cast<uintptr_t>(scales_and_zeros) & 3u) || (reinterpret_cast<uintptr_t>(packed) & 3u))
    return E2H_ERR_MISALIGNED;
  if (k % 256 != 0) return E2H_ERR_BAD_SHAPE;  // callers fall back to quantize + pack
  hipStream_t s = static_cast<hipStream_t>(stream);
  uint32_t *out = reinterpret_cast<uint32_t *>(packed);
  switch (groupsize) {
    case 32: launch_quantize_pack<32>(w, out, scales_and_zeros, n, k, inner_k_tiles, s); break;
    case 64: launch_quantize_pack<64>(w, out, scales_and_zeros, n, k, inner_k_tiles, s); break;
    case 128: launch_quantize_pack<128>(w, out, scales_and_zeros, n, k, inner_k_tiles, s); break;
    default: launch_quantize_pack<256>(w, out, scales_and_zeros, n, k, inner_k_tiles, s); break;
  }
  return launch_status();
}
