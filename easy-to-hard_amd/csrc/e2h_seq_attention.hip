// Windowed softmax attention with kept first tokens over a per-sequence key/value cache (e2h_seq_window_attention).
//
// A query at position i sees the keys first .. min(i, first + keep_first - 1) and max(first, i - window + 1) .. i.  The keys a
// group of queries needs are walked as one list: the kept ones first, then the window, so both ends cost only what they hold.
//
// bfloat16: both products on v_mfma_f32_16x16x32_bf16 in transposed form.  S^T = K Q^T puts one query into each lane column
// (lane 16 b + c holds keys 4 b .. 4 b + 3 of query c), so the softmax statistics of a query are in-lane sums plus two
// shuffles, and the weights are, without moving, the B operand of O^T = V^T P^T over a key order that the V operand follows.
// Weights enter that product as two bfloat16 terms (value and remainder), which keeps them at float32 accuracy against
// bfloat16 values.
// float32: one wave per query and head on the vector units.
//
// Norm and rotation of a query happen where a kernel loads it (a lane of the matrix kernels holds 8 neighbouring dimensions, so the
// rotated pairs are in-lane and a head's sum of squares is two shuffles); those of a key where it is appended.  A sink joins the
// softmax sum at the end.
#include "e2h_attention_tiles.h"
#include "e2h_seq_common.h"

namespace e2h {
namespace {

constexpr float kMasked = -1e30f;

struct KeyList {  // virtual index n -> key position
  int first, kept, start, count;
  __device__ int at(int n) const { return n < kept ? first + n : start + (n - kept); }
};

// keys of the queries at positions pa .. pb of one sequence
__device__ __forceinline__ KeyList key_list(int pa, int pb, int first, int window, int keep_first) {
  KeyList k;
  k.first = first;
  if (pb < first) {
    k.kept = k.count = 0;
    k.start = first;
    return k;
  }
  const int live = pb - first + 1;
  k.kept = keep_first < live ? keep_first : live;
  k.start = pa - window + 1;  // window > 0: no overflow
  if (k.start < first + k.kept) k.start = first + k.kept;
  k.count = k.kept + (k.start <= pb ? pb - k.start + 1 : 0);
  return k;
}

// window and keep_first fit 31 bits here, window 0 has become the largest value
__device__ __forceinline__ bool sees(int i, int j, int first, int window, int keep_first) {
  return j <= i && j >= first && (i - j < window || j - first < keep_first);
}

// eight consecutive bfloat16 values starting at p, of which `valid` exist; VEC: 16-byte accesses are aligned and valid is 8 or <= 0
template <bool VEC>
__device__ __forceinline__ u32x4_t load8(const bf16_t *p, int valid) {
  u32x4_t r = {0u, 0u, 0u, 0u};
  if (VEC) {
    if (valid > 0) r = *reinterpret_cast<const u32x4_t *>(p);
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (i < valid) r[i >> 1] |= static_cast<uint32_t>(p[i]) << (16 * (i & 1));
  }
  return r;
}

__device__ __forceinline__ u32x4_t add_bias8(u32x4_t r, const float *bias, int valid) {
  if (!bias) return r;
  u32x4_t o = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    if (i < valid) {
      const float v = __builtin_bit_cast(float, (i & 1) ? (r[i >> 1] & 0xFFFF0000u) : (r[i >> 1] << 16)) + bias[i];
      o[i >> 1] |= static_cast<uint32_t>(f32_to_bf16_rne(v)) << (16 * (i & 1));
    }
  }
  return o;
}

// eight consecutive values of either type as float32, zero beyond `valid`
template <typename T, bool VEC>
__device__ __forceinline__ void load8_f32(const T *p, int valid, float (&v)[8]) {
  if (VEC) {
    f32x4_t lo = {0.f, 0.f, 0.f, 0.f}, hi = lo;
    if (valid > 0) {
      lo = load4(p);
      hi = load4(p + 4);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[i] = lo[i];
      v[4 + i] = hi[i];
    }
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = i < valid ? to_f32(p[i]) : 0.f;
  }
}

template <typename T, bool VEC>
__device__ __forceinline__ void store8_f32(T *p, int valid, const float (&v)[8]) {
  if (VEC) {
    if (valid > 0) {
      store4(p, f32x4_t{v[0], v[1], v[2], v[3]});
      store4(p + 4, f32x4_t{v[4], v[5], v[6], v[7]});
    }
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (i < valid) p[i] = from_f32<T>(v[i]);
  }
}

__device__ __forceinline__ float square_sum8(const float (&v)[8]) {
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) s = __builtin_fmaf(v[i], v[i], s);
  return s;
}

// What norm and rotation do to dimensions d .. d + 7 (d a multiple of 8) of a head, loaded before the norm's sum is known.  VEC: the
// norm's weights are aligned and valid is 8 or <= 0.
struct NormRotate8 {
  float weight[8], turn[8];  // turn: (cos, sin) of four pairs
  bool normed;

  template <bool VEC>
  __device__ __forceinline__ void load(int d, int valid, const float *norm, const float *row_turn, int pairs) {
    normed = norm != nullptr;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      weight[i] = 1.f;
      turn[i] = i & 1 ? 0.f : 1.f;
    }
    if (norm && VEC && valid > 0) {
      const f32x4_t lo = load4(norm + d), hi = load4(norm + d + 4);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        weight[i] = lo[i];
        weight[4 + i] = hi[i];
      }
    } else if (norm && !VEC) {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (i < valid) weight[i] = norm[d + i];
    }
    if (row_turn && d / 2 + 4 <= pairs && pairs % 2 == 0) {
      const f32x4_t lo = load4(row_turn + d), hi = load4(row_turn + d + 4);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        turn[i] = lo[i];
        turn[4 + i] = hi[i];
      }
    } else if (row_turn) {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (d / 2 + i / 2 < pairs) turn[i] = row_turn[d + i];
    }
  }

  // r: one over the head's root mean square
  __device__ __forceinline__ void apply(float (&v)[8], float r) const {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = v[i] * (normed ? r : 1.f) * weight[i];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float c = turn[2 * i], s = turn[2 * i + 1], x = v[2 * i], y = v[2 * i + 1];
      v[2 * i] = x * c - y * s;
      v[2 * i + 1] = y * c + x * s;
    }
  }
};

__device__ __forceinline__ const float *row_turns(const e2h_window_attention_args &a, size_t row) {
  return a.rotary ? a.rotary + row * a.rot_pairs * 2 : nullptr;
}

// norm and rotation of the query that a lane column holds as matrix operands (lane b4 of the column: dimensions 32 s + 8 b4 .. + 7)
template <int KS, bool VEC>
__device__ __forceinline__ void prepare_query(bf16x8_t (&qf)[KS], const e2h_window_attention_args &a, size_t row, int D, int b4) {
  if (!a.q_norm && !a.rotary) return;
  float v[KS][8], ss = 0.f;
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const u32x4_t raw = __builtin_bit_cast(u32x4_t, qf[s]);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[s][i] = __builtin_bit_cast(float, (i & 1) ? (raw[i >> 1] & 0xFFFF0000u) : (raw[i >> 1] << 16));
    ss += square_sum8(v[s]);
  }
  ss += __shfl_xor(ss, 16);
  ss += __shfl_xor(ss, 32);
  const float r = 1.0f / sqrtf(ss / static_cast<float>(D) + a.norm_eps);
  const float *turn = row_turns(a, row);
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const int d = 32 * s + 8 * b4;
    NormRotate8 f;
    f.load<VEC>(d, D - d, a.q_norm, turn, static_cast<int>(a.rot_pairs));
    f.apply(v[s], r);
    qf[s] = __builtin_bit_cast(bf16x8_t, u32x4_t{pack_bf16(v[s][0], v[s][1]), pack_bf16(v[s][2], v[s][3]), pack_bf16(v[s][4], v[s][5]),
                                                 pack_bf16(v[s][6], v[s][7])});
  }
}

// (cos, sin) of every row's position and rotated pair; the turn fraction is taken in float64, so far positions stay exact
__global__ __launch_bounds__(256) void rotary_table_kernel(const double *turns, const int64_t *input_pos, const int64_t *first, float *table,
                                                           int64_t n, int seqlen, int pairs) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= n) return;
  const int64_t row = i / pairs, b = row / seqlen;
  const int64_t pos = input_pos[0] + row % seqlen - (first ? first[b] : 0);
  const double t = static_cast<double>(pos) * turns[i % pairs];
  float s, c;
  sincospif(static_cast<float>(2.0 * (t - rint(t))), &s, &c);
  table[2 * i] = c;
  table[2 * i + 1] = s;
}

// ---- new keys and values into the caches ---------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void kv_append_kernel(const e2h_window_attention_args a) {
  const int per_row = static_cast<int>(a.kv_heads * (a.dim + a.vdim));
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (idx >= a.batch * a.seqlen * per_row) return;
  const int64_t row = idx / per_row;
  int c = static_cast<int>(idx % per_row);
  const int64_t b = row / a.seqlen, pos = a.input_pos[0] + row % a.seqlen;
  if (pos < 0 || pos >= a.cache_len) return;
  const T *src = static_cast<const T *>(a.proj) + row * a.ld;
  const int kw = static_cast<int>(a.kv_heads * a.dim);
  const bool is_k = c < kw;
  if (!is_k) c -= kw;
  const int d = static_cast<int>(is_k ? a.dim : a.vdim);
  float v = to_f32(src[(is_k ? a.k_off : a.v_off) + c]);
  const float *bias = is_k ? a.k_bias : a.v_bias;
  if (bias) v += bias[c];
  T *dst = static_cast<T *>(is_k ? a.k_cache : a.v_cache);
  dst[((b * a.kv_heads + c / d) * a.cache_len + pos) * d + c % d] = from_f32<T>(v);
}

// the same for bfloat16, eight values per thread (head sizes and columns multiples of eight)
__global__ __launch_bounds__(256) void kv_append8_kernel(const e2h_window_attention_args a) {
  const int kw = static_cast<int>(a.kv_heads * a.dim) / 8, per_row = kw + static_cast<int>(a.kv_heads * a.vdim) / 8;
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (idx >= a.batch * a.seqlen * per_row) return;
  const int row = static_cast<int>(idx / per_row), seqlen = static_cast<int>(a.seqlen);
  const bool is_k = idx % per_row < kw;
  const int c = static_cast<int>(idx % per_row - (is_k ? 0 : kw)) * 8;
  const int64_t b = row / seqlen, pos = a.input_pos[0] + row % seqlen;
  if (pos < 0 || pos >= a.cache_len) return;
  const int d = static_cast<int>(is_k ? a.dim : a.vdim);
  const bf16_t *src = static_cast<const bf16_t *>(a.proj) + row * a.ld + (is_k ? a.k_off : a.v_off) + c;
  f32x4_t lo = load4(src), hi = load4(src + 4);
  const float *bias = is_k ? a.k_bias : a.v_bias;
  if (bias) {
    lo += load4(bias + c);
    hi += load4(bias + c + 4);
  }
  bf16_t *dst = static_cast<bf16_t *>(is_k ? a.k_cache : a.v_cache) + ((b * a.kv_heads + c / d) * a.cache_len + pos) * d + c % d;
  store4(dst, lo);
  store4(dst + 4, hi);
}

// Appending with norm or rotation of the keys: `lanes` neighbouring lanes (a power of two, 8 dimensions each) per head; the key
// heads of a row first, then its value heads.
template <typename T, bool VEC>
__global__ __launch_bounds__(256) void kv_prepare_kernel(const e2h_window_attention_args a, int lanes) {
  const int G = static_cast<int>(a.kv_heads), D = static_cast<int>(a.dim), DV = static_cast<int>(a.vdim);
  const int shift = __builtin_ctz(lanes), items = static_cast<int>(a.batch * a.seqlen) * 2 * G, seqlen = static_cast<int>(a.seqlen);
  const int id = static_cast<int>((blockIdx.x * 256 + threadIdx.x) >> shift);
  const bool active = id < items;  // idle lanes stay for the shuffles
  const int row = active ? id / (2 * G) : 0, head = active ? id - row * 2 * G : 0;
  const bool is_k = head < G;
  const int g = is_k ? head : head - G, size = is_k ? D : DV, d = static_cast<int>(threadIdx.x & (lanes - 1)) * 8;
  const int64_t b = row / seqlen, pos = a.input_pos[0] + row % seqlen;
  const int valid = active ? size - d : 0;
  const int64_t col = static_cast<int64_t>(g) * size + d;
  float v[8];
  load8_f32<T, VEC>(static_cast<const T *>(a.proj) + static_cast<size_t>(row) * a.ld + (is_k ? a.k_off : a.v_off) + col, valid, v);
  const float *bias = is_k ? a.k_bias : a.v_bias;
  if (bias) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (i < valid) v[i] += bias[col + i];
  }
  NormRotate8 f;
  f.load<VEC>(d, is_k ? valid : 0, is_k ? a.k_norm : nullptr, is_k ? row_turns(a, row) : nullptr, static_cast<int>(a.rot_pairs));
  float ss = square_sum8(v);
  for (int off = lanes / 2; off > 0; off >>= 1) ss += __shfl_xor(ss, off);
  if (!active || pos < 0 || pos >= a.cache_len) return;
  if (is_k) f.apply(v, 1.0f / sqrtf(ss / static_cast<float>(D) + a.norm_eps));
  T *dst = static_cast<T *>(is_k ? a.k_cache : a.v_cache) + ((b * G + g) * a.cache_len + pos) * size + d;
  store8_f32<T, VEC>(dst, valid, v);
}

// ---- float32: one wave per (row, head) ------------------------------------------------------------------------------------
constexpr int kMaxHeadDim = 256;

template <typename T>
__global__ __launch_bounds__(256) void attention_rows_kernel(const e2h_window_attention_args a) {
  __shared__ float sh_q[4][kMaxHeadDim], sh_p[4][64];
  __shared__ int sh_j[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t item = static_cast<int64_t>(blockIdx.x) * 4 + wave;
  const bool active = item < a.batch * a.seqlen * a.heads;  // every wave reaches the end; idle ones hold no keys
  const int64_t row = active ? item / a.heads : 0;
  const int h = active ? static_cast<int>(item % a.heads) : 0;
  const int64_t b = row / a.seqlen;
  const int g = h / static_cast<int>(a.heads / a.kv_heads);
  const int pos = static_cast<int>(a.input_pos[0] + row % a.seqlen);
  const int first = a.first ? static_cast<int>(a.first[b]) : 0;
  const int D = static_cast<int>(a.dim), DV = static_cast<int>(a.vdim);
  const T *src = static_cast<const T *>(a.proj) + row * a.ld;
  for (int d = lane; d < D; d += 64) sh_q[wave][d] = to_f32(src[a.q_off + static_cast<int64_t>(h) * D + d]) + (a.q_bias ? a.q_bias[h * D + d] : 0.f);
  if (a.q_norm) {
    float ss = 0.f;
    for (int d = lane; d < D; d += 64) ss = __builtin_fmaf(sh_q[wave][d], sh_q[wave][d], ss);
    const float r = 1.0f / sqrtf(wave_add(ss) / static_cast<float>(D) + a.norm_eps);
    for (int d = lane; d < D; d += 64) sh_q[wave][d] = sh_q[wave][d] * r * a.q_norm[d];
  }
  if (a.rotary) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // wave-private LDS: the pairs cross lanes
    const float *turn = row_turns(a, row);
    for (int i = lane; i < a.rot_pairs; i += 64) {
      const float c = turn[2 * i], s = turn[2 * i + 1], x = sh_q[wave][2 * i], y = sh_q[wave][2 * i + 1];
      sh_q[wave][2 * i] = x * c - y * s;
      sh_q[wave][2 * i + 1] = y * c + x * s;
    }
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  const int last = pos < a.cache_len ? pos : static_cast<int>(a.cache_len) - 1;
  const KeyList kl = key_list(pos, last, first, static_cast<int>(a.window), static_cast<int>(a.keep_first));
  const int count = active ? kl.count : 0;
  const T *kc = static_cast<const T *>(a.k_cache) + (b * a.kv_heads + g) * a.cache_len * D;
  const T *vc = static_cast<const T *>(a.v_cache) + (b * a.kv_heads + g) * a.cache_len * DV;
  float m = kMasked, l = 0.f, acc[kMaxHeadDim / 64] = {0.f, 0.f, 0.f, 0.f};
  for (int n0 = 0; n0 < count; n0 += 64) {
    const int n = n0 + lane;
    float s = kMasked;
    int j = first;
    if (n < count) {
      j = kl.at(n);
      const T *kr = kc + static_cast<size_t>(j) * D;
      float dot = 0.f;
      for (int d = 0; d < D; ++d) dot = __builtin_fmaf(sh_q[wave][d], to_f32(kr[d]), dot);
      if (sees(pos, j, first, static_cast<int>(a.window), static_cast<int>(a.keep_first))) s = dot * a.scale;
    }
    float mx = s;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
    const float m_new = fmaxf(m, mx);
    const float corr = expf(m - m_new);
    const float p = s > 0.5f * kMasked ? expf(s - m_new) : 0.f;
    m = m_new;
    l = l * corr + wave_add(p);
    sh_p[wave][lane] = p;
    sh_j[wave][lane] = j;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // wave-private LDS
    const int live = count - n0 < 64 ? count - n0 : 64;
#pragma unroll
    for (int i = 0; i < kMaxHeadDim / 64; ++i) {
      const int d = i * 64 + lane;
      if (d < DV) {
        float o = acc[i] * corr;
        for (int n2 = 0; n2 < live; ++n2) o = __builtin_fmaf(sh_p[wave][n2], to_f32(vc[static_cast<size_t>(sh_j[wave][n2]) * DV + d]), o);
        acc[i] = o;
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
  if (!active) return;
  if (a.sink) l += expf(a.sink[h] - m);
#pragma unroll
  for (int i = 0; i < kMaxHeadDim / 64; ++i) {
    const int d = i * 64 + lane;
    if (d < DV) {
      float o = l > 0.f ? acc[i] / l : 0.f;
      if (a.g_off >= 0) o *= sigmoid_f32(to_f32(src[a.g_off + static_cast<int64_t>(h) * DV + d]));
      static_cast<T *>(a.out)[row * a.ld_out + a.out_off + static_cast<int64_t>(h) * DV + d] = from_f32<T>(o * a.out_scale);
    }
  }
}

// weights of two key tiles (keys 4b .. 4b+3 and 16+4b .. 16+4b+3 of this lane's query) as value + remainder operands
__device__ __forceinline__ void split_weights(const float (&p)[8], bf16x8_t &hi, bf16x8_t &lo) {
  u32x4_t h, l;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t a = __builtin_bit_cast(uint32_t, p[2 * i]) & 0xFFFF0000u, b = __builtin_bit_cast(uint32_t, p[2 * i + 1]) & 0xFFFF0000u;
    h[i] = (a >> 16) | b;
    l[i] = pack_bf16(p[2 * i] - __builtin_bit_cast(float, a), p[2 * i + 1] - __builtin_bit_cast(float, b));
  }
  hi = __builtin_bit_cast(bf16x8_t, h);
  lo = __builtin_bit_cast(bf16x8_t, l);
}

// ---- bfloat16, many tokens: 4 waves x 16 queries of one head, key tiles of 64 shared through LDS ----------------------
// KS: head dimension in steps of 32 (zero padded), VT: value dimension in tiles of 16.
template <int KS, int VT, bool VEC>
__global__ __launch_bounds__(256) void attention_prefill_kernel(const e2h_window_attention_args a, int q_blocks) {
  constexpr int kKeys = 64;
  constexpr int kKRow = KS * 64 + 16;   // bytes per key row (padding spreads the rows over the banks)
  constexpr int kVRow = kKeys * 2 + 8;  // bytes per row of V^T (one value column, 64 keys)
  __shared__ __attribute__((aligned(16))) uint8_t sh_k[kKeys * kKRow];
  __shared__ __attribute__((aligned(16))) uint8_t sh_v[VT * 16 * kVRow];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 15, b4 = lane >> 4;
  const int D = static_cast<int>(a.dim), DV = static_cast<int>(a.vdim), seqlen = static_cast<int>(a.seqlen);
  // consecutive workgroups share a key/value head: query heads of one group first, then query blocks
  int w = blockIdx.x;
  const int rep = static_cast<int>(a.heads / a.kv_heads);
  const int r = w % rep;
  w /= rep;
  const int qb = q_blocks - 1 - w % q_blocks;  // blocks with the most keys start first
  w /= q_blocks;
  const int g = w % static_cast<int>(a.kv_heads);
  const int bi = w / static_cast<int>(a.kv_heads);
  const int h = g * rep + r;
  const int pos0 = static_cast<int>(a.input_pos[0]);
  const int first = a.first ? static_cast<int>(a.first[bi]) : 0;
  const int t0 = qb * 64;
  const int t_last = t0 + 63 < seqlen - 1 ? t0 + 63 : seqlen - 1;
  const int cache_last = static_cast<int>(a.cache_len) - 1;
  const int pb = pos0 + t_last < cache_last ? pos0 + t_last : cache_last;
  const KeyList kl = key_list(pos0 + t0, pb, first, static_cast<int>(a.window), static_cast<int>(a.keep_first));
  const bf16_t *proj = static_cast<const bf16_t *>(a.proj);
  const bf16_t *kc = static_cast<const bf16_t *>(a.k_cache) + (static_cast<size_t>(bi) * a.kv_heads + g) * a.cache_len * D;
  const bf16_t *vc = static_cast<const bf16_t *>(a.v_cache) + (static_cast<size_t>(bi) * a.kv_heads + g) * a.cache_len * DV;
  const size_t row0 = static_cast<size_t>(bi) * seqlen;

  const int tq = t0 + wave * 16 + c, tc = tq < seqlen ? tq : seqlen - 1;
  bf16x8_t qf[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const int d = 32 * s + 8 * b4;
    u32x4_t raw = load8<VEC>(proj + (row0 + tc) * a.ld + a.q_off + static_cast<int64_t>(h) * D + d, D - d);
    if (a.q_bias) raw = add_bias8(raw, a.q_bias + static_cast<int64_t>(h) * D + d, D - d);
    qf[s] = __builtin_bit_cast(bf16x8_t, raw);
  }
  prepare_query<KS, VEC>(qf, a, row0 + tc, D, b4);
  f32x4_t oacc[VT];
  float m_run = kMasked, l_run = 0.f;
#pragma unroll
  for (int v = 0; v < VT; ++v) oacc[v] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const float sc = a.scale * kLog2e;

  constexpr int kKPieces = kKeys * KS * 4, kVPieces = kKeys * VT * 2;  // 16-byte pieces per tile
  constexpr int kKPer = kKPieces / 256, kVPer = (kVPieces + 255) / 256;
  u32x4_t kr[kKPer], vr[kVPer];
  auto fetch = [&](int n0) {
#pragma unroll
    for (int i = 0; i < kKPer; ++i) {
      const int piece = i * 256 + threadIdx.x, n = n0 + piece / (KS * 4), d = (piece % (KS * 4)) * 8;
      kr[i] = u32x4_t{0u, 0u, 0u, 0u};
      if (n < kl.count) kr[i] = load8<VEC>(kc + static_cast<size_t>(kl.at(n)) * D + d, D - d);
    }
    // V pieces: consecutive threads take consecutive keys of one column group, so the transposed 2-byte LDS writes of a wave
    // fill whole rows
#pragma unroll
    for (int i = 0; i < kVPer; ++i) {
      const int piece = i * 256 + threadIdx.x, n = n0 + piece % kKeys, d = (piece / kKeys) * 8;
      vr[i] = u32x4_t{0u, 0u, 0u, 0u};
      if (piece < kVPieces && n < kl.count) vr[i] = load8<VEC>(vc + static_cast<size_t>(kl.at(n)) * DV + d, DV - d);
    }
  };
  if (kl.count > 0) fetch(0);
  for (int n0 = 0; n0 < kl.count; n0 += kKeys) {
    __syncthreads();  // the previous tile has been read
#pragma unroll
    for (int i = 0; i < kKPer; ++i) {
      const int piece = i * 256 + threadIdx.x;
      *reinterpret_cast<u32x4_t *>(sh_k + (piece / (KS * 4)) * kKRow + (piece % (KS * 4)) * 16) = kr[i];
    }
#pragma unroll
    for (int i = 0; i < kVPer; ++i) {
      const int piece = i * 256 + threadIdx.x, n = piece % kKeys, d = (piece / kKeys) * 8;
      if (piece < kVPieces) {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          *reinterpret_cast<uint16_t *>(sh_v + (d + e) * kVRow + n * 2) = static_cast<uint16_t>(vr[i][e >> 1] >> (16 * (e & 1)));
      }
    }
    __syncthreads();
    if (n0 + kKeys < kl.count) fetch(n0 + kKeys);

    f32x4_t st[4];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
      st[kt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const bf16x8_t kf = *reinterpret_cast<const bf16x8_t *>(sh_k + (16 * kt + c) * kKRow + s * 64 + b4 * 16);
        st[kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[s], st[kt], 0, 0, 0);
      }
    }
    // a tile inside every query's window needs no masks: whole, behind the kept keys, not beyond the first query, not out of
    // the last one's window
    const int q_lo = pos0 + t0 + wave * 16, q_hi = q_lo + 15;
    const bool open = n0 >= kl.kept && n0 + kKeys <= kl.count && kl.at(n0 + kKeys - 1) <= q_lo && q_hi - kl.at(n0) < static_cast<int>(a.window);
    if (!__builtin_amdgcn_readfirstlane(open)) {
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int n = n0 + 16 * kt + 4 * b4 + e;
          const int j = n < kl.count ? kl.at(n) : INT32_MAX;
          if (!sees(pos0 + tq, j, first, static_cast<int>(a.window), static_cast<int>(a.keep_first))) st[kt][e] = kMasked;
        }
    }
    float mx = st[0][0];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
      for (int e = 0; e < 4; ++e) mx = fmaxf(mx, st[kt][e]);
    mx = fmaxf(mx, __shfl_xor(mx, 16));
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    const float m_new = fmaxf(m_run, mx);
    // while a query has seen no key its maximum is the mask value: exponents are then taken against 0, where masked scores give 0
    const float m_ref = m_new > 0.5f * kMasked ? m_new * sc : 0.f;
    const float corr = __builtin_amdgcn_exp2f(__builtin_fmaf(m_run, sc, -m_ref));
    m_run = m_new;
    float ls = 0.f;
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        st[kt][e] = __builtin_amdgcn_exp2f(__builtin_fmaf(st[kt][e], sc, -m_ref));
        ls += st[kt][e];
      }
    l_run = l_run * corr + ls;
#pragma unroll
    for (int v = 0; v < VT; ++v)
#pragma unroll
      for (int e = 0; e < 4; ++e) oacc[v][e] *= corr;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      bf16x8_t hi, lo;
      float p[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) p[e] = st[2 * half + (e >> 2)][e & 3];
      split_weights(p, hi, lo);
#pragma unroll
      for (int v = 0; v < VT; ++v) {
        const uint8_t *vp = sh_v + (16 * v + c) * kVRow + half * 64 + b4 * 8;
        const u32x2_t v0 = *reinterpret_cast<const u32x2_t *>(vp), v1 = *reinterpret_cast<const u32x2_t *>(vp + 32);
        const bf16x8_t vf = __builtin_bit_cast(bf16x8_t, u32x4_t{v0[0], v0[1], v1[0], v1[1]});
        oacc[v] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, hi, oacc[v], 0, 0, 0);
        oacc[v] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, lo, oacc[v], 0, 0, 0);
      }
    }
  }
  // lane (b, c): value columns 16 v + 4 b .. + 3 of query c
  float l = l_run;
  l += __shfl_xor(l, 16);
  l += __shfl_xor(l, 32);
  if (a.sink) l += __builtin_amdgcn_exp2f(__builtin_fmaf(a.sink[h], kLog2e, -m_run * sc));
  const float inv = l > 0.f ? a.out_scale / l : 0.f;
  if (tq >= seqlen) return;
  const size_t row = row0 + tq;
#pragma unroll
  for (int v = 0; v < VT; ++v) {
    const int d = 16 * v + 4 * b4;
    f32x4_t o = oacc[v] * inv;
    const bf16_t *gate = proj + row * a.ld + a.g_off + static_cast<int64_t>(h) * DV + d;
    bf16_t *dst = static_cast<bf16_t *>(a.out) + row * a.ld_out + a.out_off + static_cast<int64_t>(h) * DV + d;
    if (VEC) {
      if (d < DV) {
        if (a.g_off >= 0) {
          const f32x4_t g = load4(gate);
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] *= fast_sigmoid(g[e]);
        }
        store4(dst, o);
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (d + e < DV) dst[e] = from_f32<bf16_t>(a.g_off >= 0 ? o[e] * fast_sigmoid(to_f32(gate[e])) : o[e]);
    }
  }
}

// ---- the same for many queries with heads of 64 or 128 dimensions: 4 waves x 32 queries (e2h_attention_tiles.h) -----------------------------------------
template <int D>
__global__ __launch_bounds__(256, 2) void attention_prompt_kernel(const e2h_window_attention_args a, int q_blocks) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int KS = D / 32, VT = D / 16;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[attention::kLdsBytes<D>];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = lane & 15, b4 = lane >> 4;
  const int seqlen = static_cast<int>(a.seqlen);
  const int rep = static_cast<int>(a.heads / a.kv_heads);
  const attention::Place at = attention::place(blockIdx.x, static_cast<int>(a.batch * a.kv_heads), rep, q_blocks);
  const int qb = q_blocks - 1 - at.back, g = at.pair % static_cast<int>(a.kv_heads), bi = at.pair / static_cast<int>(a.kv_heads), h = g * rep + at.rep;
  const int pos0 = static_cast<int>(a.input_pos[0]), first = a.first ? static_cast<int>(a.first[bi]) : 0;
  const int t0 = qb * attention::kQueries, t1 = t0 + attention::kQueries - 1 < seqlen - 1 ? t0 + attention::kQueries - 1 : seqlen - 1;
  const int cache_last = static_cast<int>(a.cache_len) - 1, pb = pos0 + t1 < cache_last ? pos0 + t1 : cache_last;
  const KeyList list = key_list(pos0 + t0, pb, first, static_cast<int>(a.window), static_cast<int>(a.keep_first));
  const attention::Keys keys = {list.first, list.kept, list.start, list.count};
  const attention::Rule rule = {first, static_cast<int>(a.window), static_cast<int>(a.keep_first)};
  const bf16_t *proj = static_cast<const bf16_t *>(a.proj);
  const size_t row0 = static_cast<size_t>(bi) * seqlen, head = static_cast<size_t>(bi) * a.kv_heads + g;
  bf16x8_t qf[2][KS];
  int pos[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int tq = t0 + wave * 32 + 16 * i + c, tc = tq < seqlen ? tq : seqlen - 1;
    pos[i] = pos0 + tq;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int64_t d = static_cast<int64_t>(h) * D + 32 * s + 8 * b4;
      u32x4_t raw = *reinterpret_cast<const u32x4_t *>(proj + (row0 + tc) * a.ld + a.q_off + d);
      if (a.q_bias) raw = add_bias8(raw, a.q_bias + d, 8);
      qf[i][s] = __builtin_bit_cast(bf16x8_t, raw);
    }
    prepare_query<KS, true>(qf[i], a, row0 + tc, D, b4);
  }
  f32x4_t o[2][VT];
  float m[2], l[2];
  const float sc = a.scale * kLog2e;
  const int lo = pos0 + t0 + wave * 32;
  attention::attend<D, true, false>(qf, pos, lo, lo + 31, keys, rule, sc, static_cast<const bf16_t *>(a.k_cache) + head * a.cache_len * D,
                             static_cast<const bf16_t *>(a.v_cache) + head * a.cache_len * D, static_cast<uint32_t>(a.cache_len), lds, o, m, l);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int tq = t0 + wave * 32 + 16 * i + c;
    float sum = l[i];
    sum += __shfl_xor(sum, 16);
    sum += __shfl_xor(sum, 32);
    if (a.sink) sum += __builtin_amdgcn_exp2f(__builtin_fmaf(a.sink[h], kLog2e, m[i] > attention::kMaskedScore ? -m[i] * sc : 0.f));
    const float inv = sum > 0.f ? a.out_scale / sum : 0.f;
    if (tq >= seqlen) continue;
    const size_t row = row0 + tq;
#pragma unroll
    for (int v = 0; v < VT; ++v) {
      const int64_t d = static_cast<int64_t>(h) * D + 16 * v + 4 * b4;
      f32x4_t out = o[i][v] * inv;
      if (a.g_off >= 0) {
        const f32x4_t gate = load4(proj + row * a.ld + a.g_off + d);
#pragma unroll
        for (int e = 0; e < 4; ++e) out[e] *= fast_sigmoid(gate[e]);
      }
      store4(static_cast<bf16_t *>(a.out) + row * a.ld_out + a.out_off + d, out);
    }
  }
#endif
}

// ---- bfloat16, one token per sequence: `splits` workgroups per (sequence, key/value head) --------------------------------------
// The lane columns are the query heads of the group (up to 16); the waves of all its workgroups take key tiles of 32 round robin and
// are combined at the end: in LDS, then, where there are several workgroups, by attention_combine_kernel from `part`
// ([sequence and key/value head][split][head of the group][DV sums, maximum, sum of weights]).  The workgroup whose tile holds the new
// token's row appends that row first.
// A tile is a serial chain of 2.4 us (load, product, softmax, product), so what bounds few sequences is tiles per wave and not
// bytes: 4 sequences x 8 key heads over 2048 keys took 25.5 us with one workgroup each (9 tiles per wave on 32 of 256 CUs), 12.9 with eight; 1 sequence 23.9 and 11.6; 30000 keys 273 and
// 29.  32 sequences (256 workgroups, no split) read 5.2 TB/s.
// `splits` is for the cache's capacity; workgroups beyond the keys that there are end at once, and where one is left it writes the result itself.
__device__ __forceinline__ int parts_with_keys(int count, int waves, int splits) {
  const int rounds = (count + 32 * waves - 1) / (32 * waves);  // tiles of a wave of one workgroup
  return rounds < 2 ? 1 : rounds < splits ? rounds : splits;
}

template <int KS, int VT, int NW, bool VEC>
__global__ __launch_bounds__(64 * NW) void attention_step_kernel(const e2h_window_attention_args a, int splits, float *part) {
  constexpr int kVRow = VT * 32 + 8;  // bytes per value row in LDS
  constexpr int kWaveLds = 32 * kVRow;
  constexpr int kEndLds = NW * (16 * VT * 16 + 32) * 4;
  constexpr int kLds = NW * kWaveLds > kEndLds ? NW * kWaveLds : kEndLds;
  __shared__ __attribute__((aligned(16))) uint8_t lds[kLds];
  const int lane = threadIdx.x & 63, c = lane & 15, b4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int D = static_cast<int>(a.dim), DV = static_cast<int>(a.vdim);
  const int split = static_cast<int>(blockIdx.x % splits), pair = static_cast<int>(blockIdx.x / splits);
  const int bi = pair / static_cast<int>(a.kv_heads), g = pair % static_cast<int>(a.kv_heads);
  const int rep = static_cast<int>(a.heads / a.kv_heads);
  const int pos = static_cast<int>(a.input_pos[0]);
  const int first = a.first ? static_cast<int>(a.first[bi]) : 0;
  const int last = pos < a.cache_len ? pos : static_cast<int>(a.cache_len) - 1;
  const KeyList kl = key_list(pos, last, first, static_cast<int>(a.window), static_cast<int>(a.keep_first));
  const int parts = parts_with_keys(kl.count, NW, splits);
  if (split >= parts) return;  // the whole workgroup
  if (parts == 1) part = nullptr;
  // the list ends with the new token's row
  const bool appends = split == (kl.count > 0 ? (kl.count - 1) / 32 / NW % parts : 0);
  const bf16_t *proj = static_cast<const bf16_t *>(a.proj) + static_cast<size_t>(bi) * a.ld;
  bf16_t *kc = static_cast<bf16_t *>(a.k_cache) + (static_cast<size_t>(bi) * a.kv_heads + g) * a.cache_len * D;
  bf16_t *vc = static_cast<bf16_t *>(a.v_cache) + (static_cast<size_t>(bi) * a.kv_heads + g) * a.cache_len * DV;
  const bool prepared = a.k_norm || a.rotary;
  if (appends && a.k_off >= 0 && pos >= 0 && pos < a.cache_len) {
    if (prepared && wave == 0) {  // norm and rotation by the first wave, the others copy the value
      const int d = 8 * lane;
      float v[8];
      load8_f32<bf16_t, false>(proj + a.k_off + static_cast<int64_t>(g) * D + (d < D ? d : 0), D - d, v);
      if (a.k_bias) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (d + i < D) v[i] += a.k_bias[g * D + d + i];
      }
      const float r = 1.0f / sqrtf(wave_add(square_sum8(v)) / static_cast<float>(D) + a.norm_eps);
      if (d < D) {
        NormRotate8 f;
        f.load<VEC>(d, D - d, a.k_norm, row_turns(a, bi), static_cast<int>(a.rot_pairs));
        f.apply(v, r);
        store8_f32<bf16_t, VEC>(kc + static_cast<size_t>(pos) * D + d, D - d, v);
      }
    }
    for (int i = prepared ? static_cast<int>(threadIdx.x) - 64 + D : static_cast<int>(threadIdx.x); i < D + DV; i += 64 * NW - (prepared ? 64 : 0)) {
      const bool is_k = i < D;
      if (is_k && prepared) break;  // a lane of the first wave
      const int d = is_k ? i : i - D;
      const int col = g * (is_k ? D : DV) + d;
      float v = to_f32(proj[(is_k ? a.k_off : a.v_off) + col]);
      const float *bias = is_k ? a.k_bias : a.v_bias;
      if (bias) v += bias[col];
      (is_k ? kc + static_cast<size_t>(pos) * D : vc + static_cast<size_t>(pos) * DV)[d] = from_f32<bf16_t>(v);
    }
  }
  bf16x8_t qf[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const int d = 32 * s + 8 * b4;
    u32x4_t raw = {0u, 0u, 0u, 0u};
    if (c < rep) {
      raw = load8<VEC>(proj + a.q_off + static_cast<int64_t>(g * rep + c) * D + d, D - d);
      if (a.q_bias) raw = add_bias8(raw, a.q_bias + static_cast<int64_t>(g * rep + c) * D + d, D - d);
    }
    qf[s] = __builtin_bit_cast(bf16x8_t, raw);
  }
  prepare_query<KS, VEC>(qf, a, bi, D, b4);
  __threadfence_block();
  __syncthreads();  // the new row is visible to the workgroup

  f32x4_t oacc[VT];
  float m_run = kMasked, l_run = 0.f;
#pragma unroll
  for (int v = 0; v < VT; ++v) oacc[v] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const float sc = a.scale * kLog2e;
  uint8_t *v_lds = lds + wave * kWaveLds;
  constexpr int kVPer = (32 * VT * 2 + 63) / 64;

  for (int n0 = (split * NW + wave) * 32; n0 < kl.count; n0 += parts * NW * 32) {
    u32x4_t kf[2][KS], vr[kVPer];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int n = n0 + 16 * t + c;
      const int j = kl.at(n < kl.count ? n : kl.count - 1);
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const int d = 32 * s + 8 * b4;
        kf[t][s] = load8<VEC>(kc + static_cast<size_t>(j) * D + d, D - d);
      }
    }
#pragma unroll
    for (int i = 0; i < kVPer; ++i) {
      const int piece = i * 64 + lane, n = n0 + piece / (VT * 2), d = (piece % (VT * 2)) * 8;
      const int j = kl.at(n < kl.count ? n : kl.count - 1);
      vr[i] = load8<VEC>(vc + static_cast<size_t>(j) * DV + d, DV - d);
    }
    f32x4_t st[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      st[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s)
        st[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, kf[t][s]), qf[s], st[t], 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < kVPer; ++i) {
      const int piece = i * 64 + lane;
      uint8_t *dst = v_lds + (piece / (VT * 2)) * kVRow + (piece % (VT * 2)) * 16;
      *reinterpret_cast<u32x2_t *>(dst) = u32x2_t{vr[i][0], vr[i][1]};
      *reinterpret_cast<u32x2_t *>(dst + 8) = u32x2_t{vr[i][2], vr[i][3]};
    }
    float p[8], mx = kMasked;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int n = n0 + 16 * (e >> 2) + 4 * b4 + (e & 3);
      p[e] = n < kl.count ? st[e >> 2][e & 3] * sc : kMasked;  // every listed key is visible to the one query position
      mx = fmaxf(mx, p[e]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16));
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    const float m_new = fmaxf(m_run, mx);
    const float corr = __builtin_amdgcn_exp2f(m_run - m_new);
    m_run = m_new;
    float ls = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      p[e] = p[e] > 0.5f * kMasked ? __builtin_amdgcn_exp2f(p[e] - m_new) : 0.f;
      ls += p[e];
    }
    l_run = l_run * corr + ls;
    bf16x8_t hi, lo;
    split_weights(p, hi, lo);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // wave-private tile: the wave's own writes have landed
#pragma unroll
    for (int v = 0; v < VT; ++v) {
      uint32_t vw[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int k0 = 16 * (i >> 1) + 4 * b4 + 2 * (i & 1);
        const uint32_t x0 = *reinterpret_cast<const uint16_t *>(v_lds + k0 * kVRow + (16 * v + c) * 2);
        const uint32_t x1 = *reinterpret_cast<const uint16_t *>(v_lds + (k0 + 1) * kVRow + (16 * v + c) * 2);
        vw[i] = x0 | (x1 << 16);
      }
      const bf16x8_t vf = __builtin_bit_cast(bf16x8_t, u32x4_t{vw[0], vw[1], vw[2], vw[3]});
#pragma unroll
      for (int e = 0; e < 4; ++e) oacc[v][e] *= corr;
      oacc[v] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, hi, oacc[v], 0, 0, 0);
      oacc[v] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, lo, oacc[v], 0, 0, 0);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // reads done before the next tile overwrites the wave's LDS
  }
  __syncthreads();  // every wave is done with its tiles: the LDS is reused
  float *const sh_o = reinterpret_cast<float *>(lds);  // [NW][16 heads][VT * 16]
  float *const sh_m = sh_o + NW * 16 * VT * 16;        // [NW][16]
  float *const sh_l = sh_m + NW * 16;                  // [NW][16]
  l_run += __shfl_xor(l_run, 16);
  l_run += __shfl_xor(l_run, 32);
#pragma unroll
  for (int v = 0; v < VT; ++v) *reinterpret_cast<f32x4_t *>(sh_o + (wave * 16 + c) * VT * 16 + 16 * v + 4 * b4) = oacc[v];
  if (b4 == 0) {
    sh_m[wave * 16 + c] = m_run;
    sh_l[wave * 16 + c] = l_run;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < rep * DV; e += 64 * NW) {
    const int r = e / DV, d = e % DV;
    float m = sh_m[r];
#pragma unroll
    for (int w = 1; w < NW; ++w) m = fmaxf(m, sh_m[w * 16 + r]);
    float l = 0.f, o = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float cw = __builtin_amdgcn_exp2f(sh_m[w * 16 + r] - m);
      l += sh_l[w * 16 + r] * cw;
      o += sh_o[(w * 16 + r) * VT * 16 + d] * cw;
    }
    if (part) {
      float *row = part + (static_cast<size_t>(blockIdx.x) * rep + r) * (DV + 2);
      row[d] = o;
      if (d == 0) {
        row[DV] = m;
        row[DV + 1] = l;
      }
      continue;
    }
    if (a.sink) l += __builtin_amdgcn_exp2f(__builtin_fmaf(a.sink[g * rep + r], kLog2e, -m));
    const int col = (g * rep + r) * DV + d;
    o = l > 0.f ? o / l * a.out_scale : 0.f;
    if (a.g_off >= 0) o *= sigmoid_f32(to_f32(proj[a.g_off + col]));
    static_cast<bf16_t *>(a.out)[static_cast<size_t>(bi) * a.ld_out + a.out_off + col] = from_f32<bf16_t>(o);
  }
}

// one value of one head per thread: the splits' sums, each in units of its own maximum, brought to the largest
__global__ __launch_bounds__(256) void attention_combine_kernel(const e2h_window_attention_args a, int waves, int splits, const float *part) {
  const int H = static_cast<int>(a.heads), G = static_cast<int>(a.kv_heads), DV = static_cast<int>(a.vdim), rep = H / G;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= a.batch * H * DV) return;
  const int d = static_cast<int>(i % DV), h = static_cast<int>(i / DV % H), bi = static_cast<int>(i / DV / H), stride = rep * (DV + 2);
  const int pos = static_cast<int>(a.input_pos[0]), last = pos < a.cache_len ? pos : static_cast<int>(a.cache_len) - 1;
  const int parts = parts_with_keys(key_list(pos, last, a.first ? static_cast<int>(a.first[bi]) : 0, static_cast<int>(a.window), static_cast<int>(a.keep_first)).count, waves, splits);
  const float *row = part + (static_cast<size_t>(bi) * G + h / rep) * splits * stride + (h % rep) * (DV + 2);
  constexpr int kAtOnce = 8;
  float m = kMasked, l = 0.f, o = 0.f;
  int s0 = 0;
  do {  // the first sums are requested while the count of parts is on its way: what no part has written is read and left
    float ms[kAtOnce], ls[kAtOnce], os[kAtOnce];
#pragma unroll
    for (int k = 0; k < kAtOnce; ++k) {
      const float *p = row + static_cast<size_t>(s0 + k < splits ? s0 + k : 0) * stride;
      ms[k] = p[DV];
      ls[k] = p[DV + 1];
      os[k] = p[d];
    }
#pragma unroll
    for (int k = 0; k < kAtOnce; ++k)
      if (s0 + k >= parts) {
        ms[k] = kMasked;
        ls[k] = os[k] = 0.f;
      }
    float m_new = m;
#pragma unroll
    for (int k = 0; k < kAtOnce; ++k) m_new = fmaxf(m_new, ms[k]);
    const float corr = __builtin_amdgcn_exp2f(m - m_new);
    l *= corr;
    o *= corr;
    m = m_new;
#pragma unroll
    for (int k = 0; k < kAtOnce; ++k) {
      const float c = __builtin_amdgcn_exp2f(ms[k] - m);
      l = __builtin_fmaf(ls[k], c, l);
      o = __builtin_fmaf(os[k], c, o);
    }
    s0 += kAtOnce;
  } while (s0 < parts);
  if (parts == 1) return;  // the step has written the result
  if (a.sink) l += __builtin_amdgcn_exp2f(__builtin_fmaf(a.sink[h], kLog2e, -m));
  o = l > 0.f ? o / l * a.out_scale : 0.f;
  if (a.g_off >= 0) o *= sigmoid_f32(to_f32(static_cast<const bf16_t *>(a.proj)[static_cast<size_t>(bi) * a.ld + a.g_off + static_cast<int64_t>(h) * DV + d]));
  static_cast<bf16_t *>(a.out)[static_cast<size_t>(bi) * a.ld_out + a.out_off + static_cast<int64_t>(h) * DV + d] = from_f32<bf16_t>(o);
}

bool on_matrix_cores(const e2h_window_attention_args &a) {
  return a.dtype == E2H_SEQ_BF16 && a.heads / a.kv_heads <= 16 && a.scale > 0.f;
}

// waves per workgroup of the step: one walks 32 keys at a time; more of them pay once there are enough keys to share
int64_t step_span(const e2h_window_attention_args &a) {
  return a.window > 0 && a.window <= INT32_MAX && a.keep_first <= INT32_MAX && a.window + a.keep_first < a.cache_len ? a.window + a.keep_first : a.cache_len;
}
int step_waves(const e2h_window_attention_args &a) {
  const int64_t d = a.dim > a.vdim ? a.dim : a.vdim;
  const int nw = seq_options().attention_decode_waves ? seq_options().attention_decode_waves : (step_span(a) > 256 ? 8 : 4);
  return d <= 128 ? nw : 4;
}

// Workgroups per (sequence, key/value head) of the step, by the cache's capacity (the position is on the device), so that there is one per CU at most (two cost more than they share: 8 sequences x
// 8 key heads over 2052 keys in 4 parts 18.8 us, in 8 parts 24.2).  A tile takes a wave 2.4 us and the combining launch 4 to 5, so fewer than
// three tiles per wave are not shared (300 keys, 4 sequences: 9.2 us whole, 10.9 in two parts), and two parts never pay: 86 and more
// workgroups already read at the memory's rate (16 sequences 27.2 us whole, 28.3 in two parts).  A position with few keys in a long cache pays 1 to 3.5
// us for a launch that combines little or nothing (8 key heads, cache of 8192; one workgroup / this, us: 1 sequence, 17 keys 6.7 / 8.9, 256 8.8 / 11.5, 500 11.1 / 12.2, 700 13.4 / 12.2,
// 2000 25 / 12.6; 4 sequences 6.7 / 9.1, 9.3 / 12.8, 11.9 / 13.5, 15.8 / 14.0, 32 / 17.8; with all workgroups of the capacity at work 11.9 and 14.4 at 17 and 256 keys of 1 sequence).
constexpr int kMostSplits = 64;
int step_splits(const e2h_window_attention_args &a) {
  if (a.seqlen != 1 || !on_matrix_cores(a)) return 1;
  const int64_t rounds = (step_span(a) + 32 * step_waves(a) - 1) / (32 * step_waves(a));  // tiles of a wave
  const int64_t fit = 256 / (a.batch * a.kv_heads);
  int64_t s = rounds < fit ? rounds : fit;
  s = s < kMostSplits ? s : kMostSplits;
  return s < 3 ? 1 : static_cast<int>(s);
}

int64_t step_scratch_bytes(const e2h_window_attention_args &a, int splits) {
  return splits < 2 ? 0 : a.batch * a.heads * splits * (a.vdim + 2) * 4;
}

// Queries per workgroup of a prompt, heads of 64 or 128 dimensions.  64 (16 per wave) while the workgroups are one per CU at most, and for portions that would leave half of a
// 128-query workgroup's waves without a query: such a launch is as long as its longest workgroup, and a wave with 16 queries walks its keys sooner.  us, 64 / 128 queries, heads of 128
// (of 64): 32 heads x 128 tokens 12.1 / 15.0 (9.5 / 13.0), 512 tokens, 256 workgroups, 26.3 / 27.6 (19.1 / 22.1), 768 tokens 39.8 / 36.3 (26.8 / 28.2), behind 1024
// cached 81.7 / 68.6 (54.8 / 50.1); 1024 56.6 / 45.0 (37.2 / 34.0); 512 heads x 16 tokens 10.8 / 11.6, x 64 behind 1024 cached 60.4 / 65.9, x 96 115 / 73.
int prompt_queries(const e2h_window_attention_args &a) {
  if (seq_options().attention_prompt_queries) return seq_options().attention_prompt_queries;
  return a.seqlen <= 64 || a.batch * a.heads * ((a.seqlen + 63) / 64) <= 256 ? 64 : 128;
}

void launch_append(const e2h_window_attention_args &a, bool vec, hipStream_t s) {
  if (a.k_off < 0) return;
  if (a.k_norm || a.rotary) {
    int lanes = 1;
    while (lanes * 8 < a.dim || lanes * 8 < a.vdim) lanes *= 2;
    const int64_t per = 256 / lanes, items = a.batch * a.seqlen * 2 * a.kv_heads;
    const dim3 grid(static_cast<unsigned>((items + per - 1) / per)), block(256);
    if (a.dtype == E2H_SEQ_F32) hipLaunchKernelGGL((kv_prepare_kernel<float, false>), grid, block, 0, s, a, lanes);
    else if (vec) hipLaunchKernelGGL((kv_prepare_kernel<bf16_t, true>), grid, block, 0, s, a, lanes);
    else hipLaunchKernelGGL((kv_prepare_kernel<bf16_t, false>), grid, block, 0, s, a, lanes);
    return;
  }
  if (vec) {
    const int64_t n8 = a.batch * a.seqlen * a.kv_heads * (a.dim + a.vdim) / 8;
    hipLaunchKernelGGL(kv_append8_kernel, dim3(static_cast<unsigned>((n8 + 255) / 256)), dim3(256), 0, s, a);
    return;
  }
  const int64_t n = a.batch * a.seqlen * a.kv_heads * (a.dim + a.vdim);
  const dim3 grid(static_cast<unsigned>((n + 255) / 256)), block(256);
  if (a.dtype == E2H_SEQ_BF16) hipLaunchKernelGGL(kv_append_kernel<bf16_t>, grid, block, 0, s, a);
  else hipLaunchKernelGGL(kv_append_kernel<float>, grid, block, 0, s, a);
}

template <int KS, int VT, bool VEC>
void launch_mfma(const e2h_window_attention_args &a, float *part, int64_t part_bytes, hipStream_t s) {
  if (a.seqlen == 1) {
    int splits = step_splits(a);
    if (!part || step_scratch_bytes(a, splits) > part_bytes) splits = 1;
    if (splits == 1) part = nullptr;
    const dim3 grid(static_cast<unsigned>(a.batch * a.kv_heads * splits));
    if (step_waves(a) == 8) hipLaunchKernelGGL((attention_step_kernel<KS, VT, (KS <= 4 ? 8 : 4), VEC>), grid, dim3(KS <= 4 ? 512 : 256), 0, s, a, splits, part);
    else hipLaunchKernelGGL((attention_step_kernel<KS, VT, 4, VEC>), grid, dim3(256), 0, s, a, splits, part);
    if (part) hipLaunchKernelGGL(attention_combine_kernel, dim3(static_cast<unsigned>((a.batch * a.heads * a.vdim + 255) / 256)), dim3(256), 0, s, a, step_waves(a), splits, part);
    return;
  }
  launch_append(a, VEC && aligned16(a.k_bias) && aligned16(a.v_bias) && a.k_off % 8 == 0 && a.v_off % 8 == 0, s);
  if constexpr (VEC && (KS == 2 || KS == 4) && VT == 2 * KS) {
    constexpr int D = 32 * KS;
    if (prompt_queries(a) == 128 && a.dim == D && a.vdim == D && a.cache_len <= static_cast<int64_t>(UINT32_MAX) / (2 * D)) {
      const int blocks = static_cast<int>((a.seqlen + attention::kQueries - 1) / attention::kQueries);
      hipLaunchKernelGGL(attention_prompt_kernel<D>, dim3(static_cast<unsigned>(a.batch * a.heads * blocks)), dim3(256), 0, s, a, blocks);
      return;
    }
  }
  const int q_blocks = static_cast<int>((a.seqlen + 63) / 64);
  hipLaunchKernelGGL((attention_prefill_kernel<KS, VT, VEC>), dim3(static_cast<unsigned>(a.batch * a.heads * q_blocks)), dim3(256), 0, s, a, q_blocks);
}

template <bool VEC>
void launch_mfma_by_size(const e2h_window_attention_args &a, float *part, int64_t part_bytes, hipStream_t s) {
  const int64_t d = a.dim > a.vdim ? a.dim : a.vdim;
  if (d <= 32) launch_mfma<1, 2, VEC>(a, part, part_bytes, s);
  else if (d <= 64) launch_mfma<2, 4, VEC>(a, part, part_bytes, s);
  else if (d <= 128) launch_mfma<4, 8, VEC>(a, part, part_bytes, s);
  else launch_mfma<8, 16, VEC>(a, part, part_bytes, s);
}

void launch_rows(const e2h_window_attention_args &a, hipStream_t s) {
  launch_append(a, false, s);
  const dim3 grid(static_cast<unsigned>((a.batch * a.seqlen * a.heads + 3) / 4)), block(256);
  if (a.dtype == E2H_SEQ_BF16) hipLaunchKernelGGL(attention_rows_kernel<bf16_t>, grid, block, 0, s, a);
  else hipLaunchKernelGGL(attention_rows_kernel<float>, grid, block, 0, s, a);
}

}  // namespace
}  // namespace e2h

using namespace e2h;

extern "C" int e2h_seq_rotary_table(const double *turns, const int64_t *input_pos, const int64_t *first, float *table, int64_t batch, int64_t seqlen,
                                    int64_t pairs, void *stream) {
  if (!turns || !input_pos || !table) return E2H_ERR_NULL_POINTER;
  if (batch < 1 || seqlen < 1 || pairs < 1 || seqlen > INT32_MAX / 4 || pairs > INT32_MAX / 4) return E2H_ERR_BAD_SHAPE;
  const int64_t n = batch * seqlen * pairs, blocks = (n + 255) / 256;
  if (blocks > INT32_MAX) return E2H_ERR_BAD_SHAPE;
  hipLaunchKernelGGL(rotary_table_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, static_cast<hipStream_t>(stream), turns, input_pos, first,
                     table, n, static_cast<int>(seqlen), static_cast<int>(pairs));
  return launch_status();
}

static int check_attention(const e2h_window_attention_args *a) {
  if (!a || !a->proj || !a->k_cache || !a->v_cache || !a->input_pos || !a->out) return E2H_ERR_NULL_POINTER;
  if (a->dtype != E2H_SEQ_BF16 && a->dtype != E2H_SEQ_F32) return E2H_ERR_BAD_SHAPE;
  if (a->batch < 1 || a->seqlen < 1 || a->heads < 1 || a->kv_heads < 1 || a->heads % a->kv_heads != 0 || a->dim < 1 || a->vdim < 1 ||
      a->dim > kMaxHeadDim || a->vdim > kMaxHeadDim || a->cache_len < 1 || a->cache_len > INT32_MAX / 2 || a->seqlen > INT32_MAX / 4)
    return E2H_ERR_BAD_SHAPE;
  if (a->window < 0 || a->keep_first < 0 || a->q_off < 0 || (a->k_off < 0) != (a->v_off < 0) || a->out_off < 0) return E2H_ERR_BAD_SHAPE;
  if (a->rotary && (a->rot_pairs < 1 || 2 * a->rot_pairs > a->dim)) return E2H_ERR_BAD_SHAPE;
  if (!aligned16(a->rotary)) return E2H_ERR_MISALIGNED;
  if ((a->k_norm || a->rotary) && a->batch * a->seqlen * a->kv_heads >= 1 << 25) return E2H_ERR_BAD_SHAPE;  // threads of the appending kernel
  if (a->q_off + a->heads * a->dim > a->ld || a->k_off + a->kv_heads * a->dim > a->ld || a->v_off + a->kv_heads * a->vdim > a->ld ||
      (a->g_off >= 0 && a->g_off + a->heads * a->vdim > a->ld) || a->out_off + a->heads * a->vdim > a->ld_out)
    return E2H_ERR_BAD_SHAPE;
  if (a->batch * a->seqlen * a->heads > INT32_MAX || a->batch * a->seqlen * a->kv_heads * (a->dim + a->vdim) / 256 > INT32_MAX - 1)
    return E2H_ERR_BAD_SHAPE;
  return E2H_OK;
}

extern "C" int64_t e2h_seq_window_attention_scratch_bytes(const e2h_window_attention_args *a) {
  if (const int rc = check_attention(a)) return rc;
  return step_scratch_bytes(*a, step_splits(*a));
}

extern "C" int e2h_seq_window_attention(const e2h_window_attention_args *a, void *stream) {
  return e2h_seq_window_attention_split(a, nullptr, 0, stream);
}

extern "C" int e2h_seq_window_attention_split(const e2h_window_attention_args *a, void *scratch, int64_t scratch_bytes, void *stream) {
  if (const int rc = check_attention(a)) return rc;
  if (reinterpret_cast<uintptr_t>(scratch) & 3) return E2H_ERR_MISALIGNED;
  hipStream_t s = static_cast<hipStream_t>(stream);
  e2h_window_attention_args v = *a;
  const int64_t most = INT32_MAX / 2;  // no limit, as far as any cache reaches
  v.window = v.window == 0 || v.window > most ? most : v.window;
  v.keep_first = v.keep_first > most ? most : v.keep_first;
  a = &v;
  if (!on_matrix_cores(*a)) {
    launch_rows(*a, s);
    return launch_status();
  }
  const bool vec = a->dim % 8 == 0 && a->vdim % 8 == 0 && a->ld % 8 == 0 && a->q_off % 8 == 0 && (a->g_off < 0 || a->g_off % 4 == 0) &&
                   a->ld_out % 4 == 0 && a->out_off % 4 == 0 && aligned16(a->proj) && aligned16(a->k_cache) && aligned16(a->v_cache) && aligned16(a->out) &&
                   aligned16(a->q_norm) && aligned16(a->k_norm);
  float *const part = static_cast<float *>(scratch);
  if (vec) launch_mfma_by_size<true>(*a, part, scratch_bytes, s);
  else launch_mfma_by_size<false>(*a, part, scratch_bytes, s);
  return launch_status();
}
