// Gated delta rule with short convolutions (e2h_seq_delta).  Per head: S = g S, u = beta (v - S^T k), S = S + k u^T, o = S^T q,
// then RMS norm over the head and a silu gate.
//
// delta_tokens_kernel: one workgroup per (sequence, head) with the head's state in registers.  For a single token it runs the
// convolutions, the unit norms and the gates itself; for more tokens delta_prepare_kernel has put them into scratch memory.
//
// Chunked form (many tokens), float32 matrix cores throughout.  Within a chunk of 64 tokens that starts from state S0, with
// G_t the decay from the chunk's start through token t,
//   u_t + sum_{s<t} beta_t (G_t / G_s) (k_t . k_s) u_s = beta_t (v_t - G_t S0^T k_t)
//   o_t = G_t S0^T q_t + sum_{s<=t} (G_t / G_s) (q_t . k_s) u_s,   S = G_end S0 + sum_s (G_end / G_s) k_s u_s^T
// 1. delta_chunk_kernel, parallel over chunks, everything that needs no state: T = (I + M)^-1 diag(beta) for the strictly lower
//    triangular M above (the four 16 x 16 diagonal blocks by substitution, the others from products of blocks), W = T diag(G) K
//    and U0 = T V, so that u = U0 - W S0, and the masked, decayed products q k^T;
// 2. delta_scan_kernel, one workgroup per (sequence, head, 16 value columns), chunk after chunk: u and q's read-out, then
//    outputs and the next state;
// 3. delta_gate_kernel: RMS norm over the head and the silu gate.
#include "e2h_seq_common.h"

namespace e2h {
namespace {

constexpr int kMaxDim = 256;
constexpr float kUnitEps = 1e-6f;

constexpr int kChunk = 64;  // tokens that the chunked form takes together

struct Prepared {
  float *q, *k;   // unit vectors, q scaled: [rows, kv_heads, dim], or by fragments of matrix operands where tiles > 0 (see head_value)
  float *v;       // [rows, heads, vdim]
  float *beta;    // [rows, heads]
  float *log_g;   // [rows, heads] logarithm of the decay
  int tiles, chunks;  // the chunked form: tiles of 16 channels that hold a head's keys, and chunks of a sequence
};

// Where channel d of token t's query or key stands.  By fragments: [sequence, chunk, head][block of 16 tokens][tile of 16 channels]
// [four channels][token][channel], so that what a wave wants of a tile, lane (c, b4) the channels 4 b4 .. of token c, is one run
// of 1 KB.  From rows of tokens every lane of a quarter wave meets another cache line, and such a load takes the L1 cache 64 clocks
// instead of 16.
__device__ __forceinline__ size_t head_value(const Prepared &o, int b, int t, size_t row, int head, int kvh, int D, int d) {
  if (o.tiles == 0) return (row * kvh + head) * D + d;
  const size_t block = ((static_cast<size_t>(b) * o.chunks + t / kChunk) * kvh + head) * (kChunk / 16) + t % kChunk / 16;
  return ((block * o.tiles + d / 16) * 64 + d % 16 / 4 * 16 + t % 16) * 4 + d % 4;
}

// causal convolution of one channel ending at token t (position pos0 + t), then silu
template <typename T>
__device__ __forceinline__ float conv_silu(const e2h_delta_args &a, size_t row0, int b, int t, int64_t pos0, int64_t first, int64_t col, int ch,
                                           int channels) {
  const T *proj = static_cast<const T *>(a.proj), *tail = static_cast<const T *>(a.tail_in);
  const float *w = a.conv + static_cast<size_t>(ch) * a.taps;
  float acc = 0.f;
  for (int j = 0; j < a.taps; ++j) {
    const int s = t - a.taps + 1 + j;
    const int64_t pos = pos0 + s;
    float x = 0.f;
    if (pos >= first && pos >= 0) x = s >= 0 ? to_f32(proj[(row0 + s) * a.ld + col]) : to_f32(tail[(static_cast<size_t>(b) * a.taps + pos % a.taps) * channels + ch]);
    acc = __builtin_fmaf(w[j], x, acc);
  }
  return silu_f32(acc);
}

__device__ __forceinline__ float delta_log_decay(float a_proj, float a_log, float dt_bias) { return -expf(a_log) * softplus_f32(a_proj + dt_bias); }

// one wave per (token, unit): unit = a query head, a key head, a value head, or (the last one) the per-head gates
template <typename T>
__global__ __launch_bounds__(256) void delta_prepare_kernel(const e2h_delta_args a, Prepared o) {
  const int lane = threadIdx.x & 63;
  const int kvh = static_cast<int>(a.kv_heads), H = static_cast<int>(a.heads), D = static_cast<int>(a.dim), DV = static_cast<int>(a.vdim);
  const int units = 2 * kvh + H + 1, seqlen = static_cast<int>(a.seqlen);
  const int64_t item = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  const int64_t row = item / units;
  if (row >= a.batch * a.seqlen) return;  // whole waves; no barrier below
  const int u = static_cast<int>(item % units);
  const int b = static_cast<int>(row / seqlen), t = static_cast<int>(row % seqlen);
  const size_t row0 = static_cast<size_t>(b) * seqlen;
  const int64_t pos0 = a.input_pos[0], first = a.first ? a.first[b] : 0;
  const int channels = 2 * kvh * D + H * DV;
  const T *proj = static_cast<const T *>(a.proj);
  if (u == units - 1) {
    for (int h = lane; h < H; h += 64) {
      const bool live = pos0 + t >= first;
      o.beta[row * H + h] = live ? sigmoid_f32(to_f32(proj[row * a.ld + a.b_off + h])) : 0.f;
      o.log_g[row * H + h] = live ? delta_log_decay(to_f32(proj[row * a.ld + a.a_off + h]), a.a_log[h], a.dt_bias[h]) : 0.f;
    }
    return;
  }
  const bool is_q = u < kvh, is_k = !is_q && u < 2 * kvh;
  const int head = is_q ? u : is_k ? u - kvh : u - 2 * kvh;
  const int n = is_q || is_k ? D : DV;
  const int ch0 = is_q ? head * D : is_k ? (kvh + head) * D : 2 * kvh * D + head * DV;
  const int64_t col0 = is_q ? a.q_off + static_cast<int64_t>(head) * D : is_k ? a.k_off + static_cast<int64_t>(head) * D : a.v_off + static_cast<int64_t>(head) * DV;
  float x[kMaxDim / 64], ss = 0.f;
#pragma unroll
  for (int i = 0; i < kMaxDim / 64; ++i) {
    const int d = i * 64 + lane;
    x[i] = d < n ? conv_silu<T>(a, row0, b, t, pos0, first, col0 + d, ch0 + d, channels) : 0.f;
    ss = __builtin_fmaf(x[i], x[i], ss);
  }
  float scale = 1.f;
  if (is_q || is_k) {
    scale = 1.0f / sqrtf(wave_add(ss) + kUnitEps);
    if (is_q) scale /= sqrtf(static_cast<float>(D));
  }
  const int padded = o.tiles > 0 ? o.tiles * 16 : n;  // zeros in the head's last tile
#pragma unroll
  for (int i = 0; i < kMaxDim / 64; ++i) {
    const int d = i * 64 + lane;
    if (d < (is_q || is_k ? padded : n)) *(is_q || is_k ? (is_q ? o.q : o.k) + head_value(o, b, t, row, head, kvh, D, d) : o.v + (row * H + head) * DV + d) = x[i] * scale;
  }
  // the last taps - 1 convolution inputs of the call; those from before it (a call shorter than the convolution) are carried over
  if (a.taps > 1 && t >= seqlen - (a.taps - 1)) {
    T *tail = static_cast<T *>(a.tail_out) + static_cast<size_t>(b) * a.taps * channels;
    for (int d = lane; d < n; d += 64) tail[((pos0 + t) % a.taps) * channels + ch0 + d] = proj[row * a.ld + col0 + d];
  }
  if (a.taps > 1 && t == 0) {
    const T *src = static_cast<const T *>(a.tail_in) + static_cast<size_t>(b) * a.taps * channels;
    T *tail = static_cast<T *>(a.tail_out) + static_cast<size_t>(b) * a.taps * channels;
    for (int s = seqlen - (a.taps - 1); s < 0; ++s) {
      if (pos0 + s < 0) continue;
      for (int d = lane; d < n; d += 64) tail[((pos0 + s) % a.taps) * channels + ch0 + d] = src[((pos0 + s) % a.taps) * channels + ch0 + d];
    }
  }
}

// The same for convolutions of up to four taps with everything in multiples of four channels: `cp` lanes (a power of two) hold
// one head's channels, four each, and walk kPrepareRun tokens with the previous inputs in registers.
constexpr int kPrepareRun = 8;
constexpr int kRunPitch = kPrepareRun * 4 + 4;
static_assert(kPrepareRun == 8, "a run of tokens is half a block of 16");

template <typename T>
__global__ __launch_bounds__(256) void delta_prepare4_kernel(const e2h_delta_args a, Prepared o, int cp, int runs) {
  const int kvh = static_cast<int>(a.kv_heads), H = static_cast<int>(a.heads), D = static_cast<int>(a.dim), DV = static_cast<int>(a.vdim);
  const int heads = 2 * kvh + H, per_wave = 64 / cp, groups = (heads + per_wave - 1) / per_wave, seqlen = static_cast<int>(a.seqlen), taps = a.taps;
  const int lane = threadIdx.x & 63;
  const int64_t item = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);  // (sequence, run, group of heads)
  if (item >= a.batch * runs * groups) return;  // whole waves
  const int u = static_cast<int>(item % groups) * per_wave + lane / cp;
  const int64_t br = item / groups;
  const int b = static_cast<int>(br / runs), t_begin = static_cast<int>(br % runs) * kPrepareRun;
  const int t_end = t_begin + kPrepareRun < seqlen ? t_begin + kPrepareRun : seqlen;
  const bool is_q = u < kvh, is_k = !is_q && u < 2 * kvh;
  const int head = is_q ? u : is_k ? u - kvh : u - 2 * kvh, n = is_q || is_k ? D : DV, d = (lane & (cp - 1)) * 4;
  const bool mine = u < heads && d < n;
  const int ch = mine ? (is_q ? head * D : is_k ? (kvh + head) * D : 2 * kvh * D + head * DV) + d : 0;
  const int64_t col = mine ? (is_q ? a.q_off : is_k ? a.k_off : a.v_off) + static_cast<int64_t>(head) * n + d : a.q_off;
  const int64_t pos0 = a.input_pos[0], first = a.first ? a.first[b] : 0;
  const int channels = 2 * kvh * D + H * DV;
  const size_t row0 = static_cast<size_t>(b) * seqlen;
  const T *src = static_cast<const T *>(a.proj) + row0 * a.ld + col;
  const T *tail = static_cast<const T *>(a.tail_in) + static_cast<size_t>(b) * taps * channels + ch;
  __shared__ __attribute__((aligned(16))) float turned[4 * 64 * kRunPitch];
  float *const mem = turned + (threadIdx.x >> 6) * 64 * kRunPitch;
  // where the run's first token goes if it goes by fragments, or 0; a head's last tile is filled with zeros
  const bool by_fragments = o.tiles > 0 && (is_q || is_k) && d < o.tiles * 16;
  const auto place = by_fragments ? reinterpret_cast<unsigned long long>((is_q ? o.q : o.k) + head_value(o, b, t_begin, 0, head, kvh, D, d)) : 0ull;
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  f32x4_t w[4];  // shallower convolutions: zero weights in front
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    w[j] = zero;
    const int jj = j - (4 - taps);
    if (jj >= 0) {
#pragma unroll
      for (int e = 0; e < 4; ++e) w[j][e] = a.conv[static_cast<size_t>(ch + e) * taps + jj];
    }
  }
  Quad<T> x[kPrepareRun + 3];
  bool there[kPrepareRun + 3];
#pragma unroll
  for (int i = 0; i < kPrepareRun + 3; ++i) {
    const int t = t_begin - 3 + i;
    const int64_t pos = pos0 + t;
    there[i] = pos >= first && pos >= 0 && t >= -(taps - 1);
    if (t >= 0) x[i] = load_quad(src + static_cast<int64_t>(t < seqlen ? t : seqlen - 1) * a.ld);
    else x[i] = load_quad(there[i] ? tail + (pos % taps) * channels : src);
  }
#pragma unroll
  for (int i = 0; i < kPrepareRun; ++i) {
    const int t = t_begin + i;
    if (t >= t_end) break;
    f32x4_t y = zero;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (there[i + j]) {
        const f32x4_t v = x[i + j].f32();
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = __builtin_fmaf(w[j][e], v[e], y[e]);
      }
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      y[e] = mine ? fast_silu(y[e]) : 0.f;
      ss = __builtin_fmaf(y[e], y[e], ss);
    }
    for (int off = 1; off < cp; off <<= 1) ss += __shfl_xor(ss, off);
    if (is_q || is_k) y *= is_q ? 1.0f / (sqrtf(ss + kUnitEps) * sqrtf(static_cast<float>(D))) : 1.0f / sqrtf(ss + kUnitEps);
    const size_t row = row0 + t;
    if (place) store4(mem + lane * kRunPitch + i * 4, y);
    else if (mine) store4(is_q || is_k ? (is_q ? o.q : o.k) + (row * kvh + head) * D + d : o.v + (row * H + head) * DV + d, y);
  }
  // a run is half a block's tokens, 128 bytes of each four channels in a row: eight lanes take one of them (by a lane's 16 bytes at a
  // time this kernel took 209 us for 8192 tokens of 64 heads of 128, so 142)
  if (o.tiles > 0) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int from = i * 8 + lane / 8, t = lane % 8;
      float *const to = reinterpret_cast<float *>(__shfl(place, from));
      if (to && t_begin + t < t_end) store4(to + t * 4, load4(mem + from * kRunPitch + t * 4));
    }
  }
  if (taps > 1 && t_end == seqlen && mine) {  // the last taps - 1 inputs, some of them carried over when the call is that short
    T *dst = static_cast<T *>(a.tail_out) + static_cast<size_t>(b) * taps * channels + ch;
#pragma unroll
    for (int i = 0; i < kPrepareRun + 3; ++i) {
      const int t = t_begin - 3 + i;
      if (t < t_end && t >= t_end - (taps - 1) && pos0 + t >= 0)
        *reinterpret_cast<decltype(x[i].raw) *>(dst + ((pos0 + t) % taps) * channels) = x[i].raw;
    }
  }
}

template <typename T>
__global__ __launch_bounds__(256) void delta_gates_kernel(const e2h_delta_args a, Prepared o) {
  const int H = static_cast<int>(a.heads);
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= a.batch * a.seqlen * H) return;
  const int64_t row = i / H;
  const int h = static_cast<int>(i % H);
  const bool live = a.input_pos[0] + row % a.seqlen >= (a.first ? a.first[row / a.seqlen] : 0);
  const T *src = static_cast<const T *>(a.proj) + row * a.ld;
  o.beta[i] = live ? sigmoid_f32(to_f32(src[a.b_off + h])) : 0.f;
  o.log_g[i] = live ? delta_log_decay(to_f32(src[a.a_off + h]), a.a_log[h], a.dt_bias[h]) : 0.f;
}

// RMS norm over the head, norm weight and silu gate of one head's read-out; four columns per lane of wave 0
template <typename T>
__device__ __forceinline__ void gated_norm_store(const e2h_delta_args &a, size_t row, int h, int cg, bool mine, f32x4_t o) {
  const int DV = static_cast<int>(a.vdim);
  const float ss = wave_add(mine ? o[0] * o[0] + o[1] * o[1] + o[2] * o[2] + o[3] * o[3] : 0.f);
  const float inv = a.out_scale / sqrtf(ss / static_cast<float>(DV) + a.eps);
  if (mine) {
    const T *gate = static_cast<const T *>(a.proj) + row * a.ld + a.g_off + static_cast<int64_t>(h) * DV + cg * 4;
    T *dst = static_cast<T *>(a.out) + row * a.ld_out + a.out_off + static_cast<int64_t>(h) * DV + cg * 4;
#pragma unroll
    for (int e = 0; e < 4; ++e) dst[e] = from_f32<T>(o[e] * inv * a.norm_weight[cg * 4 + e] * silu_f32(to_f32(gate[e])));
  }
}

template <typename T, int BLOCK, int RPT, bool ONE>
__global__ __launch_bounds__(BLOCK) void delta_tokens_kernel(const e2h_delta_args a, Prepared p, int cp) {
  __shared__ float sh_q[kMaxDim], sh_k[kMaxDim], sh_red[BLOCK / 64 * 2];
  __shared__ __attribute__((aligned(16))) float sh_v[kMaxDim], sh_u[kMaxDim];
  __shared__ __attribute__((aligned(16))) f32x4_t part_k[BLOCK], part_q[BLOCK];
  const int D = static_cast<int>(a.dim), DV = static_cast<int>(a.vdim), seqlen = ONE ? 1 : static_cast<int>(a.seqlen);
  const int H = static_cast<int>(a.heads), kvh = static_cast<int>(a.kv_heads);
  const int b = blockIdx.x / H, h = blockIdx.x % H, hk = h / (H / kvh);
  const int cg = threadIdx.x & (cp - 1), rg = threadIdx.x / cp, RG = BLOCK / cp;
  const bool col_ok = cg * 4 < DV;
  const int64_t pos0 = a.input_pos[0], first = a.first ? a.first[b] : 0;
  float *st = a.state + (static_cast<size_t>(b) * H + h) * D * DV;
  f32x4_t s[RPT];
#pragma unroll
  for (int i = 0; i < RPT; ++i) {
    const int r = rg + RG * i;
    s[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    if (pos0 > 0 && col_ok && r < D) s[i] = load4_stream(st + static_cast<size_t>(r) * DV + cg * 4);
  }
  const T *proj = static_cast<const T *>(a.proj);
  for (int t = 0; t < seqlen; ++t) {
    const size_t row = static_cast<size_t>(b) * seqlen + t;
    float log_g, beta;
    if (ONE) {
      const int channels = 2 * kvh * D + H * DV;
      float qs = 0.f, ks = 0.f;
      const bool owner = h % (H / kvh) == 0;  // of the shared query/key head's ring slot; nobody reads that slot in this call
      const uint32_t taps = static_cast<uint32_t>(a.taps), at = static_cast<uint32_t>(pos0 > 0 ? pos0 : 0);
      T *slot = static_cast<T *>(a.tail_out) + (static_cast<size_t>(b) * a.taps + at % taps) * channels;
      size_t kept[3];  // ring rows of the three tokens before this one
      bool there[3];
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        const int64_t pos = pos0 - 3 + j;
        there[j] = taps > 3u - j && pos >= first && pos >= 0;
        kept[j] = (static_cast<size_t>(b) * a.taps + (there[j] ? static_cast<uint32_t>(pos) % taps : 0u)) * channels;
      }
      for (int i = threadIdx.x; i < 2 * D + DV; i += BLOCK) {  // channels of q, k, v
        const bool is_q = i < D, is_k = !is_q && i < 2 * D;
        const int d = is_q ? i : is_k ? i - D : i - 2 * D;
        const int ch = is_q ? hk * D + d : is_k ? (kvh + hk) * D + d : 2 * kvh * D + h * DV + d;
        const int64_t c0 = is_q ? a.q_off + hk * D + d : is_k ? a.k_off + hk * D + d : a.v_off + static_cast<int64_t>(h) * DV + d;
        float y;
        if (taps <= 4) {  // everything in flight at once
          const T now = proj[row * a.ld + c0];
          const T *tail = static_cast<const T *>(a.tail_in);
          T x[3];
          float w[4];
#pragma unroll
          for (int j = 0; j < 3; ++j) x[j] = *(there[j] ? tail + kept[j] + ch : proj + row * a.ld + c0);
#pragma unroll
          for (int j = 0; j < 4; ++j) w[j] = a.conv[static_cast<size_t>(ch) * taps + (j + taps >= 4u ? j + taps - 4u : 0u)];
          y = w[3] * to_f32(now);
#pragma unroll
          for (int j = 0; j < 3; ++j) y = __builtin_fmaf(w[j], there[j] ? to_f32(x[j]) : 0.f, y);
          y = silu_f32(y);
          if (taps > 1 && (owner || !(is_q || is_k))) slot[ch] = now;
        } else {
          y = conv_silu<T>(a, row, b, 0, pos0, first, c0, ch, channels);
          if (owner || !(is_q || is_k)) slot[ch] = proj[row * a.ld + c0];
        }
        if (is_q) qs = __builtin_fmaf(y, y, qs);
        if (is_k) ks = __builtin_fmaf(y, y, ks);
        (is_q ? sh_q : is_k ? sh_k : sh_v)[d] = y;
      }
      qs = wave_add(qs);
      ks = wave_add(ks);
      if ((threadIdx.x & 63) == 0) {
        sh_red[(threadIdx.x >> 6) * 2] = qs;
        sh_red[(threadIdx.x >> 6) * 2 + 1] = ks;
      }
      __syncthreads();
      qs = ks = 0.f;
#pragma unroll
      for (int w = 0; w < BLOCK / 64; ++w) {
        qs += sh_red[2 * w];
        ks += sh_red[2 * w + 1];
      }
      qs = 1.0f / (sqrtf(qs + kUnitEps) * sqrtf(static_cast<float>(D)));
      ks = 1.0f / sqrtf(ks + kUnitEps);
      for (int i = threadIdx.x; i < D; i += BLOCK) {
        sh_q[i] *= qs;
        sh_k[i] *= ks;
      }
      const bool live = pos0 >= first;
      log_g = live ? delta_log_decay(to_f32(proj[row * a.ld + a.a_off + h]), a.a_log[h], a.dt_bias[h]) : 0.f;
      beta = live ? sigmoid_f32(to_f32(proj[row * a.ld + a.b_off + h])) : 0.f;
    } else {
      for (int i = threadIdx.x; i < D; i += BLOCK) {
        sh_q[i] = p.q[(row * kvh + hk) * D + i];
        sh_k[i] = p.k[(row * kvh + hk) * D + i];
      }
      for (int i = threadIdx.x; i < DV; i += BLOCK) sh_v[i] = p.v[(row * H + h) * DV + i];
      log_g = p.log_g[row * H + h];
      beta = p.beta[row * H + h];
    }
    __syncthreads();
    const Decay g = decay_of(expf(log_g), -expm1f(log_g));
    // both read-outs of the decayed state in one pass: (S + k u^T)^T q = S^T q + (k . q) u
    f32x4_t ak = {0.f, 0.f, 0.f, 0.f}, aq = ak;
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
      const int r = rg + RG * i;
      if (r < D) {
        const float k = sh_k[r], q = sh_q[r];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          s[i][e] = decayed(g, s[i][e]);
          ak[e] = __builtin_fmaf(k, s[i][e], ak[e]);
          aq[e] = __builtin_fmaf(q, s[i][e], aq[e]);
        }
      }
    }
    part_k[threadIdx.x] = ak;
    part_q[threadIdx.x] = aq;
    __syncthreads();
    if (threadIdx.x < 64) {  // all column groups of the head lie in wave 0
      float kq = 0.f;
      for (int i = threadIdx.x; i < D; i += 64) kq = __builtin_fmaf(sh_k[i], sh_q[i], kq);
      kq = wave_add(kq);
      const bool mine = threadIdx.x < cp && col_ok;
      f32x4_t o = {0.f, 0.f, 0.f, 0.f};
      if (mine) {
        f32x4_t u = o;
        for (int j = 0; j < RG; ++j) {
          u += part_k[j * cp + threadIdx.x];
          o += part_q[j * cp + threadIdx.x];
        }
        u = (load4(sh_v + cg * 4) - u) * beta;
        store4(sh_u + cg * 4, u);
        o += u * kq;
      }
      gated_norm_store<T>(a, row, h, cg, mine, o);
    }
    __syncthreads();
    if (col_ok) {
      const f32x4_t u = load4(sh_u + cg * 4);
#pragma unroll
      for (int i = 0; i < RPT; ++i) {
        const int r = rg + RG * i;
        if (r < D) {
          const float k = sh_k[r];
#pragma unroll
          for (int e = 0; e < 4; ++e) s[i][e] = __builtin_fmaf(k, u[e], s[i][e]);
        }
      }
    }
    if (!ONE) __syncthreads();  // k and u are read before the next token replaces them
  }
#pragma unroll
  for (int i = 0; i < RPT; ++i) {
    const int r = rg + RG * i;
    if (col_ok && r < D) store4_stream(st + static_cast<size_t>(r) * DV + cg * 4, s[i]);
  }
}

// ---- chunked form ----------------------------------------------------------------------------------------------------------
struct ChunkScratch {
  float *w;     // [batch * heads, chunks] by fragments as the keys
  float *p;     // [batch * heads, chunks] by fragments, four tiles
  float *g, *e; // [batch * heads, chunks, 64] decay from the chunk's start through the token, and from the token to the chunk's end
};

// step 1: 4 waves, one (sequence, head, chunk) each; wave w owns the token rows 16 w .. 16 w + 15.  TILES: tiles of 16 that hold a
// head's keys and its values.  U0 takes the place of the values.  Products are formed turned, a lane its token's row of four keys:
// that is both the layout of the left operand that M's blocks become and 16 bytes of a fragment.
// What bounds it: 76 us of float32 matrix work and 560 MB at 8192 tokens of 32 heads of 128, with phases that wait for one another;
// 52 KB of LDS and 112 registers let three workgroups of a CU overlap theirs.  290 us with M in LDS and two workgroups, 190 so; the
// two products that it took over from the scan cost it 50.
template <int TILES>
__global__ __launch_bounds__(256, TILES <= 8 ? 3 : 1) void delta_chunk_kernel(const e2h_delta_args a, Prepared p, ChunkScratch cs) {
  constexpr int kRow = kChunk + 4, kWide = TILES * 16 + 4, kQuads = TILES * 4, kEvery = 256 / kQuads;
  __shared__ __attribute__((aligned(16))) float sw[kChunk * kWide];  // keys, then values
  __shared__ __attribute__((aligned(16))) float si[kChunk * kRow];  // inverse; M's diagonal blocks stand in blocks above its diagonal
  __shared__ __attribute__((aligned(16))) float sg[kChunk], sb[kChunk];
  const int D = static_cast<int>(a.dim), DV = static_cast<int>(a.vdim), H = static_cast<int>(a.heads), kvh = static_cast<int>(a.kv_heads), seqlen = static_cast<int>(a.seqlen);
  const int chunk = blockIdx.x % p.chunks, bh = blockIdx.x / p.chunks;
  const int b = bh / H, h = bh % H, hk = h / (H / kvh);
  // the last rows take four times the first ones' products: neighbours on a CU hand them to different SIMDs (205 to 201 us)
  const int wave = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) + blockIdx.x / 8 + blockIdx.x / 256) & 3;
  const int lane = threadIdx.x & 63, c = lane & 15, b4 = lane >> 4;
  const size_t row0 = static_cast<size_t>(b) * seqlen + static_cast<size_t>(chunk) * kChunk;
  const int live = seqlen - chunk * kChunk < kChunk ? seqlen - chunk * kChunk : kChunk;  // tokens past the end: beta 0, decay 1, q = k = 0
  const f32x4_t none = {0.f, 0.f, 0.f, 0.f};
  // tokens past the sequence's end are read from its last one or as whatever the memory holds, and masked when they are used: no
  // load waits in a branch
  const size_t gate_row = (row0 + (lane < live ? lane : live - 1)) * H + h;
  const float log_g = p.log_g[gate_row], beta = p.beta[gate_row];
  f32x4_t mine[TILES], query[TILES];  // this wave's rows of keys and queries
  const size_t head = (((static_cast<size_t>(b) * p.chunks + chunk) * kvh + hk) * (kChunk / 16) + wave) * p.tiles * 256 + lane * 4;
  const int tr = 16 * wave + c;
#pragma unroll
  for (int dt = 0; dt < TILES; ++dt) {
    const int there = dt < p.tiles ? dt : p.tiles - 1;
    mine[dt] = load4(p.k + head + there * 256);
    query[dt] = load4(p.q + head + there * 256);
  }
  if (threadIdx.x < 64) {
    const int t = threadIdx.x;
    float g = t < live ? log_g : 0.f;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const float up = __shfl_up(g, off);
      if (t >= off) g += up;
    }
    sg[t] = g * kLog2e;
    sb[t] = t < live ? beta : 0.f;
  }
#pragma unroll
  for (int dt = 0; dt < TILES; ++dt) {
    const bool there = tr < live && dt < p.tiles;
    mine[dt] = there ? mine[dt] : none;
    query[dt] = there ? query[dt] : none;
    store4(sw + tr * kWide + dt * 16 + 4 * b4, mine[dt]);
  }
  lds_barrier();
  // M's blocks left of the diagonal, and q k^T for the blocks up to it
  f32x4_t m[4];
  float *pt = cs.p + (static_cast<size_t>(bh) * p.chunks + chunk) * kChunk * kChunk + wave * 1024 + lane * 4;
  const float g_mine = sg[tr], b_mine = sb[tr];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    m[j] = none;
    if (j > wave) continue;
    f32x4_t kk = none, kq = none;
#pragma unroll
    for (int dt = 0; dt < TILES; ++dt) {
      const f32x4_t kc = load4(sw + (16 * j + c) * kWide + dt * 16 + 4 * b4);
      kk = mfma4(kc, mine[dt], kk);
      kq = mfma4(kc, query[dt], kq);
    }
    const f32x4_t g = load4(sg + 16 * j + 4 * b4);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int key = 16 * j + 4 * b4 + r;
      const float dec = __builtin_amdgcn_exp2f(key <= tr ? g_mine - g[r] : -INFINITY);
      m[j][r] = key < tr ? b_mine * dec * kk[r] : 0.f;
      kq[r] *= dec;
    }
    store4(pt + j * 256, kq);
  }
  // inverse of the unit lower triangular diagonal blocks: wave w, lane c = column c of block w, substitution down the rows
  float *const diagonal = si + (wave < 3 ? 16 * wave * kRow + 16 * (wave + 1) : 32);
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (j == wave) store4(diagonal + c * kRow + 4 * b4, m[j]);
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  if (b4 == 0) {
    f32x4_t row[2][4];  // of this step and the next
    float x[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) {
#pragma unroll
      for (int s = 0; s < 4; ++s)
        if (t < 15 && 4 * s <= t) row[(t + 1) & 1][s] = load4(diagonal + (t + 1) * kRow + 4 * s);
      float v = t == c ? 1.f : 0.f;
#pragma unroll
      for (int s = 0; s < 16; ++s)
        if (s < t) v = __builtin_fmaf(-row[t & 1][s / 4][s % 4], x[s], v);
      x[t] = v;
      si[(16 * wave + t) * kRow + 16 * wave + c] = v;
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  lds_barrier();
  // the values in whole rows, a thread four columns of every kEvery-th token, are wanted behind the products of the keys
  const int vt = threadIdx.x / kQuads, vd = threadIdx.x % kQuads * 4;
  f32x4_t val[kChunk / kEvery];
#pragma unroll
  for (int i = 0; i < kChunk / kEvery; ++i) {
    const int t = vt + i * kEvery;
    val[i] = load4(p.v + ((row0 + (t < live ? t : live - 1)) * H + h) * DV + (vd < DV ? vd : 0));
  }
  // blocks off the diagonal, by distance: I_ij = -I_ii sum_{j <= l < i} M_il I_lj
#pragma unroll
  for (int dist = 1; dist < 4; ++dist) {
    const int i = wave, j = wave - dist;
    f32x4_t acc = none;
    if (j >= 0) {
#pragma unroll
      for (int l = 0; l < 3; ++l) {
        if (l < j || l >= i) continue;
        f32x4_t bb;
#pragma unroll
        for (int r = 0; r < 4; ++r) bb[r] = si[(16 * l + 4 * b4 + r) * kRow + 16 * j + c];
        acc = mfma4(m[l], bb, acc);
      }
      const f32x4_t res = mfma4(load4(si + (16 * i + c) * kRow + 16 * i + 4 * b4), acc, none);
#pragma unroll
      for (int r = 0; r < 4; ++r) si[(16 * i + 4 * b4 + r) * kRow + 16 * j + c] = -res[r];
    }
    lds_barrier();
  }
  const size_t at = static_cast<size_t>(bh) * p.chunks + chunk;
  if (threadIdx.x < kChunk) {
    cs.g[at * kChunk + threadIdx.x] = __builtin_amdgcn_exp2f(sg[threadIdx.x]);
    cs.e[at * kChunk + threadIdx.x] = __builtin_amdgcn_exp2f(sg[kChunk - 1] - sg[threadIdx.x]);
  }
  // rows 16 w .. of (I + M)^-1 diag(coefficient), which multiply the rows in sw, two tiles of columns at a time
  f32x4_t inv[4], by[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    inv[j] = by[j] = none;
    if (j > wave) continue;
    const f32x4_t g = load4(sg + 16 * j + 4 * b4);
    by[j] = load4(si + tr * kRow + 16 * j + 4 * b4) * load4(sb + 16 * j + 4 * b4);
#pragma unroll
    for (int r = 0; r < 4; ++r) inv[j][r] = by[j][r] * __builtin_amdgcn_exp2f(g[r]);
  }
  const auto column = [&](int j, int tile) {
    f32x4_t x;
#pragma unroll
    for (int r = 0; r < 4; ++r) x[r] = sw[(16 * j + 4 * b4 + r) * kWide + tile * 16 + c];
    return x;
  };
  float *wt = cs.w + at * kChunk * 16 * p.tiles + wave * p.tiles * 256 + lane * 4;
  for (int tile = 0; tile < p.tiles; tile += 2) {
    f32x4_t w0 = none, w1 = none;  // turned
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j <= wave) {
        w0 = mfma4(column(j, tile), inv[j], w0);
        w1 = mfma4(column(j, tile + 1), inv[j], w1);
      }
    store4(wt + tile * 256, w0);
    if (tile + 1 < p.tiles) store4(wt + tile * 256 + 256, w1);
  }
  lds_barrier();  // the keys have been read
#pragma unroll
  for (int i = 0; i < kChunk / kEvery; ++i) store4(sw + (vt + i * kEvery) * kWide + vd, vt + i * kEvery < live && vd < DV ? val[i] : none);
  lds_barrier();
  float *const u_at = p.v + ((row0 + 16 * wave + 4 * b4) * H + h) * DV + c;
  const size_t u_stride = static_cast<size_t>(H) * DV;
  for (int tile = 0; tile * 16 < DV; tile += 2) {
    f32x4_t u0 = none, u1 = none;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j <= wave) {
        u0 = mfma4(by[j], column(j, tile), u0);
        u1 = mfma4(by[j], column(j, tile + 1), u1);
      }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (16 * wave + 4 * b4 + r >= live) continue;
      if (tile * 16 + c < DV) u_at[r * u_stride + tile * 16] = u0[r];
      if (tile * 16 + 16 + c < DV) u_at[r * u_stride + tile * 16 + 16] = u1[r];
    }
  }
}

// step 2: DT = head dimension in tiles of 16.  Eight waves: wave w < 4 owns the token rows 16 w .. 16 w + 15 on the writing side
// (u = U0 - W S0), wave w + 4 the same rows on the reading side (q and the outputs); the state's row tiles w, w + 8
// are wave w's.  The state is kept twice: in accumulators by its owner, and in LDS, transposed, as the B operand of
// everybody's read-outs.  The keys, decayed to the chunk's end, go through LDS once to be read transposed in the state update.
// What bounds it: one workgroup per CU of dependent chunks (32 heads of 128 values, one sequence), each two matrix phases in
// float32 with a barrier behind either, 2048 and up to 1536 matrix clocks a SIMD of the 6600 that a chunk takes, and 112 KB that
// pass the L1 cache at 64 bytes a clock (1800).  All of it comes by fragments, 1 KB to a load: from rows of tokens a chunk took
// 1.0 us more, and 1.2 us more with the loads in one block ahead of the products instead of between them.  With T applied here
// (u = T (v - G S0^T k), a phase and a barrier more), decays formed by every lane, sums by single LDS words and rows of
// tokens, 8192 tokens took 709 us; now 400.
// WHOLE: the head dimension fills its tiles, so that every tile's place is a constant from the first one's.
template <int DT, bool WHOLE>
__global__ __launch_bounds__(512) void delta_scan_kernel(const e2h_delta_args a, Prepared p, ChunkScratch cs, int v_blocks) {
  constexpr int DP = DT * 16, OWN = (DT + 7) / 8, kRow = DP + 4, kTok = kChunk + 4;
  constexpr bool kTwo = DT <= 8;  // the next chunk's rows are requested between this one's products; two sets of more do not fit the registers
  __shared__ __attribute__((aligned(16))) float st[16 * kRow];       // state, [value column][row]
  __shared__ __attribute__((aligned(16))) float sk[kChunk * kRow];   // keys, [token][channel]
  __shared__ __attribute__((aligned(16))) float su[16 * kTok];       // u, [value column][token]
  const int D = static_cast<int>(a.dim), DV = static_cast<int>(a.vdim), H = static_cast<int>(a.heads), kvh = static_cast<int>(a.kv_heads);
  const int seqlen = static_cast<int>(a.seqlen), bh_count = static_cast<int>(a.batch) * H;
  // the value blocks of one head read the same keys and queries: keep them on one die (workgroups go round robin over 8)
  int bh, vb;
  const int whole = bh_count / 8 * 8 * v_blocks;
  if (static_cast<int>(blockIdx.x) < whole) {
    const int die = blockIdx.x & 7, i = blockIdx.x >> 3;
    bh = (i / v_blocks) * 8 + die;
    vb = i % v_blocks;
  } else {
    bh = bh_count / 8 * 8 + (blockIdx.x - whole) / v_blocks;
    vb = (blockIdx.x - whole) % v_blocks;
  }
  const int b = bh / H, h = bh % H, hk = h / (H / kvh);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = threadIdx.x & 15, b4 = (threadIdx.x & 63) >> 4;
  const bool reader = wave >= 4;
  const int block = wave & 3;  // of 16 tokens
  const int col = vb * 16 + c;
  const bool col_ok = col < DV;
  float *state = a.state + static_cast<size_t>(bh) * D * DV;
  const bool carried = a.input_pos[0] > 0;
  f32x4_t s[OWN];
#pragma unroll
  for (int i = 0; i < OWN; ++i) {
    const int dt = wave + 8 * i;
    s[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int d = dt * 16 + 4 * b4 + r;
      if (carried && d < D && col_ok) s[i][r] = state[static_cast<size_t>(d) * DV + col];
    }
    if (dt < DT) store4(st + c * kRow + dt * 16 + 4 * b4, s[i]);
  }
  const int tr = 16 * block + c, half = reader ? DT / 2 : 0;  // first tile of the keys that this wave brings
  const size_t seq0 = static_cast<size_t>(b) * seqlen, first_chunk = static_cast<size_t>(bh) * p.chunks;

  // a chunk's place is uniform, a lane's part of it one offset of 32 bits
  const uint32_t v_stride = static_cast<uint32_t>(H) * static_cast<uint32_t>(DV), lane4 = static_cast<uint32_t>(threadIdx.x & 63) * 4;
  const uint32_t my_rows = static_cast<uint32_t>(block * p.tiles) * 256 + lane4, my_square = static_cast<uint32_t>(block) * 1024 + lane4;
  const uint32_t my_v = static_cast<uint32_t>(16 * block + 4 * b4) * v_stride, my_col = col_ok ? col : 0;
  const size_t head_size = static_cast<size_t>(kChunk) * 16 * p.tiles;
  const auto head_at = [&](int chunk) { return ((static_cast<size_t>(b) * p.chunks + chunk) * kvh + hk) * head_size; };
  // a tile of this wave's 16 tokens; rows past the sequence's end are whatever the memory holds, tiles past the head's last one that one again: they
  // meet the state's zeros, since keys are put away as zeros there.  Nothing is masked on arrival: that would wait for each load in turn.
  const f32x4_t none = {0.f, 0.f, 0.f, 0.f};
  const auto tile = [&](const float *from, int dt) { return load4(from + (my_rows + (WHOLE || dt < p.tiles ? dt : p.tiles - 1) * 256)); };
  // rows of W or of q; of dead tokens: u that is set to zero, and outputs that are not stored
  const auto rows_of = [&](int chunk) { return reader ? p.q + head_at(chunk) : cs.w + (first_chunk + chunk) * head_size; };
  f32x4_t key[DT / 2], square[4], v = none, g = none;  // v: writers, square and g: readers
  float e, decay;
  const auto bring_keys = [&](int chunk) {
    const size_t at = first_chunk + chunk;
    const float *const keys = p.k + head_at(chunk);
    e = cs.e[at * kChunk + tr];
    decay = cs.g[at * kChunk + kChunk - 1];
    if (reader) {
      g = load4(cs.g + at * kChunk + (16 * block + 4 * b4));
    } else {
      const float *const values = p.v + ((seq0 + static_cast<size_t>(chunk) * kChunk) * H + h) * DV;
      const uint32_t last = static_cast<uint32_t>(seqlen - chunk * kChunk < kChunk ? seqlen - chunk * kChunk : kChunk) - 1;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const uint32_t t = my_v + r * v_stride;
        v[r] = values[(t < last * v_stride ? t : last * v_stride) + my_col];
      }
    }
#pragma unroll
    for (int i = 0; i < DT / 2; ++i) key[i] = tile(keys, half + i);
  };
  const auto bring_square = [&](int chunk) {
    const float *const from = cs.p + (first_chunk + chunk) * kChunk * kChunk;
#pragma unroll
    for (int j = 0; j < 4; ++j) square[j] = load4(from + (my_square + 256 * j));
  };

  const auto step = [&](int chunk, f32x4_t (&cur)[DT], f32x4_t (&next)[DT]) {
    const int live = seqlen - chunk * kChunk < kChunk ? seqlen - chunk * kChunk : kChunk;
    const int after = chunk + 1 < p.chunks ? chunk + 1 : chunk;
    const float *const next_rows = rows_of(after);
    f32x4_t y = none;  // W S0 or S0^T q
    f32x4_t sf[DT];
    sf[0] = load4(st + c * kRow + 4 * b4);
    sf[1] = load4(st + c * kRow + 16 + 4 * b4);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      if (kTwo) next[dt] = tile(next_rows, dt);
      if (dt + 2 < DT) sf[dt + 2] = load4(st + c * kRow + (dt + 2) * 16 + 4 * b4);
      y = mfma4(cur[dt], sf[dt], y);
      __builtin_amdgcn_sched_barrier(0);
    }
    const float into = decay;
    if (reader) {
      y *= g;
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) y[r] = 16 * block + 4 * b4 + r < live ? v[r] - y[r] : 0.f;
      store4(su + c * kTok + 16 * block + 4 * b4, y);
    }
#pragma unroll
    for (int i = 0; i < DT / 2; ++i) store4(sk + tr * kRow + (half + i) * 16 + 4 * b4, tr < live && (WHOLE || half + i < p.tiles) ? key[i] * e : none);
    lds_barrier();  // u and the keys are in LDS, the state has been read; the loads above stay in flight
    bring_keys(after);
    if (!kTwo) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) next[dt] = tile(next_rows, dt);
    }
    f32x4_t u[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) u[j] = load4(su + c * kTok + 16 * j + 4 * b4);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < OWN; ++i) {
      if (wave + 8 * i >= DT) break;
      s[i] *= into;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        f32x4_t kt;
#pragma unroll
        for (int r = 0; r < 4; ++r) kt[r] = sk[(16 * j + 4 * b4 + r) * kRow + (wave + 8 * i) * 16 + c];
        s[i] = mfma4(kt, u[j], s[i]);
      }
      store4(st + c * kRow + (wave + 8 * i) * 16 + 4 * b4, s[i]);
    }
    if (reader) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (j <= block) y = mfma4(square[j], u[j], y);
      bring_square(after);
      float *const out = p.v + ((seq0 + static_cast<size_t>(chunk) * kChunk) * H + h) * DV;
#pragma unroll
      for (int r = 0; r < 4; ++r)  // over the values this workgroup has read
        if (16 * block + 4 * b4 + r < live && col_ok) out[my_v + r * v_stride + my_col] = y[r];
    }
    lds_barrier();  // the next state is in LDS, and the keys and u have been read
  };
  f32x4_t even[DT], odd[kTwo ? DT : 1];
  {
    const float *const rows = rows_of(0);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) even[dt] = tile(rows, dt);
  }
  bring_keys(0);
  if (reader) bring_square(0);
  lds_barrier();
  if constexpr (kTwo) {
#pragma unroll 1
    for (int chunk = 0; chunk < p.chunks; chunk += 2) {
      step(chunk, even, odd);
      if (chunk + 1 < p.chunks) step(chunk + 1, odd, even);
    }
  } else {
#pragma unroll 1
    for (int chunk = 0; chunk < p.chunks; ++chunk) step(chunk, even, even);
  }
#pragma unroll
  for (int i = 0; i < OWN; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int d = (wave + 8 * i) * 16 + 4 * b4 + r;
      if (d < D && col_ok) state[static_cast<size_t>(d) * DV + col] = s[i][r];
    }
}

// step 3: `cp` lanes per (token, head), four columns each; the read-outs stand where the values were
template <typename T>
__global__ __launch_bounds__(256) void delta_gate_kernel(const e2h_delta_args a, Prepared p, int cp) {
  const int64_t item = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) / cp;
  const int d = static_cast<int>(threadIdx.x & (cp - 1)) * 4, DV = static_cast<int>(a.vdim), H = static_cast<int>(a.heads);
  const bool mine = d < DV && item < a.batch * a.seqlen * H;
  const int64_t row = mine ? item / H : 0;
  const int h = mine ? static_cast<int>(item % H) : 0, dc = mine ? d : 0;
  const f32x4_t o = load4(p.v + (row * H + h) * DV + dc), w = load4(a.norm_weight + dc);
  const f32x4_t gate = load4(static_cast<const T *>(a.proj) + row * a.ld + a.g_off + static_cast<int64_t>(h) * DV + dc);
  float ss = mine ? o[0] * o[0] + o[1] * o[1] + o[2] * o[2] + o[3] * o[3] : 0.f;
  for (int off = 1; off < cp; off <<= 1) ss += __shfl_xor(ss, off);
  const float inv = a.out_scale / sqrtf(ss / static_cast<float>(DV) + a.eps);
  if (!mine) return;
  f32x4_t y;
#pragma unroll
  for (int e = 0; e < 4; ++e) y[e] = o[e] * inv * w[e] * fast_silu(gate[e]);
  store4(static_cast<T *>(a.out) + row * a.ld_out + a.out_off + static_cast<int64_t>(h) * DV + d, y);
}

int lanes_for(int64_t values) {  // power of two, four values per lane
  int cp = 1;
  while (cp * 4 < values) cp *= 2;
  return cp;
}

// four channels per access everywhere
bool quads_ok(const e2h_delta_args &a) {
  return a.dim % 4 == 0 && a.ld % 4 == 0 && a.q_off % 4 == 0 && a.k_off % 4 == 0 && a.v_off % 4 == 0 && a.g_off % 4 == 0 && a.ld_out % 4 == 0 &&
         a.out_off % 4 == 0 && aligned16(a.proj) && aligned16(a.tail_in) && aligned16(a.tail_out) && aligned16(a.out) && aligned16(a.norm_weight);
}

// Chunks from 24 tokens on, where token by token loses even with the chip full of sequences: us, tokens / chunks, 16 sequences of 32 heads of 128: 16 tokens 93 / 131, 20 114 / 133,
// 24 133 / 134, 32 169 / 135, 63 306 / 145; one sequence of them 16 tokens 90 / 38, 24 128 / 39, 63 305 / 40.  (The scan counts a chunk's values in 31 bits.)
bool use_chunks(const e2h_delta_args &a) {
  if (a.seqlen == 1 || seq_options().recurrence_form == 1 || !quads_ok(a) || a.heads * a.vdim > INT32_MAX / kChunk) return false;
  return seq_options().recurrence_form == 2 || a.seqlen >= 24;
}

template <int DT>
void launch_scan(const e2h_delta_args &a, const Prepared &p, const ChunkScratch &cs, hipStream_t s) {
  const int v_blocks = static_cast<int>((a.vdim + 15) / 16);
  const dim3 grid(static_cast<unsigned>(a.batch * a.heads * v_blocks)), block(512);
  if (a.dim == DT * 16) hipLaunchKernelGGL((delta_scan_kernel<DT, true>), grid, block, 0, s, a, p, cs, v_blocks);
  else hipLaunchKernelGGL((delta_scan_kernel<DT, false>), grid, block, 0, s, a, p, cs, v_blocks);
}

template <typename T>
void launch_chunks(const e2h_delta_args &a, const Prepared &p, const ChunkScratch &cs, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(a.batch * a.heads * p.chunks)), block(256);
  const int64_t widest = a.dim > a.vdim ? a.dim : a.vdim;
  if (widest <= 64) hipLaunchKernelGGL(delta_chunk_kernel<4>, grid, block, 0, s, a, p, cs);
  else if (widest <= 128) hipLaunchKernelGGL(delta_chunk_kernel<8>, grid, block, 0, s, a, p, cs);
  else hipLaunchKernelGGL(delta_chunk_kernel<16>, grid, block, 0, s, a, p, cs);
  if (a.dim <= 64) launch_scan<4>(a, p, cs, s);
  else if (a.dim <= 128) launch_scan<8>(a, p, cs, s);
  else launch_scan<16>(a, p, cs, s);
  const int cp = lanes_for(a.vdim);
  hipLaunchKernelGGL(delta_gate_kernel<T>, dim3(static_cast<unsigned>((a.batch * a.seqlen * a.heads * cp + 255) / 256)), block, 0, s, a, p, cp);
}

template <typename T, bool ONE>
void launch_tokens(const e2h_delta_args &a, const Prepared &p, hipStream_t s) {
  int cp = 1;
  while (cp * 4 < a.vdim) cp *= 2;
  const dim3 grid(static_cast<unsigned>(a.batch * a.heads));
  const int64_t need = (a.dim * cp + 255) / 256;  // rows per thread with 256 threads
  if (need <= 4) hipLaunchKernelGGL((delta_tokens_kernel<T, 256, 4, ONE>), grid, dim3(256), 0, s, a, p, cp);
  else if (need <= 16) hipLaunchKernelGGL((delta_tokens_kernel<T, 256, 16, ONE>), grid, dim3(256), 0, s, a, p, cp);
  else hipLaunchKernelGGL((delta_tokens_kernel<T, 1024, 16, ONE>), grid, dim3(1024), 0, s, a, p, cp);
}

int64_t round256(int64_t n) { return (n + 255) / 256 * 256; }

// scratch layout; returns its size in bytes
int64_t carve(const e2h_delta_args &a, Prepared *p, ChunkScratch *cs) {
  if (a.seqlen == 1) return 0;
  const bool chunked = use_chunks(a);
  const int64_t rows = a.batch * a.seqlen, chunks = (a.seqlen + kChunk - 1) / kChunk, tiles = (a.dim + 15) / 16;
  const int64_t qk = round256((chunked ? a.batch * chunks * kChunk * a.kv_heads * tiles * 16 : rows * a.kv_heads * a.dim) * 4);
  const int64_t v = round256(rows * a.heads * a.vdim * 4), g = round256(rows * a.heads * 4);
  if (p) {
    uint8_t *base = static_cast<uint8_t *>(a.scratch);
    p->q = reinterpret_cast<float *>(base);
    p->k = reinterpret_cast<float *>(base + qk);
    p->v = reinterpret_cast<float *>(base + 2 * qk);
    p->beta = reinterpret_cast<float *>(base + 2 * qk + v);
    p->log_g = reinterpret_cast<float *>(base + 2 * qk + v + g);
    p->tiles = chunked ? static_cast<int>(tiles) : 0;
    p->chunks = static_cast<int>(chunks);
  }
  const int64_t prepared = 2 * qk + v + 2 * g;
  if (!chunked) return prepared;
  const int64_t gates = a.batch * a.heads * chunks * kChunk * 4, w = gates * tiles * 16, squares = gates * kChunk;
  if (cs) {
    uint8_t *base = static_cast<uint8_t *>(a.scratch) + prepared;
    cs->w = reinterpret_cast<float *>(base);
    cs->p = reinterpret_cast<float *>(base + w);
    cs->g = reinterpret_cast<float *>(base + w + squares);
    cs->e = reinterpret_cast<float *>(base + w + squares + gates);
  }
  return prepared + w + squares + 2 * gates;
}

template <typename T>
int launch_delta(const e2h_delta_args &a, hipStream_t s) {
  Prepared p = {};
  if (a.seqlen == 1) {
    launch_tokens<T, true>(a, p, s);
    return launch_status();
  }
  ChunkScratch cs = {};
  carve(a, &p, &cs);
  if (a.taps <= 4 && quads_ok(a)) {
    const int64_t widest = a.dim > a.vdim ? a.dim : a.vdim;
    const int cp = lanes_for(p.tiles > 0 && widest < 16 ? 16 : widest), runs = static_cast<int>((a.seqlen + kPrepareRun - 1) / kPrepareRun);
    const int64_t waves = a.batch * runs * ((2 * a.kv_heads + a.heads + 64 / cp - 1) / (64 / cp));
    hipLaunchKernelGGL(delta_prepare4_kernel<T>, dim3(static_cast<unsigned>((waves + 3) / 4)), dim3(256), 0, s, a, p, cp, runs);
    hipLaunchKernelGGL(delta_gates_kernel<T>, dim3(static_cast<unsigned>((a.batch * a.seqlen * a.heads + 255) / 256)), dim3(256), 0, s, a, p);
  } else {
    const int64_t items = a.batch * a.seqlen * (2 * a.kv_heads + a.heads + 1);
    hipLaunchKernelGGL(delta_prepare_kernel<T>, dim3(static_cast<unsigned>((items + 3) / 4)), dim3(256), 0, s, a, p);
  }
  if (use_chunks(a)) launch_chunks<T>(a, p, cs, s);
  else launch_tokens<T, false>(a, p, s);
  return launch_status();
}

bool shape_ok(const e2h_delta_args &a) {
  if (a.dtype != E2H_SEQ_BF16 && a.dtype != E2H_SEQ_F32) return false;
  if (a.batch < 1 || a.seqlen < 1 || a.heads < 1 || a.kv_heads < 1 || a.heads % a.kv_heads != 0 || a.dim < 1 || a.dim > kMaxDim || a.vdim < 4 ||
      a.vdim % 4 != 0 || a.vdim > kMaxDim || a.taps < 1 || a.taps > 64 || a.seqlen > INT32_MAX / 2)
    return false;
  if (a.q_off < 0 || a.k_off < 0 || a.v_off < 0 || a.b_off < 0 || a.a_off < 0 || a.g_off < 0 || a.out_off < 0) return false;
  if (a.q_off + a.kv_heads * a.dim > a.ld || a.k_off + a.kv_heads * a.dim > a.ld || a.v_off + a.heads * a.vdim > a.ld || a.b_off + a.heads > a.ld ||
      a.a_off + a.heads > a.ld || a.g_off + a.heads * a.vdim > a.ld || a.out_off + a.heads * a.vdim > a.ld_out)
    return false;
  return a.batch * a.heads * ((a.seqlen + kChunk - 1) / kChunk) <= INT32_MAX && a.batch * a.heads * ((a.vdim + 15) / 16) <= INT32_MAX &&
         a.batch * a.seqlen * (2 * a.kv_heads + a.heads + 1) / 4 < INT32_MAX &&
         2 * a.kv_heads * a.dim + a.heads * a.vdim <= INT32_MAX;
}

}  // namespace
}  // namespace e2h

using namespace e2h;

extern "C" int64_t e2h_seq_delta_scratch_bytes(const e2h_delta_args *a) {
  if (!a) return E2H_ERR_NULL_POINTER;
  if (!shape_ok(*a)) return E2H_ERR_BAD_SHAPE;
  return carve(*a, nullptr, nullptr);
}

extern "C" int e2h_seq_delta(const e2h_delta_args *a, void *stream) {
  if (!a || !a->proj || !a->conv || !a->a_log || !a->dt_bias || !a->norm_weight || !a->state || !a->input_pos || !a->out) return E2H_ERR_NULL_POINTER;
  if (!shape_ok(*a)) return E2H_ERR_BAD_SHAPE;
  if (a->taps > 1 && (!a->tail_in || !a->tail_out)) return E2H_ERR_NULL_POINTER;
  if (a->taps > 1 && a->seqlen > 1 && a->tail_in == a->tail_out) return E2H_ERR_BAD_SHAPE;
  if (!aligned16(a->state) || !aligned16(a->scratch)) return E2H_ERR_MISALIGNED;
  const int64_t need = carve(*a, nullptr, nullptr);
  if (need > 0 && !a->scratch) return E2H_ERR_NULL_POINTER;
  if (need > a->scratch_bytes) return E2H_ERR_SCRATCH_TOO_SMALL;
  if (a->dtype == E2H_SEQ_BF16) return launch_delta<bf16_t>(*a, static_cast<hipStream_t>(stream));
  return launch_delta<float>(*a, static_cast<hipStream_t>(stream));
}
