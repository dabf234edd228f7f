// Row kernels of the stateful decoder layers: residual add of a normalised sublayer output, the next sublayer's norm and
// its input convolution over time in one pass over the float32 residual stream, and the elementwise steps.
#include <string.h>

#include "e2h_seq_common.h"

namespace e2h {

SeqOptions &seq_options() {
  static SeqOptions o = {};
  return o;
}

namespace {

// One workgroup per run of `run` consecutive tokens of one sequence, NB tokens at a time so that the loads of NB rows are in
// flight together and one barrier serves NB row sums.  A thread owns NP pieces of four channels, so the convolution's previous
// inputs stay in its registers from token to token; the taps - 1 tokens ahead of the run are normalised again by the
// workgroup (inside the call) or come from the ring of kept inputs (before the call).  TAPS is the compiled depth of the
// convolution (0 = none); shallower ones pad their weights with zeros in front.  LAYER: layer norms; the waves' means and squared
// deviations are merged by their counts, so a row still costs one barrier per norm and no sum of squares cancels.
template <typename T, int BLOCK, int NP, int TAPS, int NB, bool LAYER>
__global__ __launch_bounds__(BLOCK) void norm_conv_kernel(const e2h_norm_conv_args a, int runs, int run) {
  constexpr int kWaves = BLOCK / 64;
  constexpr int RING = TAPS > 1 ? TAPS - 1 : 1;
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  const int W = static_cast<int>(a.width), seqlen = static_cast<int>(a.seqlen), taps = a.taps;
  const int b = blockIdx.x / runs, t_begin = (blockIdx.x % runs) * run;
  const int t_end = t_begin + run < seqlen ? t_begin + run : seqlen;
  const int pos0 = TAPS ? static_cast<int>(a.input_pos[0]) : 0;
  const int first = TAPS && a.first ? static_cast<int>(a.first[b]) : 0;
  const size_t row0 = static_cast<size_t>(b) * seqlen;
  __shared__ float part[2][kWaves][NB * (LAYER ? 2 : 1)];
  int phase = 0;

  auto wave_count = [&](int w) {  // channels of the row that wave w holds
    int n = 0;
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int left = W - (p * BLOCK + w * 64) * 4;
      n += left < 0 ? 0 : left > 256 ? 256 : left;
    }
    return static_cast<float>(n);
  };
  // z -> (z - mean) / sqrt(variance + eps) * weight + bias for NB rows
  auto layer_norm = [&](f32x4_t (&z)[NB][NP], const f32x4_t (&weight)[NP], const float *bias) {
    const float own = wave_count(threadIdx.x >> 6);
    float mean[NB], dev[NB];
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      float s = 0.f;  // pieces beyond the width are zero
#pragma unroll
      for (int p = 0; p < NP; ++p) s += z[k][p][0] + z[k][p][1] + z[k][p][2] + z[k][p][3];
      mean[k] = own > 0.f ? wave_add(s) / own : 0.f;
      float q = 0.f;
#pragma unroll
      for (int p = 0; p < NP; ++p)
        if ((p * BLOCK + static_cast<int>(threadIdx.x)) * 4 < W) {
          const f32x4_t c = z[k][p] - mean[k];
#pragma unroll
          for (int e = 0; e < 4; ++e) q = __builtin_fmaf(c[e], c[e], q);
        }
      dev[k] = wave_add(q);
    }
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
      for (int k = 0; k < NB; ++k) {
        part[phase][threadIdx.x >> 6][k] = mean[k];
        part[phase][threadIdx.x >> 6][(LAYER ? NB : 0) + k] = dev[k];
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      float m = 0.f, v = 0.f;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) m = __builtin_fmaf(wave_count(w), part[phase][w][k], m);
      m /= static_cast<float>(W);
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        const float c = part[phase][w][k] - m;
        v += __builtin_fmaf(wave_count(w) * c, c, part[phase][w][(LAYER ? NB : 0) + k]);
      }
      const float r = 1.0f / sqrtf(v / static_cast<float>(W) + a.eps);
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        const int i = (p * BLOCK + threadIdx.x) * 4;
        f32x4_t b = zero;
        if (bias && i < W) b = load4(bias + i);
        z[k][p] = (z[k][p] - m) * r * weight[p] + b;
      }
    }
    phase ^= 1;
  };

  auto block_sum = [&](float (&v)[NB]) {
#pragma unroll
    for (int k = 0; k < NB; ++k) v[k] = wave_add(v[k]);
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
      for (int k = 0; k < NB; ++k) part[phase][threadIdx.x >> 6][k] = v[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      v[k] = 0.f;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) v[k] += part[phase][w][k];
      v[k] = 1.0f / sqrtf(v[k] / static_cast<float>(W) + a.eps);
    }
    phase ^= 1;  // the next sums go to the other half, so one barrier per sum is enough
  };

  // everything that does not depend on the rows; zero weights and rows beyond the width contribute nothing
  f32x4_t wconv[TAPS > 0 ? TAPS : 1][NP], wd[NP], wn[NP], ring[RING][NP];
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int i = (p * BLOCK + threadIdx.x) * 4;
    wd[p] = wn[p] = zero;
    if (a.delta_weight && i < W) wd[p] = load4(a.delta_weight + i) + a.delta_offset;
    if (a.norm_weight && i < W) wn[p] = load4(a.norm_weight + i) + a.norm_offset;
    if (TAPS) {
#pragma unroll
      for (int j = 0; j < TAPS; ++j) {
        const int jj = j - (TAPS - taps);
        wconv[j][p] = zero;
        if (i < W && jj >= 0) wconv[j][p] = load4(a.conv + static_cast<size_t>(jj) * W + i);
      }
    }
  }

  // kept inputs of the positions before the call, for a run at its start
  auto kept = [&](int t, f32x4_t (&h)[NP]) {
    const int pos = pos0 + t;
    const bool live = pos >= first && pos >= 0 && t >= -(taps - 1);
    const float *src = a.tail_in + (static_cast<size_t>(b) * taps + (live ? static_cast<uint32_t>(pos) % static_cast<uint32_t>(taps) : 0u)) * W;
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int i = (p * BLOCK + threadIdx.x) * 4;
      h[p] = zero;
      if (live && i < W) h[p] = load4(src + i);
    }
  };

  // h (the convolution's inputs) of the tokens t .. t + NB - 1; emit: also store the updated residual rows
  auto norm_rows = [&](int t, bool emit, f32x4_t (&h)[NB][NP]) {
    f32x4_t d[NB][NP];
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      const int tc = t + k < 0 ? 0 : t + k < seqlen ? t + k : seqlen - 1;
      const size_t base = (row0 + tc) * W;
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        const int i = (p * BLOCK + threadIdx.x) * 4;
        h[k][p] = d[k][p] = zero;
        if (i < W) {
          h[k][p] = load4(a.x + base + i);
          if (a.delta) d[k][p] = load4(static_cast<const T *>(a.delta) + base + i);
        }
      }
      if (TAPS == 0 && a.terms) {
        const float *tw = a.term_weights + (row0 + tc) * a.n_terms;
        const T *term = static_cast<const T *>(a.terms) + (row0 + tc) * a.n_terms * W;
        constexpr int kAhead = 4;  // terms whose loads are in flight together
        for (int j0 = 0; j0 < static_cast<int>(a.n_terms); j0 += kAhead, term += kAhead * W) {
          Quad<T> y[kAhead][NP];
          float c[kAhead];
#pragma unroll
          for (int j = 0; j < kAhead; ++j) {
            const bool live = j0 + j < a.n_terms;
            c[j] = live ? tw[j0 + j] : 0.f;
#pragma unroll
            for (int p = 0; p < NP; ++p) {
              const int i = (p * BLOCK + threadIdx.x) * 4;
              y[j][p].raw = {};
              if (live && i < W) y[j][p] = load_quad(term + j * W + i);
            }
          }
#pragma unroll
          for (int j = 0; j < kAhead; ++j)
#pragma unroll
            for (int p = 0; p < NP; ++p) {
              const f32x4_t v = y[j][p].f32();
#pragma unroll
              for (int e = 0; e < 4; ++e) d[k][p][e] = __builtin_fmaf(c[j], v[e], d[k][p][e]);
            }
        }
      }
    }
    if (LAYER && (a.delta || a.terms)) {
      layer_norm(d, wd, a.delta_bias);
#pragma unroll
      for (int k = 0; k < NB; ++k)
#pragma unroll
        for (int p = 0; p < NP; ++p) {
          const int i = (p * BLOCK + threadIdx.x) * 4;
          if (i < W) {
            h[k][p] += d[k][p];
            if (emit && a.x_out && t + k < t_end) store4(a.x_out + (row0 + t + k) * W + i, h[k][p]);
          }
        }
    }
    if (!LAYER && (a.delta || a.terms)) {
      float ss[NB];
#pragma unroll
      for (int k = 0; k < NB; ++k) {
        ss[k] = 0.f;
#pragma unroll
        for (int p = 0; p < NP; ++p)
#pragma unroll
          for (int e = 0; e < 4; ++e) ss[k] = __builtin_fmaf(d[k][p][e], d[k][p][e], ss[k]);
      }
      block_sum(ss);
#pragma unroll
      for (int k = 0; k < NB; ++k)
#pragma unroll
        for (int p = 0; p < NP; ++p) {
          const int i = (p * BLOCK + threadIdx.x) * 4;
          h[k][p] += d[k][p] * ss[k] * wd[p];
          if (emit && a.x_out && i < W && t + k < t_end) store4(a.x_out + (row0 + t + k) * W + i, h[k][p]);
        }
    }
    if (LAYER && a.norm_weight) layer_norm(h, wn, a.norm_bias);
    if (!LAYER && a.norm_weight) {
      float ss[NB];
#pragma unroll
      for (int k = 0; k < NB; ++k) {
        ss[k] = 0.f;
#pragma unroll
        for (int p = 0; p < NP; ++p)
#pragma unroll
          for (int e = 0; e < 4; ++e) ss[k] = __builtin_fmaf(h[k][p][e], h[k][p][e], ss[k]);
      }
      block_sum(ss);
#pragma unroll
      for (int k = 0; k < NB; ++k)
#pragma unroll
        for (int p = 0; p < NP; ++p) h[k][p] = h[k][p] * ss[k] * wn[p];
    }
    if (TAPS) {
#pragma unroll
      for (int k = 0; k < NB; ++k)
        if (pos0 + t + k < first) {  // padding: the convolution must not see it
#pragma unroll
          for (int p = 0; p < NP; ++p) h[k][p] = zero;
        }
    }
  };
  auto push = [&](const f32x4_t (&h)[NP]) {
#pragma unroll
    for (int p = 0; p < NP; ++p) {
#pragma unroll
      for (int j = 0; j + 1 < RING; ++j) ring[j][p] = ring[j + 1][p];
      ring[RING - 1][p] = h[p];
    }
  };

  if (TAPS > 1) {
    if (t_begin == 0) {
#pragma unroll
      for (int j = 0; j < RING; ++j) kept(j - RING, ring[j]);
    } else {
#pragma unroll
      for (int s = -((RING + NB - 1) / NB * NB); s < 0; s += NB) {
        f32x4_t h[NB][NP];
        norm_rows(t_begin + s, false, h);
#pragma unroll
        for (int k = 0; k < NB; ++k) {
          if (t_begin + s + k < 0) kept(t_begin + s + k, h[k]);
          push(h[k]);
        }
      }
    }
  }
  for (int t = t_begin; t < t_end; t += NB) {
    f32x4_t h[NB][NP];
    norm_rows(t, true, h);
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      if (t + k < t_end) {
        const size_t base = (row0 + t + k) * W;
#pragma unroll
        for (int p = 0; p < NP; ++p) {
          const int i = (p * BLOCK + threadIdx.x) * 4;
          f32x4_t y = h[k][p];
          if (TAPS) {
            f32x4_t c = y * wconv[TAPS > 0 ? TAPS - 1 : 0][p];
            if (TAPS > 1) {
#pragma unroll
              for (int j = 0; j < RING; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) c[e] = __builtin_fmaf(ring[j][p][e], wconv[j][p][e], c[e]);
            }
            y += c;
          }
          if (a.out && i < W) store4(static_cast<T *>(a.out) + base + i, y);
        }
        if (TAPS > 1) push(h[k]);
      }
    }
  }
  if (TAPS > 1 && t_end == seqlen) {  // the last inputs of the call, oldest first in the ring registers; one token replaces one slot
#pragma unroll
    for (int j = 0; j < RING; ++j) {
      const int pos = pos0 + seqlen - RING + j;
      if (j >= RING - (seqlen == 1 ? 1 : taps - 1) && pos >= 0 && taps > 1) {
        float *dst = a.tail_out + (static_cast<size_t>(b) * taps + static_cast<uint32_t>(pos) % static_cast<uint32_t>(taps)) * W;
#pragma unroll
        for (int p = 0; p < NP; ++p) {
          const int i = (p * BLOCK + threadIdx.x) * 4;
          if (i < W) store4(dst + i, ring[j][p]);
        }
      }
    }
  }
}

template <typename T, int BLOCK, int NP, int TAPS, bool LAYER>
void launch_norm_conv_rows(const e2h_norm_conv_args &a, int runs, int run, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(a.batch * runs)), block(BLOCK);
  constexpr int NB = NP > 1 || TAPS > 4 ? 1 : TAPS || LAYER ? 2 : 4;  // rows that fit the registers
  if (run == 1) hipLaunchKernelGGL((norm_conv_kernel<T, BLOCK, NP, TAPS, 1, LAYER>), grid, block, 0, s, a, runs, run);
  else hipLaunchKernelGGL((norm_conv_kernel<T, BLOCK, NP, TAPS, NB, LAYER>), grid, block, 0, s, a, runs, run);
}

template <typename T, int BLOCK, int NP>
void launch_norm_conv_taps(const e2h_norm_conv_args &a, int runs, int run, hipStream_t s) {
  if constexpr (BLOCK != 1024 || NP != 1) {  // (that geometry is for convolutions only)
    if (a.norm_kind == E2H_SEQ_LAYER_NORM) return launch_norm_conv_rows<T, BLOCK, NP, 0, true>(a, runs, run, s);
    if (!a.conv) return launch_norm_conv_rows<T, BLOCK, NP, 0, false>(a, runs, run, s);
  }
  if (a.taps <= 4) launch_norm_conv_rows<T, BLOCK, NP, 4, false>(a, runs, run, s);
  else launch_norm_conv_rows<T, BLOCK, NP, 8, false>(a, runs, run, s);
}

template <typename T>
void launch_norm_conv(const e2h_norm_conv_args &a, int runs, int run, hipStream_t s) {
  if (a.width <= 1024) launch_norm_conv_taps<T, 256, 1>(a, runs, run, s);
  else if (a.width <= 2048) launch_norm_conv_taps<T, 512, 1>(a, runs, run, s);
  else if (a.width <= 4096 && a.conv) launch_norm_conv_taps<T, 1024, 1>(a, runs, run, s);
  else if (a.width <= 4096) launch_norm_conv_taps<T, 512, 2>(a, runs, run, s);
  else if (a.width <= 8192) launch_norm_conv_taps<T, 512, 4>(a, runs, run, s);
  else launch_norm_conv_taps<T, 1024, 4>(a, runs, run, s);
}

// ---- elementwise -----------------------------------------------------------------------------------------------------
enum { kSquareRelu = 0, kSoftcap = 1 };

template <int OP>
__device__ __forceinline__ float elementwise_op(float v, float cap) {
  if (OP == kSquareRelu) {
    const float r = fmaxf(v, 0.f);
    return r * r;
  }
  return cap * tanhf(v / cap);
}

template <typename T, int OP>
__global__ __launch_bounds__(256) void elementwise_kernel(const T *x, T *y, int64_t n, float cap) {
  const int64_t i = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * 4;
  if (i + 4 <= n) {
    f32x4_t v = load4(x + i);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = elementwise_op<OP>(v[e], cap);
    store4(y + i, v);
  } else {
    for (int64_t j = i; j < n; ++j) y[j] = from_f32<T>(elementwise_op<OP>(to_f32(x[j]), cap));
  }
}

template <int OP>
int launch_elementwise(int dtype, const void *x, void *y, int64_t n, float cap, void *stream) {
  if (!x || !y) return E2H_ERR_NULL_POINTER;
  const int64_t blocks = (n + 1023) / 1024;
  if (n < 1 || blocks > INT32_MAX || (dtype != E2H_SEQ_BF16 && dtype != E2H_SEQ_F32)) return E2H_ERR_BAD_SHAPE;
  if (!aligned16(x) || !aligned16(y)) return E2H_ERR_MISALIGNED;
  const dim3 grid(static_cast<unsigned>(blocks)), block(256);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == E2H_SEQ_BF16)
    hipLaunchKernelGGL((elementwise_kernel<bf16_t, OP>), grid, block, 0, s, static_cast<const bf16_t *>(x), static_cast<bf16_t *>(y), n, cap);
  else
    hipLaunchKernelGGL((elementwise_kernel<float, OP>), grid, block, 0, s, static_cast<const float *>(x), static_cast<float *>(y), n, cap);
  return launch_status();
}

template <typename T>
__global__ __launch_bounds__(256) void gelu_gate_rows_kernel(const T *__restrict__ gate, const T *__restrict__ table, const int64_t *__restrict__ tokens,
                                                             T *__restrict__ y, int64_t n, int dim, int64_t ld, int64_t column, int64_t table_rows) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= n) return;
  const int64_t r = i / dim, c = i % dim;
  const int64_t tok = tokens[r];
  const float z = to_f32(gate[i]);
  const float e = tok >= 0 && tok < table_rows ? to_f32(table[tok * ld + column + c]) : 0.f;
  const float g = 0.5f * z * (1.0f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
  y[i] = from_f32<T>(g * e);
}

}  // namespace
}  // namespace e2h

using namespace e2h;

extern "C" int e2h_seq_abi_version(void) { return E2H_SEQ_ABI_VERSION; }

extern "C" int e2h_seq_set_option(const char *name, int value) {
  if (!name) return E2H_ERR_NULL_POINTER;
  SeqOptions &o = seq_options();
  if (!strcmp(name, "recurrence_form")) {
    if (value < 0 || value > 2) return E2H_ERR_BAD_OPTION;
    o.recurrence_form = value;
  } else if (!strcmp(name, "recurrence_chunk")) {
    if (value < 0 || value % 64 != 0) return E2H_ERR_BAD_OPTION;
    o.recurrence_chunk = value;
  } else if (!strcmp(name, "norm_run")) {
    if (value < 0 || value > 256) return E2H_ERR_BAD_OPTION;
    o.norm_run = value;
  } else if (!strcmp(name, "attention_decode_waves")) {
    if (value != 0 && value != 4 && value != 8) return E2H_ERR_BAD_OPTION;
    o.attention_decode_waves = value;
  } else if (!strcmp(name, "attention_prompt_queries")) {
    if (value != 0 && value != 64 && value != 128) return E2H_ERR_BAD_OPTION;
    o.attention_prompt_queries = value;
  } else if (!strcmp(name, "expert_form")) {
    if (value < 0 || value > 3) return E2H_ERR_BAD_OPTION;
    o.expert_form = value;
  } else {
    return E2H_ERR_BAD_OPTION;
  }
  return E2H_OK;
}

extern "C" int e2h_seq_norm_conv(const e2h_norm_conv_args *a, void *stream) {
  if (!a || !a->x || ((a->delta || a->terms) && !a->delta_weight) || (a->terms && !a->term_weights)) return E2H_ERR_NULL_POINTER;
  if (!a->out && !a->x_out) return E2H_ERR_NULL_POINTER;
  if (a->conv && (!a->input_pos || (a->taps > 1 && (!a->tail_in || !a->tail_out)))) return E2H_ERR_NULL_POINTER;
  if (a->batch < 1 || a->seqlen < 1 || a->width < 4 || a->width % 4 != 0 || a->width > 16384 || a->seqlen > INT32_MAX / 4)
    return E2H_ERR_BAD_SHAPE;
  if (a->dtype != E2H_SEQ_BF16 && a->dtype != E2H_SEQ_F32) return E2H_ERR_BAD_SHAPE;
  if (a->conv && (a->taps < 1 || a->taps > 8)) return E2H_ERR_BAD_SHAPE;
  if (a->norm_kind != E2H_SEQ_RMS_NORM && a->norm_kind != E2H_SEQ_LAYER_NORM) return E2H_ERR_BAD_SHAPE;
  if (a->conv && (a->norm_kind == E2H_SEQ_LAYER_NORM || a->terms)) return E2H_ERR_BAD_SHAPE;
  if (a->terms && a->n_terms < 1) return E2H_ERR_BAD_SHAPE;
  if (a->seqlen > 1 && a->conv && ((a->taps > 1 && a->tail_in == a->tail_out) || (a->delta && a->x == a->x_out && a->taps > 1))) return E2H_ERR_BAD_SHAPE;
  if (!aligned16(a->x) || !aligned16(a->delta) || !aligned16(a->delta_weight) || !aligned16(a->x_out) || !aligned16(a->norm_weight) ||
      !aligned16(a->conv) || !aligned16(a->tail_in) || !aligned16(a->tail_out) || !aligned16(a->out) ||
      !aligned16(a->delta_bias) || !aligned16(a->norm_bias) || !aligned16(a->terms))
    return E2H_ERR_MISALIGNED;
  // enough workgroups to fill the chip first, then longer runs so that fewer tokens are normalised twice
  int run = seq_options().norm_run;
  if (!run) {
    run = static_cast<int>(a->batch * a->seqlen / (a->conv ? 256 : 1024));
    run = run < 1 ? 1 : run > 32 ? 32 : run;
  }
  const int64_t runs = (a->seqlen + run - 1) / run;
  if (a->batch * runs > INT32_MAX) return E2H_ERR_BAD_SHAPE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (a->dtype == E2H_SEQ_BF16) launch_norm_conv<bf16_t>(*a, static_cast<int>(runs), run, s);
  else launch_norm_conv<float>(*a, static_cast<int>(runs), run, s);
  return launch_status();
}

extern "C" int e2h_seq_square_relu(int dtype, const void *x, void *y, int64_t n, void *stream) {
  return launch_elementwise<kSquareRelu>(dtype, x, y, n, 0.f, stream);
}

extern "C" int e2h_seq_softcap(int dtype, const void *x, void *y, int64_t n, float cap, void *stream) {
  if (!(cap > 0.f)) return E2H_ERR_BAD_SHAPE;
  return launch_elementwise<kSoftcap>(dtype, x, y, n, cap, stream);
}

extern "C" int e2h_seq_gelu_gate_rows(int dtype, const void *gate, const void *table, const int64_t *tokens, void *y, int64_t rows, int64_t dim,
                                      int64_t ld, int64_t column, int64_t table_rows, void *stream) {
  if (!gate || !table || !tokens || !y) return E2H_ERR_NULL_POINTER;
  if (rows < 1 || dim < 1 || dim > INT32_MAX || column < 0 || column + dim > ld || table_rows < 1) return E2H_ERR_BAD_SHAPE;
  if (dtype != E2H_SEQ_BF16 && dtype != E2H_SEQ_F32) return E2H_ERR_BAD_SHAPE;
  const int64_t n = rows * dim, blocks = (n + 255) / 256;
  if (blocks > INT32_MAX) return E2H_ERR_BAD_SHAPE;
  const dim3 grid(static_cast<unsigned>(blocks)), block(256);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == E2H_SEQ_BF16)
    hipLaunchKernelGGL(gelu_gate_rows_kernel<bf16_t>, grid, block, 0, s, static_cast<const bf16_t *>(gate), static_cast<const bf16_t *>(table), tokens,
                       static_cast<bf16_t *>(y), n, static_cast<int>(dim), ld, column, table_rows);
  else
    hipLaunchKernelGGL(gelu_gate_rows_kernel<float>, grid, block, 0, s, static_cast<const float *>(gate), static_cast<const float *>(table), tokens,
                       static_cast<float *>(y), n, static_cast<int>(dim), ld, column, table_rows);
  return launch_status();
}
