// Row kernels of the stateful decoder layers: residual add of a normalised sublayer output, the next sublayer's norm and
// its input convolution over time in one pass over the float32 residual stream, and the elementwise steps.
#include <string.h>

#include <algorithm>

#include "e2h_seq_common.h"

namespace e2h {

SeqOptions &seq_options() {
  static SeqOptions o = {};
  return o;
}

namespace {

#if defined(__HIP_DEVICE_COMPILE__)
constexpr int kStreamed = 2;  // cache policy of a buffer store whose line nobody reads soon

// four values of a row from piece `at` (four channels each) on
template <typename T>
__device__ __forceinline__ Quad<T> buffer_quad(__amdgpu_buffer_rsrc_t row, int at) {
  Quad<T> q;
  if constexpr (sizeof(T) == 4) q.raw = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(row, at * 16, 0, 0));
  else q.raw = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_raw_buffer_load_b64(row, at * 8, 0, 0));
  return q;
}
template <int POLICY>
__device__ __forceinline__ void buffer_store(__amdgpu_buffer_rsrc_t row, int at, f32x4_t v, float) {
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, v), row, at * 16, 0, POLICY);
}
template <int POLICY>
__device__ __forceinline__ void buffer_store(__amdgpu_buffer_rsrc_t row, int at, f32x4_t v, bf16_t) {
  __builtin_amdgcn_raw_buffer_store_b64(u32x2_t{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])}, row, at * 8, 0, POLICY);
}
#endif

// delta as the float32 sums of K slices [slices][rows][width] that its linear left (e2h_seq_linear_sums): rounded as the linear's own output.  The launch that adds them costs a step of 32
// rows more than the norm, which waits for its row anyway, takes longer for reading four times as much.  Not with runs, whose rows are asked for ahead.
struct DeltaSums {
  const float *from;
  int slices;
};

// One row per workgroup, or with a convolution (which needs its previous inputs) a run of `run` consecutive tokens of one sequence.  A thread owns NP pieces of four channels, so the
// convolution's previous inputs stay in its registers from token to token; the taps - 1 tokens ahead of the run are normalised again by the
// workgroup (inside the call) or come from the ring of kept inputs (before the call).  TAPS is the compiled depth of the
// convolution (0 = none); shallower ones pad their weights with zeros in front.  LAYER: layer norms; the waves' means and squared
// deviations are merged by their counts, so a row still costs one barrier per norm and no sum of squares cancels.
//
// What bounds it: memory, once enough rows are on their way.  A run's workgroup asks for its next row before it waits for anything of this one (AHEAD): loads and stores have no branch
// between them, or a wait for one row's loads would be one for all.  Without a convolution rows next to each other are at work at the same time, which beats runs with the next row on its
// way (8192 x 4096, sum and norm 72 us, 80 in runs of 8), and large residual rows, which are not read again soon, are stored past the caches (58).
// us at 4096 channels, in brackets runs of 8 (convolution: 1024 threads, two rows together) that waited for every row: 8192 rows with residual 60 (97), layer norm 66 (92), eight experts'
// terms 166 (187), convolution 85 (112); 8000 rows 58 (86), 62 (106), 160 (214), 80 (167: one workgroup too many for a round); 2048 rows 18 (18), 21 (21), 40 (38), 28 (32).
template <typename T, int BLOCK, int NP, int TAPS, bool LAYER, bool TERMS, bool AHEAD, int SPLIT>
__global__ __launch_bounds__(BLOCK) void norm_conv_kernel(const e2h_norm_conv_args a, const DeltaSums sums, int runs, int run, int streamed) {
#if defined(__HIP_DEVICE_COMPILE__)
  static_assert(SPLIT == 1 || SPLIT == NP, "a thread's pieces are summed together or each for itself");
  constexpr int kWaves = BLOCK / 64, kSums = SPLIT * kWaves, kEach = NP / SPLIT;  // a row's partial sums, and the pieces that a thread adds to each
  constexpr int RING = TAPS > 1 ? TAPS - 1 : 1;
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  const int W = static_cast<int>(a.width), seqlen = static_cast<int>(a.seqlen), taps = a.taps;
  // without a convolution rows know nothing of their sequence
  const int b = TAPS ? blockIdx.x / runs : 0, t_begin = TAPS ? (blockIdx.x % runs) * run : blockIdx.x;
  const int64_t t_end = TAPS ? t_begin + run < seqlen ? t_begin + run : seqlen : a.batch * a.seqlen;
  const int step = TAPS ? 1 : static_cast<int>(gridDim.x);
  const int pos0 = TAPS ? static_cast<int>(a.input_pos[0]) : 0;
  const int first = TAPS && a.first ? static_cast<int>(a.first[b]) : 0;
  const size_t row0 = static_cast<size_t>(b) * seqlen;
  const uint32_t row_f32 = static_cast<uint32_t>(W) * 4, row_t = static_cast<uint32_t>(W) * sizeof(T);
  __shared__ __attribute__((aligned(16))) float part[2][kSums][LAYER ? 2 : 1];
  int phase = 0;

  auto sum_count = [&](int u) {  // channels of the row in partial sum u, of wave u % kWaves
    int n = 0;
#pragma unroll
    for (int p = 0; p < kEach; ++p) {
      const int left = W - ((u / kWaves * kEach + p) * BLOCK + u % kWaves * 64) * 4;
      n += left < 0 ? 0 : left > 256 ? 256 : left;
    }
    return static_cast<float>(n);
  };
  const int wave = threadIdx.x >> 6;
  auto piece = [&](int p) { return p * BLOCK + static_cast<int>(threadIdx.x); };
  // Rows beyond 8192 leave no registers for weights and biases in front of the row (kLate): read where they are used.  (2048 x 12288, two layer norms: 169 us, 1590 with 655 values of every thread spilled.)
  constexpr bool kLate = TAPS == 0 && BLOCK * NP > 2048;
  auto channel = [&](const float *from, int p, float offset) {
    f32x4_t v = zero;
    if (from && piece(p) * 4 < W) v = load4(from + piece(p) * 4) + offset;
    return v;
  };
  // z -> (z - mean) / sqrt(variance + eps) * weight + bias
  auto layer_norm = [&](f32x4_t (&z)[NP], f32x4_t (&weight)[NP], f32x4_t (&bias)[NP], const float *late_weight, float offset, const float *late_bias) {
#pragma unroll
    for (int u = 0; u < SPLIT; ++u) {
      const float own = sum_count(u * kWaves + wave);
      float s = 0.f;  // pieces beyond the width are zero
#pragma unroll
      for (int p = u * kEach; p < (u + 1) * kEach; ++p) s += z[p][0] + z[p][1] + z[p][2] + z[p][3];
      const float mean = own > 0.f ? wave_add(s) / own : 0.f;
      float q = 0.f;
#pragma unroll
      for (int p = u * kEach; p < (u + 1) * kEach; ++p)
        if (piece(p) * 4 < W) {
          const f32x4_t c = z[p] - mean;
#pragma unroll
          for (int e = 0; e < 4; ++e) q = __builtin_fmaf(c[e], c[e], q);
        }
      q = wave_add(q);
      if ((threadIdx.x & 63) == 0) {
        part[phase][u * kWaves + wave][0] = mean;
        part[phase][u * kWaves + wave][LAYER ? 1 : 0] = q;
      }
    }
    __syncthreads();
    float m = 0.f, v = 0.f;
#pragma unroll
    for (int w = 0; w < kSums; ++w) m = __builtin_fmaf(sum_count(w), part[phase][w][0], m);
    m /= static_cast<float>(W);
#pragma unroll
    for (int w = 0; w < kSums; ++w) {
      const float c = part[phase][w][0] - m;
      v += __builtin_fmaf(sum_count(w) * c, c, part[phase][w][LAYER ? 1 : 0]);
    }
    const float r = 1.0f / sqrtf(v / static_cast<float>(W) + a.eps);
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      if (kLate) weight[p] = channel(late_weight, p, offset), bias[p] = channel(late_bias, p, 0.f);
      z[p] = (z[p] - m) * r * weight[p] + bias[p];
    }
    phase ^= 1;
  };

  auto inverse_rms = [&](const f32x4_t (&z)[NP]) {
    float v[SPLIT];
#pragma unroll
    for (int u = 0; u < SPLIT; ++u) {
      v[u] = 0.f;
#pragma unroll
      for (int p = u * kEach; p < (u + 1) * kEach; ++p)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[u] = __builtin_fmaf(z[p][e], z[p][e], v[u]);
    }
#pragma unroll
    for (int u = 0; u < SPLIT; ++u) {
      v[u] = wave_add(v[u]);
      if ((threadIdx.x & 63) == 0) part[phase][u * kWaves + wave][0] = v[u];
    }
    __syncthreads();
    float sum = 0.f;
#pragma unroll
    for (int w = 0; w < kSums; ++w) sum += part[phase][w][0];
    phase ^= 1;  // the next sums go to the other half, so one barrier per sum is enough
    return 1.0f / sqrtf(sum / static_cast<float>(W) + a.eps);
  };

  // everything that does not depend on the rows; zero weights and rows beyond the width contribute nothing
  f32x4_t wconv[TAPS > 0 ? TAPS : 1][NP], wd[NP], wn[NP], bd[NP], bn[NP], ring[RING][NP];
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int i = piece(p) * 4;
    wd[p] = wn[p] = bd[p] = bn[p] = zero;
    if (!kLate && a.delta_weight && i < W) wd[p] = load4(a.delta_weight + i) + a.delta_offset;
    if (!kLate && a.norm_weight && i < W) wn[p] = load4(a.norm_weight + i) + a.norm_offset;
    if (!kLate && LAYER && a.delta_bias && i < W) bd[p] = load4(a.delta_bias + i);
    if (!kLate && LAYER && a.norm_bias && i < W) bn[p] = load4(a.norm_bias + i);
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
      const int i = piece(p) * 4;
      h[p] = zero;
      if (live && i < W) h[p] = load4(src + i);
    }
  };

  // What row t needs from memory, by loads that return zero past the width and for what the call does not have: no branch stands
  // between them, so what waits for one knows how many were asked for behind it.
  struct Raw {
    f32x4_t h[NP];
    Quad<T> d[NP];
  };
  auto request = [&](int64_t t, Raw &raw) {
    const size_t base = (row0 + (t < 0 ? 0 : t < t_end ? t : t_end - 1)) * W;
    const __amdgpu_buffer_rsrc_t x = make_rsrc(a.x + base, row_f32), d = make_rsrc(static_cast<const T *>(a.delta) + (a.delta ? base : 0), a.delta ? row_t : 0);
#pragma unroll
    for (int p = 0; p < NP; ++p) raw.h[p] = buffer_quad<float>(x, piece(p)).raw;
#pragma unroll
    for (int p = 0; p < NP; ++p) raw.d[p] = buffer_quad<T>(d, piece(p));
  };

  // h (the convolution's input) of row t; emit: also store the updated residual row.  ahead: asked for in front of everything that waits
  auto norm_row = [&](int64_t t, bool emit, const Raw &raw, auto ahead, f32x4_t (&h)[NP]) {
    f32x4_t d[NP];
    ahead();
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      h[p] = raw.h[p];
      d[p] = raw.d[p].f32();
    }
    const bool summed = !AHEAD && !TERMS && !LAYER && sums.from;
    if (summed) {
      constexpr int kMost = 4;
      f32x4_t part[kMost][NP];
      const size_t slice = static_cast<size_t>(a.batch) * seqlen * W;
#pragma unroll
      for (int k = 0; k < kMost; ++k) {
        const __amdgpu_buffer_rsrc_t r = make_rsrc(sums.from + (k < sums.slices ? k : 0) * slice + (row0 + t) * W, k < sums.slices ? row_f32 : 0);
#pragma unroll
        for (int p = 0; p < NP; ++p) part[k][p] = buffer_quad<float>(r, piece(p)).raw;
      }
#pragma unroll
      for (int p = 0; p < NP; ++p) {
#pragma unroll
        for (int k = 1; k < kMost; ++k) part[0][p] += part[k][p];
#pragma unroll
        for (int e = 0; e < 4; ++e) d[p][e] = to_f32(from_f32<T>(part[0][p][e]));
      }
    }
    if constexpr (TERMS) {
      const int n = static_cast<int>(a.n_terms);
      const float *tw = a.term_weights + (row0 + t) * n;
      const T *term = static_cast<const T *>(a.terms) + (row0 + t) * n * W;
      constexpr int kAhead = 4;  // terms whose loads are in flight together
      for (int j0 = 0; j0 < n; j0 += kAhead) {
        Quad<T> y[kAhead][NP];
#pragma unroll
        for (int j = 0; j < kAhead; ++j) {
          const bool live = j0 + j < n;
          const __amdgpu_buffer_rsrc_t r = make_rsrc(term + static_cast<size_t>(live ? j0 + j : 0) * W, live ? row_t : 0);
#pragma unroll
          for (int p = 0; p < NP; ++p) y[j][p] = buffer_quad<T>(r, piece(p));
        }
#pragma unroll
        for (int j = 0; j < kAhead; ++j) {
          const float c = j0 + j < n ? tw[j0 + j] : 0.f;
#pragma unroll
          for (int p = 0; p < NP; ++p) {
            const f32x4_t v = y[j][p].f32();
#pragma unroll
            for (int e = 0; e < 4; ++e) d[p][e] = __builtin_fmaf(c, v[e], d[p][e]);
          }
        }
      }
    }
    if (a.delta || TERMS || summed) {
      if constexpr (LAYER) {
        layer_norm(d, wd, bd, a.delta_weight, a.delta_offset, a.delta_bias);
#pragma unroll
        for (int p = 0; p < NP; ++p)
          if (piece(p) * 4 < W) h[p] += d[p];
      } else {
        const float r = inverse_rms(d);
#pragma unroll
        for (int p = 0; p < NP; ++p) {
          if (kLate) wd[p] = channel(a.delta_weight, p, a.delta_offset);
          h[p] += d[p] * r * wd[p];
        }
      }
      const bool there = emit && a.x_out;
      const __amdgpu_buffer_rsrc_t to = make_rsrc(a.x_out + (there ? (row0 + t) * W : 0), there ? row_f32 : 0);
      if (streamed) {
#pragma unroll
        for (int p = 0; p < NP; ++p) buffer_store<kStreamed>(to, piece(p), h[p], float{});
      } else {
#pragma unroll
        for (int p = 0; p < NP; ++p) buffer_store<0>(to, piece(p), h[p], float{});
      }
    }
    if (a.norm_weight) {
      if constexpr (LAYER) {
        layer_norm(h, wn, bn, a.norm_weight, a.norm_offset, a.norm_bias);
      } else {
        const float r = inverse_rms(h);
#pragma unroll
        for (int p = 0; p < NP; ++p) {
          if (kLate) wn[p] = channel(a.norm_weight, p, a.norm_offset);
          h[p] = h[p] * r * wn[p];
        }
      }
    }
    if (TAPS && pos0 + t < first) {  // padding: the convolution must not see it
#pragma unroll
      for (int p = 0; p < NP; ++p) h[p] = zero;
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

  Raw cur, next;
  if (AHEAD) request(TAPS > 1 && t_begin > 0 ? t_begin - RING : t_begin, cur);
  // the row that is asked for in front of row t's work is the one behind it (behind the last one that again, for nothing)
  auto take = [&](int64_t t, bool emit, f32x4_t (&h)[NP]) {
    if (!AHEAD) request(t, cur);
    norm_row(t, emit, cur, [&] { if (AHEAD) request(t + 1, next); }, h);
    if (AHEAD) cur = next;
  };
  if (TAPS > 1) {
    if (t_begin == 0) {
#pragma unroll
      for (int j = 0; j < RING; ++j) kept(j - RING, ring[j]);
    } else {
#pragma unroll
      for (int s = -RING; s < 0; ++s) {
        f32x4_t h[NP];
        take(t_begin + s, false, h);
        if (t_begin + s < 0) kept(t_begin + s, h);
        push(h);
      }
    }
  }
  for (int64_t t = t_begin; t < t_end; t += step) {
    f32x4_t h[NP];
    take(t, true, h);
    const __amdgpu_buffer_rsrc_t out = make_rsrc(static_cast<const T *>(a.out) + (a.out ? (row0 + t) * W : 0), a.out ? row_t : 0);
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      f32x4_t y = h[p];
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
      buffer_store<0>(out, piece(p), y, T{});
    }
    if (TAPS > 1) push(h);
  }
  if (TAPS > 1 && t_end == seqlen) {  // the last inputs of the call, oldest first in the ring registers; one token replaces one slot
#pragma unroll
    for (int j = 0; j < RING; ++j) {
      const int pos = pos0 + seqlen - RING + j;
      if (j >= RING - (seqlen == 1 ? 1 : taps - 1) && pos >= 0 && taps > 1) {
        float *dst = a.tail_out + (static_cast<size_t>(b) * taps + static_cast<uint32_t>(pos) % static_cast<uint32_t>(taps)) * W;
#pragma unroll
        for (int p = 0; p < NP; ++p) {
          const int i = piece(p) * 4;
          if (i < W) store4(dst + i, ring[j][p]);
        }
      }
    }
  }
#endif
}

template <typename T, int BLOCK, int NP, int TAPS, bool LAYER, bool TERMS, int SPLIT>
void launch_norm_conv_rows(const e2h_norm_conv_args &a, const DeltaSums &sums, int runs, int run, hipStream_t s) {
  const int64_t workgroups = TAPS ? a.batch * runs : a.batch * a.seqlen < (1 << 20) ? a.batch * a.seqlen : 1 << 20;
  const dim3 grid(static_cast<unsigned>(workgroups)), block(BLOCK);
  // from 22.4 million values on (x, the new x and two 16-bit operands are 12 bytes each) they do not stay in 256 MB of cache anyway; 4096 x 4096 takes as long with either store
  const int streamed = a.batch * a.seqlen * a.width >= (int64_t{1} << 28) / 12;
  if constexpr (TAPS > 0) {
    if (run > 1) {
      hipLaunchKernelGGL((norm_conv_kernel<T, BLOCK, NP, TAPS, LAYER, TERMS, true, SPLIT>), grid, block, 0, s, a, sums, runs, run, streamed);
      return;
    }
  }
  hipLaunchKernelGGL((norm_conv_kernel<T, BLOCK, NP, TAPS, LAYER, TERMS, false, SPLIT>), grid, block, 0, s, a, sums, runs, run, streamed);
}

// CONV: with a convolution or not
template <typename T, int BLOCK, int NP, bool CONV, int SPLIT = 1>
void launch_norm_conv_taps(const e2h_norm_conv_args &a, const DeltaSums &sums, int runs, int run, hipStream_t s) {
  if constexpr (CONV) {
    if (a.taps <= 4) launch_norm_conv_rows<T, BLOCK, NP, 4, false, false, SPLIT>(a, sums, runs, run, s);
    else launch_norm_conv_rows<T, BLOCK, NP, 8, false, false, SPLIT>(a, sums, runs, run, s);
  } else if (a.norm_kind == E2H_SEQ_LAYER_NORM) {
    if (a.terms) launch_norm_conv_rows<T, BLOCK, NP, 0, true, true, SPLIT>(a, sums, runs, run, s);
    else launch_norm_conv_rows<T, BLOCK, NP, 0, true, false, SPLIT>(a, sums, runs, run, s);
  } else {
    if (a.terms) launch_norm_conv_rows<T, BLOCK, NP, 0, false, true, SPLIT>(a, sums, runs, run, s);
    else launch_norm_conv_rows<T, BLOCK, NP, 0, false, false, SPLIT>(a, sums, runs, run, s);
  }
}

// A row's sums have one order (one with a convolution, one without) whatever the number of rows beside it and the length of runs: forms of half the threads keep a thread's two pieces apart
// (SPLIT), as two threads of the other form have them.  8192 x 4096 with convolution 84 us, 78 with them added first; 8192 x 2048 31.7, 31.1, layer norm 34.6, 32.9.
template <typename T>
void launch_norm_conv(const e2h_norm_conv_args &a, const DeltaSums &sums, int runs, int run, hipStream_t s) {
  if (a.conv) {
    if (a.width <= 1024) launch_norm_conv_taps<T, 256, 1, true>(a, sums, runs, run, s);
    else if (a.width <= 2048) launch_norm_conv_taps<T, 512, 1, true>(a, sums, runs, run, s);
    else if (a.width <= 4096 && run == 1) launch_norm_conv_taps<T, 1024, 1, true>(a, sums, runs, run, s);
    else if (a.width <= 4096) launch_norm_conv_taps<T, 512, 2, true, 2>(a, sums, runs, run, s);
    else if (a.width <= 8192) launch_norm_conv_taps<T, 512, 4, true>(a, sums, runs, run, s);
    else launch_norm_conv_taps<T, 1024, 4, true>(a, sums, runs, run, s);
    return;
  }
  if (a.width <= 1024) launch_norm_conv_taps<T, 256, 1, false>(a, sums, runs, run, s);
  // eight values per thread where many rows are waiting: half the waves, which repeat a row's sums each (8192 x 2048, layer norm 35 us, 38 with four values; final norm 30, 31)
  else if (a.width <= 2048 && a.batch * a.seqlen > 256) launch_norm_conv_taps<T, 256, 2, false, 2>(a, sums, runs, run, s);
  else if (a.width <= 2048) launch_norm_conv_taps<T, 512, 1, false>(a, sums, runs, run, s);
  else if (a.width <= 4096) launch_norm_conv_taps<T, 512, 2, false>(a, sums, runs, run, s);
  else if (a.width <= 8192) launch_norm_conv_taps<T, 512, 4, false>(a, sums, runs, run, s);
  else launch_norm_conv_taps<T, 1024, 4, false>(a, sums, runs, run, s);
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
  y[i] = from_f32<T>(gelu_tanh_f32(z) * e);
}

// Rows of a 16-bit embedding as float32 values, where the residual stream starts, and (h not null) as they are; eight values per thread.  Bound by memory: 8192 x 4096 (201 MB, 268 with
// h), or in a decode step by the launch, one where a gather and a conversion were two.  A token that the table does not have becomes a row that is no number.
__global__ __launch_bounds__(256) void embed_rows_kernel(const bf16_t *__restrict__ table, const int64_t *__restrict__ tokens, float *__restrict__ x, bf16_t *__restrict__ h, int64_t pieces,
                                                         int per_row, int64_t vocab) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= pieces) return;
  const int64_t row = i / per_row, token = tokens[row];
  u32x4_t v = {0x7FC07FC0u, 0x7FC07FC0u, 0x7FC07FC0u, 0x7FC07FC0u};
  if (token >= 0 && token < vocab) v = reinterpret_cast<const u32x4_t *>(table)[token * per_row + (i - row * per_row)];
  f32x4_t lo, hi;
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    lo[2 * e] = __builtin_bit_cast(float, v[e] << 16);
    lo[2 * e + 1] = __builtin_bit_cast(float, v[e] & 0xFFFF0000u);
    hi[2 * e] = __builtin_bit_cast(float, v[2 + e] << 16);
    hi[2 * e + 1] = __builtin_bit_cast(float, v[2 + e] & 0xFFFF0000u);
  }
  store4(x + 8 * i, lo);
  store4(x + 8 * i + 4, hi);
  if (h) reinterpret_cast<u32x4_t *>(h)[i] = v;
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

namespace {
int norm_conv(const e2h_norm_conv_args *a, const DeltaSums &sums, void *stream) {
  if (!a || !a->x || ((a->delta || a->terms || sums.from) && !a->delta_weight) || (a->terms && !a->term_weights)) return E2H_ERR_NULL_POINTER;
  if (!a->out && !a->x_out) return E2H_ERR_NULL_POINTER;
  if (a->conv && (!a->input_pos || (a->taps > 1 && (!a->tail_in || !a->tail_out)))) return E2H_ERR_NULL_POINTER;
  if (a->batch < 1 || a->batch > INT32_MAX || a->seqlen < 1 || a->width < 4 || a->width % 4 != 0 || a->width > 16384 || a->seqlen > INT32_MAX / 4)
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
  // The fewest tokens per workgroup with which the convolution's workgroups are a whole number of rounds, up to 32: longer runs normalise fewer tokens twice, and one workgroup beyond a round
  // costs a round.  A round is a workgroup per CU, of narrower rows two or four (8192 x 2048: 512 workgroups 42 us, 256 54; 8192 x 1024: 1024 24, 256 49).
  int run = a->conv ? std::min<int64_t>(seq_options().norm_run, a->seqlen) : 1;  // (single tokens: the form that adds slices)
  const int64_t round = a->width <= 1024 ? 1024 : a->width <= 2048 ? 512 : 256;
  for (int64_t most = round; !run; most += round) {
    const int64_t per_sequence = most / a->batch;
    if (per_sequence > 0 && (a->seqlen + per_sequence - 1) / per_sequence <= 32) run = static_cast<int>((a->seqlen + per_sequence - 1) / per_sequence);
    if (a->seqlen <= 32 && per_sequence == 0) run = static_cast<int>(a->seqlen);
  }
  const int64_t runs = (a->seqlen + run - 1) / run;
  // without a convolution the kernel walks over rows, as many as runs of 32 would be workgroups
  if (a->batch * (a->conv ? runs : (a->seqlen + 31) / 32) > INT32_MAX) return E2H_ERR_BAD_SHAPE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (a->dtype == E2H_SEQ_BF16) launch_norm_conv<bf16_t>(*a, sums, static_cast<int>(runs), run, s);
  else launch_norm_conv<float>(*a, sums, static_cast<int>(runs), run, s);
  return launch_status();
}
}  // namespace

extern "C" int e2h_seq_norm_conv(const e2h_norm_conv_args *a, void *stream) { return norm_conv(a, DeltaSums{}, stream); }

extern "C" int e2h_seq_norm_conv_sums(const e2h_norm_conv_args *a, const float *sums, int slices, void *stream) {
  if (!a || !sums) return E2H_ERR_NULL_POINTER;
  if (slices < 1 || slices > 4 || a->seqlen != 1 || a->delta || a->terms || a->norm_kind != E2H_SEQ_RMS_NORM) return E2H_ERR_BAD_SHAPE;
  if (!aligned16(sums)) return E2H_ERR_MISALIGNED;
  return norm_conv(a, DeltaSums{sums, slices}, stream);
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

extern "C" int e2h_seq_embed_rows(const void *table, const int64_t *tokens, float *x, void *h, int64_t rows, int64_t width, int64_t table_rows, void *stream) {
  if (!table || !tokens || !x) return E2H_ERR_NULL_POINTER;
  if (rows < 1 || width < 8 || width % 8 != 0 || width > INT32_MAX || table_rows < 1) return E2H_ERR_BAD_SHAPE;
  const int64_t pieces = rows * (width / 8), blocks = (pieces + 255) / 256;
  if (blocks > INT32_MAX / 256) return E2H_ERR_BAD_SHAPE;
  if (!aligned16(table) || !aligned16(x) || !aligned16(h) || (reinterpret_cast<uintptr_t>(tokens) & 7u)) return E2H_ERR_MISALIGNED;
  hipLaunchKernelGGL(embed_rows_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, static_cast<hipStream_t>(stream), static_cast<const bf16_t *>(table), tokens, x,
                     static_cast<bf16_t *>(h), pieces, static_cast<int>(width / 8), table_rows);
  return launch_status();
}
