// int8 per-channel dequant GEMV / skinny GEMM / GEMM, streaming versions (16-byte aligned rows).
//
// Replaces  F.linear(x, weight.to(bf16)) * scales  (reference models/quantize.py:428-429).
//
//   q int8 [N][K] row-major (checkpoint layout), scales bf16 [N], x bf16 [M][K], y bf16 [M][N].
//
// Up to 64 rows: the streamed-weights kernel of e2h_stream.h with the epilogues below (plain, gated, rotary + cache write).
// Measured at one row, 7B shapes (the kernel that this replaces in brackets): 12288 x 4096 11.9 us (18.2), 4096 x 4096 5.9 and
// 4096 x 11008 11.3 (11.8 on average), gated 2 x 11008 x 4096 18.4 (29.3), 32000 x 4096 26.5 (29.3); at 32 rows 15.0, 8.6, 18.4,
// 22.8, 30.2.  A launch that only reads the same bytes in the same pattern takes 16.3 for the gated one.
//
// More rows (K % 128 == 0): int8_stream_mm_kernel, a workgroup = 4 column waves, each wave T tiles of 16 weight rows and 64 rows of x.
// Lane L = 16*b + c of v_mfma_f32_16x16x32_bf16 owns weight row n0 + c; per 64-wide half chunk it loads the 16 consecutive bytes
// k = 64h + 16b .. +15 (one buffer_load_dwordx4): bytes 0..7 feed MFMA step 2h, bytes 8..15 step 2h + 1.  The matching
// activation fragment is 16 contiguous bytes of x, staged into LDS one phase at a time in fragment order.  From enough 128 x 128
// tiles on, the 32x32-tile kernels of e2h_int8_gemm.hip.
//
// int8 -> bf16 is exact (sign-extending byte convert, keep the high half).  No per-group arithmetic: the float32 accumulators
// run over all of K and the epilogue reproduces the reference's two roundings, bf16(acc) then bf16(t * scale).
#include <type_traits>

#include "e2h_common.h"
#include "e2h_stream.h"

namespace e2h {
namespace {

constexpr int kChunk = 128;             // k per pipeline chunk
constexpr int kSteps = 4;               // MFMA steps per chunk
constexpr int kPPR = kChunk / 8;        // 16-byte activation pieces per row per chunk
constexpr int kFragBytes = 1024 + 64;   // one fragment block in LDS (+ pad)

constexpr int kColWaves = 4, kRowTiles = 4;  // a workgroup: 64 rows x 64 T columns
constexpr int NB = 2, PD = NB - 1;           // ring of weight chunks (2 KB per tile each)
constexpr int CPP = 2, XD = 1;               // chunks per phase of activations, phases that are loaded ahead

template <int T>
struct WeightRegs8 {
  u32x4_t w[T][2];
};

// ---- epilogues of the streamed-weights kernel: a unit is 16 columns x 16 rows, this lane column n and rows m0 .. m0 + 3 --------

__device__ __forceinline__ float column_scale(const uint16_t *scales, int n, int N) { return bf16_to_f32(scales[n < N ? n : N - 1]); }
// the linear's bfloat16 output: bf16(bf16(acc) * scale)
__device__ __forceinline__ float int8_linear(float acc, float scale) { return bf16_round(bf16_round(acc) * scale); }

struct Plain8 {
  static constexpr bool kGate = false, kHalves = false;
  struct Args {
    const uint16_t *scales;
    uint16_t *y;
  };
  float scale;
  __device__ __forceinline__ void load(const Args &a, int n, int N) { scale = column_scale(a.scales, n, N); }
  __device__ __forceinline__ void finish(const Args &a, f32x4_t acc, f32x4_t, int m0, int M, int n, int N) const {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (n < N && m0 + r < M) a.y[static_cast<size_t>(m0 + r) * N + n] = f32_to_bf16_rne(bf16_round(acc[r]) * scale);
  }
};

// the same columns of two weight matrices, the gate and up projections of a feed-forward block: bf16(bf16(silu(g)) * u) with g, u
// the two linears' bfloat16 outputs -- the rounding points of F.silu(w1(x)) * w3(x) on bfloat16 tensors (reference
// models/model.py:343-344)
struct Gate8 {
  static constexpr bool kGate = true, kHalves = false;
  struct Args {
    const uint16_t *scales, *scales2;
    uint16_t *y;
  };
  float s_gate, s_up;
  __device__ __forceinline__ void load(const Args &a, int n, int N) {
    s_gate = column_scale(a.scales, n, N);
    s_up = column_scale(a.scales2, n, N);
  }
  __device__ __forceinline__ void finish(const Args &a, f32x4_t g, f32x4_t u, int m0, int M, int n, int N) const {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float gate = int8_linear(g[r], s_gate), up = int8_linear(u[r], s_up);
      const float act = bf16_round(gate / (1.0f + expf(-gate)));
      if (n < N && m0 + r < M) a.y[static_cast<size_t>(m0 + r) * N + n] = f32_to_bf16_rne(act * up);
    }
  }
};

// the fused q | k | v projection of ONE new token per sequence (row m = sequence m): the bfloat16 output is rotated in float32 by the
// angle of position input_pos[0] (interleaved pairs, reference models/model.py:400-412); q goes to q_out [B, H, D], k and v into
// the caches [B, Hkv, S, D] at that position (KVCache.update, reference models/model.py:94-104)
struct Rope8 {
  static constexpr bool kGate = false, kHalves = false;
  struct Args {
    const uint16_t *scales, *freqs;  // freqs [>= S, D/2, 2] bf16 (cos, sin)
    uint16_t *q_out, *kc, *vc;
    const int64_t *input_pos;        // [1] on the device
    int H, Hkv, S, D;
  };
  float scale, cs, sn;
  int pos;
  // cos / sin depend on a position read from memory: both are fetched behind the first weight loads instead of as two dependent
  // round trips at the very end
  __device__ __forceinline__ void load(const Args &a, int n, int N) {
    scale = column_scale(a.scales, n, N);
    const int64_t p = a.input_pos[0];
    pos = p >= 0 && p < a.S ? static_cast<int>(p) : -1;
    cs = 1.f;
    sn = 0.f;
    if (n < N && pos >= 0 && n < (a.H + a.Hkv) * a.D) {
      const uint32_t f = reinterpret_cast<const uint32_t *>(a.freqs)[static_cast<size_t>(pos) * (a.D / 2) + ((n % a.D) >> 1)];
      cs = __builtin_bit_cast(float, f << 16);
      sn = __builtin_bit_cast(float, f & 0xFFFF0000u);
    }
  }
  __device__ __forceinline__ void finish(const Args &a, f32x4_t acc, f32x4_t, int m0, int M, int n, int N) const {
    const int head = n / a.D, d = n % a.D;
    const bool in_range = n < N && pos >= 0, rotated = head < a.H + a.Hkv;
    uint16_t *dst;  // row 0's element of this column; rows are row_stride apart
    size_t row_stride;
    if (head < a.H) {
      dst = a.q_out + static_cast<size_t>(head) * a.D + d;
      row_stride = static_cast<size_t>(a.H) * a.D;
    } else {
      const int hk = rotated ? head - a.H : head - a.H - a.Hkv;
      dst = (rotated ? a.kc : a.vc) + (static_cast<size_t>(hk) * a.S + (pos < 0 ? 0 : pos)) * a.D + d;
      row_stride = static_cast<size_t>(a.Hkv) * a.S * a.D;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float own = int8_linear(acc[r], scale);
      const float other = __shfl_xor(own, 1);  // the pair's other column lives in the neighbouring lane
      // even column: x0 * cos - x1 * sin; odd column: x1 * cos + x0 * sin (two rounded products, then the sum)
      const float rot = (n & 1) ? own * cs + other * sn : own * cs - other * sn;
      if (in_range && m0 + r < M) dst[static_cast<size_t>(m0 + r) * row_stride] = f32_to_bf16_rne(rotated ? rot : own);
    }
  }
};

// the unscaled float32 sums over the two halves of K, row-major [2][M][N]; the residual add + RMSNorm that follows adds them and applies the
// column scales with the two roundings.  (A workgroup computes both: cutting K over two workgroups gains 1 us at 4096 x 4096 and 4 us at
// 4096 x 11008 and 32 rows, nothing at one row, and would cost the plain form, which has to give the same sums, a meeting of two workgroups.)
struct Partial8 {
  static constexpr bool kGate = false, kHalves = true;
  struct Args {
    float *out;
  };
  __device__ __forceinline__ void load(const Args &, int, int) {}
  __device__ __forceinline__ void finish(const Args &a, f32x4_t lo, f32x4_t hi, int m0, int M, int n, int N) const {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (n >= N || m0 + r >= M) continue;
      a.out[static_cast<size_t>(m0 + r) * N + n] = lo[r];
      a.out[static_cast<size_t>(M + m0 + r) * N + n] = hi[r];
    }
  }
};

// ---- more than 64 rows ------------------------------------------------------------------------------------------------
// What is too little work for the 32x32-tile kernels: few rows, or a head of one or two columns over many.  A chunk is one round of LDS
// reads, products and a barrier, so its latency is the time.  The activations' fragments are read before the chunk's loads are issued
// (behind the fence that keeps those in place they waited for the issue), and waves past the last column only help with staging: with
// one column the fragment reads of the other three took most of the LDS bandwidth.  us before / fragments first / and idle waves out,
// K = 4096: 65 rows x 1 column 26.7 / 24.9 / 17.6, 4096 x 1 30.3 / 28.5 / 21.8, 65 x 4096 31.7 / 29.4 / 28.9, 512 x 1024 31.4 / 29.2 / 28.8.

template <int T>
__global__ __launch_bounds__(64 * kColWaves) void int8_stream_mm_kernel(const uint16_t *__restrict__ x, const int8_t *__restrict__ q,
                                                                        const uint16_t *__restrict__ scales, uint16_t *__restrict__ y,
                                                                        int M, int N, int K) {
  constexpr int MT = kRowTiles;
  constexpr int U = NB > CPP * XD ? NB : CPP * XD;
  constexpr int kThreads = kColWaves * 64;
  constexpr int kPieces = 16 * MT * kPPR;
  constexpr int kPhasePieces = CPP * kPieces;
  constexpr int kPiecesPerThread = (kPhasePieces + kThreads - 1) / kThreads;
  constexpr int kBufBytes = MT * kSteps * kFragBytes;
  constexpr int kStageBytes = CPP * kBufBytes;
  __shared__ __attribute__((aligned(16))) uint8_t lds[2 * kStageBytes];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15;
  const int b = lane >> 4;
  const int nchunks = K / kChunk;
  const int tile16_0 = (blockIdx.x * kColWaves + wave) * T;
  const int m_base = blockIdx.z * (16 * MT);

  uint32_t wlane[T];
#pragma unroll
  for (int t = 0; t < T; ++t) {
    int n = 16 * (tile16_0 + t) + c;
    n = n < N ? n : N - 1;
    wlane[t] = static_cast<uint32_t>(static_cast<size_t>(n) * K + 16 * b);
  }
  const __amdgpu_buffer_rsrc_t w_rsrc = make_rsrc(q, static_cast<uint32_t>(static_cast<size_t>(N) * K));
  const __amdgpu_buffer_rsrc_t x_rsrc = make_rsrc(x, static_cast<uint32_t>(static_cast<size_t>(M) * K * 2));

  auto load_weights = [&](WeightRegs8<T> &r, int ci) {
    const uint32_t so = static_cast<uint32_t>(ci) * kChunk;
#pragma unroll
    for (int t = 0; t < T; ++t) {
      r.w[t][0] = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, wlane[t], so, 2);
      r.w[t][1] = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, wlane[t], so + 64, 2);
    }
  };

  // activation staging: piece `within` (0..15) of a row's 128-wide chunk covers k = 8*within .. +7, which is the
  // fragment of lane block b = (within % 8) / 2 in MFMA step 2 * (within / 8) + within % 2
  uint32_t xsrc[kPiecesPerThread];
  int xdst[kPiecesPerThread];
  int xq[kPiecesPerThread];
#pragma unroll
  for (int i = 0; i < kPiecesPerThread; ++i) {
    const int p = tid + i * kThreads;
    const int qc = (p / kPieces) < CPP ? (p / kPieces) : CPP - 1;
    const int pc = p % kPieces;
    int row = pc / kPPR;
    const int within = pc % kPPR;
    const int s = 2 * (within >> 3) + (within & 1), bb = (within & 7) >> 1;
    xq[i] = qc;
    xdst[i] = qc * kBufBytes + ((row >> 4) * kSteps + s) * kFragBytes + (bb * 16 + (row & 15)) * 16;
    row += m_base;
    row = row < M ? row : M - 1;
    xsrc[i] = static_cast<uint32_t>((static_cast<size_t>(row) * K + within * 8) * 2);
  }
  auto chunk_at = [&](int i) { return i < nchunks ? i : nchunks - 1; };
  auto load_x = [&](u32x4_t (&r)[kPiecesPerThread], int phase) {
#pragma unroll
    for (int i = 0; i < kPiecesPerThread; ++i)
      if (kPhasePieces % kThreads == 0 || tid + i * kThreads < kPhasePieces)
        r[i] = __builtin_amdgcn_raw_buffer_load_b128(x_rsrc, xsrc[i], static_cast<uint32_t>(chunk_at(phase * CPP + xq[i])) * (kChunk * 2), 0);
  };
  auto store_x = [&](const u32x4_t (&r)[kPiecesPerThread], int parity) {
    uint8_t *buf = lds + (parity & 1) * kStageBytes;
#pragma unroll
    for (int i = 0; i < kPiecesPerThread; ++i)
      if (kPhasePieces % kThreads == 0 || tid + i * kThreads < kPhasePieces)
        *reinterpret_cast<u32x4_t *>(buf + xdst[i]) = r[i];
  };

  f32x4_t acc[T][MT];
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[t][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  bf16x8_t xf[MT][kSteps];
  auto read_x = [&](int parity, int qc) {
    const uint8_t *buf = lds + (parity & 1) * kStageBytes + qc * kBufBytes + lane * 16;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int s = 0; s < kSteps; ++s) xf[mt][s] = *reinterpret_cast<const bf16x8_t *>(buf + (mt * kSteps + s) * kFragBytes);
  };
  auto compute_chunk = [&](const WeightRegs8<T> &r, uint32_t live) {
#pragma unroll
    for (int t = 0; t < T; ++t) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        // live == 0 (padding iteration): zero weights contribute nothing
        u32x4_t w = r.w[t][h];
#pragma unroll
        for (int d = 0; d < 4; ++d) w[d] &= live;
        const bf16x8_t w0 = stream::Int8Weights::operand(w, 0), w1 = stream::Int8Weights::operand(w, 1);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          acc[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[mt][2 * h], w0, acc[t][mt], 0, 0, 0);
          acc[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[mt][2 * h + 1], w1, acc[t][mt], 0, 0, 0);
        }
      }
    }
  };

  WeightRegs8<T> ring[NB];
  u32x4_t xstage[XD][kPiecesPerThread];
#pragma unroll
  for (int d = 0; d < XD; ++d) load_x(xstage[d], d);
#pragma unroll
  for (int i = 0; i < PD; ++i) load_weights(ring[i], chunk_at(i));
  store_x(xstage[0], 0);
  lds_barrier();
  const auto chunks = [&](auto has_columns) {
    for (int base = 0; base < nchunks; base += U) {
#pragma unroll
      for (int j = 0; j < U; ++j) {
        const int i = base + j;
        const int phase = i / CPP;
        const uint32_t live = i < nchunks ? 0xFFFFFFFFu : 0u;
        if constexpr (has_columns) read_x(phase, j % CPP);
        if (j % CPP == 0) load_x(xstage[(j / CPP) % XD], phase + XD);
        if constexpr (has_columns) {
          load_weights(ring[(j + PD) % NB], chunk_at(i + PD));
          __builtin_amdgcn_sched_barrier(0);  // the scheduler would sink the loads to their first use (65 rows, 4096 x 4096: 40 us, so 31)
          compute_chunk(ring[j % NB], live);
        }
        if (j % CPP == CPP - 1) {
          store_x(xstage[(j / CPP + 1) % XD], phase + 1);
          lds_barrier();
        }
      }
    }
  };
  if (16 * tile16_0 >= N) {
    chunks(std::false_type{});
    return;
  }
  chunks(std::true_type{});

#pragma unroll
  for (int t = 0; t < T; ++t) {
    const int n = 16 * (tile16_0 + t) + c;
    const float scale = bf16_to_f32(scales[n < N ? n : N - 1]);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m_base + 16 * mt + 4 * b + r;
        if (n < N && m < M) {
          const float lin = bf16_round(acc[t][mt][r]);                              // F.linear output in bfloat16
          y[static_cast<size_t>(m) * N + n] = f32_to_bf16_rne(lin * scale);        // * self.scales
        }
      }
  }
}

template <int T>
int launch8(const uint16_t *x, const int8_t *q, const uint16_t *scales, uint16_t *y, int M, int N, int K, hipStream_t stream) {
  const int tiles16 = (N + 15) / 16;
  dim3 grid((tiles16 + kColWaves * T - 1) / (kColWaves * T), 1, (M + 16 * kRowTiles - 1) / (16 * kRowTiles));
  hipLaunchKernelGGL((int8_stream_mm_kernel<T>), grid, dim3(64 * kColWaves), 0, stream, x, q, scales, y, M, N, K);
  return launch_status();
}

constexpr int kCUs8 = 256;

// shapes whose sums a following norm may take: the two halves of K
int partial_slices8_for(int64_t m, int64_t n, int64_t k) {
  if (m < 1 || m > 64 || n < 8 || (n % 8) != 0 || k < 128 || (k % 128) != 0 || n > INT32_MAX || k > INT32_MAX || n * k >= (int64_t{1} << 32))
    return E2H_ERR_BAD_SHAPE;
  if (m > 32 && (n + 63) / 64 >= kCUs8) return E2H_ERR_BAD_SHAPE;  // never offered: wider than any model's residual stream
  return stream::takes(m, n, k, 1) ? 2 : E2H_ERR_BAD_SHAPE;
}

}  // namespace

// Streaming int8 matmul; the caller has checked pointers, 16-byte aligned x and q, and either M <= 64 and stream::takes or K % 128 == 0.
int int8_stream_mm(const uint16_t *x, const int8_t *q, const uint16_t *scales, uint16_t *y, int M, int N, int K, hipStream_t stream) {
  if (stream::takes(M, N, K, 1)) return stream::run<stream::Int8Weights, Plain8>({x, q, q, M, N, K}, {scales, y}, stream);
  const int tiles16 = (N + 15) / 16;
  const int m_chunks = (M + 16 * kRowTiles - 1) / (16 * kRowTiles);
  int t = (static_cast<long long>((tiles16 + 7) / 8) * m_chunks >= kCUs8) ? 2 : 1;
  if (options().int8_rows_per_wave == 16 || options().int8_rows_per_wave == 32) t = options().int8_rows_per_wave / 16;
  const int64_t rows_by_bytes = ((int64_t{1} << 32) - 1) / (2 * static_cast<int64_t>(K));
  const int64_t rows_by_grid = int64_t{65535} * 16 * kRowTiles;
  int64_t max_rows = rows_by_bytes < rows_by_grid ? rows_by_bytes : rows_by_grid;
  max_rows -= max_rows % (16 * kRowTiles);
  if (max_rows < 16 * kRowTiles) return E2H_ERR_BAD_SHAPE;
  for (int64_t m0 = 0; m0 < M; m0 += max_rows) {
    const uint16_t *xs = x + m0 * K;
    uint16_t *ys = y + m0 * N;
    const int rows = static_cast<int>(M - m0 < max_rows ? M - m0 : max_rows);
    const long long wgs32 = static_cast<long long>((rows + 127) / 128) * ((N + 127) / 128);
    const bool use32 = options().int4_gemm32_min_rows > 0 ? rows >= options().int4_gemm32_min_rows : wgs32 >= 320;
    int rc;
    if (use32 && !options().int4_no_gemm32 && static_cast<int64_t>(N) * K < (int64_t{1} << 32))
      rc = int8_gemm32(xs, q, scales, ys, rows, N, K, stream);  // many rows: 32x32-tile kernels, no scratch
    else
      rc = t == 2 ? launch8<2>(xs, q, scales, ys, rows, N, K, stream) : launch8<1>(xs, q, scales, ys, rows, N, K, stream);
    if (rc != E2H_OK) return rc;
  }
  return E2H_OK;
}

}  // namespace e2h

extern "C" int e2h_int8_mm_silu_gate(const uint16_t *x, const int8_t *q_gate, const uint16_t *scales_gate, const int8_t *q_up,
                                     const uint16_t *scales_up, uint16_t *y, int64_t m, int64_t n, int64_t k, void *stream) {
  using namespace e2h;
  if (!x || !q_gate || !scales_gate || !q_up || !scales_up || !y) return E2H_ERR_NULL_POINTER;
  if (m < 1 || m > 64 || n < 1 || k < 128 || (k % 128) != 0 || n > INT32_MAX || k > INT32_MAX || n * k >= (int64_t{1} << 32)) return E2H_ERR_BAD_SHAPE;
  if (!aligned16(x) || !aligned16(q_gate) || !aligned16(q_up) || (reinterpret_cast<uintptr_t>(scales_gate) & 1u) ||
      (reinterpret_cast<uintptr_t>(scales_up) & 1u) || (reinterpret_cast<uintptr_t>(y) & 1u))
    return E2H_ERR_MISALIGNED;
  if (!stream::takes(m, n, k, 1)) return E2H_ERR_BAD_SHAPE;
  return stream::run<stream::Int8Weights, Gate8>({x, q_gate, q_up, static_cast<int>(m), static_cast<int>(n), static_cast<int>(k)},
                                                 {scales_gate, scales_up, y}, static_cast<hipStream_t>(stream));
}

extern "C" int e2h_int8_mm_rope_kv(const uint16_t *x, const int8_t *q, const uint16_t *scales, const uint16_t *freqs_cis, uint16_t *q_out,
                                   uint16_t *k_cache, uint16_t *v_cache, const int64_t *input_pos, int64_t batch, int64_t n_head,
                                   int64_t n_kv_head, int64_t head_dim, int64_t cache_len, int64_t k, void *stream) {
  using namespace e2h;
  if (!x || !q || !scales || !freqs_cis || !q_out || !k_cache || !v_cache || !input_pos) return E2H_ERR_NULL_POINTER;
  if (batch < 1 || batch > 64 || n_head < 1 || n_kv_head < 1 || head_dim < 2 || (head_dim % 2) != 0 || cache_len < 1 || k < 128 || (k % 128) != 0)
    return E2H_ERR_BAD_SHAPE;
  const int64_t n = (n_head + 2 * n_kv_head) * head_dim;
  if (n > INT32_MAX || k > INT32_MAX || cache_len > INT32_MAX || n * k >= (int64_t{1} << 32)) return E2H_ERR_BAD_SHAPE;
  if (!aligned16(x) || !aligned16(q) || (reinterpret_cast<uintptr_t>(scales) & 1u) || (reinterpret_cast<uintptr_t>(freqs_cis) & 3u) ||
      (reinterpret_cast<uintptr_t>(q_out) & 1u) || (reinterpret_cast<uintptr_t>(k_cache) & 1u) || (reinterpret_cast<uintptr_t>(v_cache) & 1u) ||
      (reinterpret_cast<uintptr_t>(input_pos) & 7u))
    return E2H_ERR_MISALIGNED;
  if (!stream::takes(batch, n, k, 1)) return E2H_ERR_BAD_SHAPE;
  return stream::run<stream::Int8Weights, Rope8>({x, q, q, static_cast<int>(batch), static_cast<int>(n), static_cast<int>(k)},
                                                 {scales, freqs_cis, q_out, k_cache, v_cache, input_pos, static_cast<int>(n_head),
                                                  static_cast<int>(n_kv_head), static_cast<int>(cache_len), static_cast<int>(head_dim)},
                                                 static_cast<hipStream_t>(stream));
}

extern "C" int e2h_int8_mm_partial_slices(int64_t m, int64_t n, int64_t k) { return e2h::partial_slices8_for(m, n, k); }

extern "C" int e2h_int8_mm_partials(const uint16_t *x, const int8_t *q, float *partials, int64_t m, int64_t n, int64_t k, int slices,
                                    void *stream) {
  using namespace e2h;
  if (!x || !q || !partials) return E2H_ERR_NULL_POINTER;
  const int want = partial_slices8_for(m, n, k);
  if (want < 0) return want;
  if (slices != want) return E2H_ERR_BAD_SHAPE;
  if (!aligned16(x) || !aligned16(q) || (reinterpret_cast<uintptr_t>(partials) & 3u)) return E2H_ERR_MISALIGNED;
  return stream::run<stream::Int8Weights, Partial8>({x, q, q, static_cast<int>(m), static_cast<int>(n), static_cast<int>(k)}, {partials},
                                                    static_cast<hipStream_t>(stream));
}

// ---- the same three behind the norm that makes their rows ---------------------------------------------------------------------------
namespace e2h {
namespace {
int check_norm(const e2h_row_norm *norm, int64_t m, int64_t n, int64_t k) {
  if (!norm || !norm->x || !norm->weight || (norm->partials && !norm->h_out)) return E2H_ERR_NULL_POINTER;
  if (!e2h_int8_norm_mm_supported(m, n, k) || (norm->partials && (norm->slices < 1 || norm->slices > 2))) return E2H_ERR_BAD_SHAPE;
  if (!aligned16(norm->x) || !aligned16(norm->partials) || !aligned16(norm->col_scales) || !aligned16(norm->weight) || !aligned16(norm->h_out)) return E2H_ERR_MISALIGNED;
  return E2H_OK;
}
stream::RowNorm row_norm(const e2h_row_norm &n) { return {n.x, n.partials, n.partials ? n.col_scales : nullptr, n.weight, n.h_out, n.slices, n.eps}; }
}  // namespace
}  // namespace e2h

extern "C" int e2h_int8_norm_mm_supported(int64_t m, int64_t n, int64_t k) {
  return n >= 1 && n <= INT32_MAX && e2h::stream::norm_fits(m, k) && n * k < (int64_t{1} << 32) && e2h::stream::takes(m, n, k, 1) ? 1 : 0;
}

extern "C" int e2h_int8_norm_mm(const e2h_row_norm *norm, const int8_t *q, const uint16_t *scales, uint16_t *y, int64_t m, int64_t n, int64_t k, void *stream) {
  using namespace e2h;
  if (!q || !scales || !y) return E2H_ERR_NULL_POINTER;
  const int rc = check_norm(norm, m, n, k);
  if (rc != E2H_OK) return rc;
  if (!aligned16(q) || (reinterpret_cast<uintptr_t>(scales) & 1u) || (reinterpret_cast<uintptr_t>(y) & 1u)) return E2H_ERR_MISALIGNED;
  return stream::run_norm<stream::Int8Weights, Plain8>({norm->x, q, q, static_cast<int>(m), static_cast<int>(n), static_cast<int>(k)}, {scales, y}, row_norm(*norm),
                                                       static_cast<hipStream_t>(stream));
}

extern "C" int e2h_int8_norm_mm_silu_gate(const e2h_row_norm *norm, const int8_t *q_gate, const uint16_t *scales_gate, const int8_t *q_up, const uint16_t *scales_up,
                                          uint16_t *y, int64_t m, int64_t n, int64_t k, void *stream) {
  using namespace e2h;
  if (!q_gate || !scales_gate || !q_up || !scales_up || !y) return E2H_ERR_NULL_POINTER;
  const int rc = check_norm(norm, m, n, k);
  if (rc != E2H_OK) return rc;
  if (!aligned16(q_gate) || !aligned16(q_up) || ((reinterpret_cast<uintptr_t>(scales_gate) | reinterpret_cast<uintptr_t>(scales_up) | reinterpret_cast<uintptr_t>(y)) & 1u))
    return E2H_ERR_MISALIGNED;
  return stream::run_norm<stream::Int8Weights, Gate8>({norm->x, q_gate, q_up, static_cast<int>(m), static_cast<int>(n), static_cast<int>(k)}, {scales_gate, scales_up, y},
                                                      row_norm(*norm), static_cast<hipStream_t>(stream));
}

extern "C" int e2h_int8_norm_mm_rope_kv(const e2h_row_norm *norm, const int8_t *q, const uint16_t *scales, const uint16_t *freqs_cis, uint16_t *q_out, uint16_t *k_cache,
                                        uint16_t *v_cache, const int64_t *input_pos, int64_t batch, int64_t n_head, int64_t n_kv_head, int64_t head_dim, int64_t cache_len,
                                        int64_t k, void *stream) {
  using namespace e2h;
  if (!q || !scales || !freqs_cis || !q_out || !k_cache || !v_cache || !input_pos) return E2H_ERR_NULL_POINTER;
  if (n_head < 1 || n_kv_head < 1 || head_dim < 2 || (head_dim % 2) != 0 || cache_len < 1 || cache_len > INT32_MAX || n_head > INT32_MAX || n_kv_head > INT32_MAX ||
      head_dim > INT32_MAX / (n_head + 2 * n_kv_head))
    return E2H_ERR_BAD_SHAPE;
  const int64_t n = (n_head + 2 * n_kv_head) * head_dim;
  const int rc = check_norm(norm, batch, n, k);
  if (rc != E2H_OK) return rc;
  if (!aligned16(q) || (reinterpret_cast<uintptr_t>(scales) & 1u) || (reinterpret_cast<uintptr_t>(freqs_cis) & 3u) || (reinterpret_cast<uintptr_t>(q_out) & 1u) ||
      (reinterpret_cast<uintptr_t>(k_cache) & 1u) || (reinterpret_cast<uintptr_t>(v_cache) & 1u) || (reinterpret_cast<uintptr_t>(input_pos) & 7u))
    return E2H_ERR_MISALIGNED;
  return stream::run_norm<stream::Int8Weights, Rope8>({norm->x, q, q, static_cast<int>(batch), static_cast<int>(n), static_cast<int>(k)},
                                                      {scales, freqs_cis, q_out, k_cache, v_cache, input_pos, static_cast<int>(n_head), static_cast<int>(n_kv_head),
                                                       static_cast<int>(cache_len), static_cast<int>(head_dim)},
                                                      row_norm(*norm), static_cast<hipStream_t>(stream));
}
