// Decode-batch int4 matmul on staged activations: staging pass, arg-max reduction, choice of geometry and entry points.  The kernel: e2h_int4_staged_kernel.h.
#include "e2h_int4_staged.h"

namespace e2h {
namespace {

using namespace staged;

constexpr int kCUs = 256;

// arg-max: the candidates of all column blocks of a row -> the row's token (one wave per row)
__global__ __launch_bounds__(64) void argmax_candidates_kernel(const unsigned long long *__restrict__ cand, int blocks, int M, int64_t *__restrict__ out) {
  const int m = blockIdx.x;
  unsigned long long best = 0ull;
  for (int i = threadIdx.x; i < blocks; i += 64) {
    const unsigned long long v = cand[static_cast<size_t>(i) * M + m];
    best = v > best ? v : best;
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const unsigned long long other = __shfl_xor(best, off);
    best = other > best ? other : best;
  }
  if (threadIdx.x == 0) out[m] = static_cast<int64_t>(~static_cast<uint32_t>(best & 0xFFFFFFFFull));
}

// ---- staging pass: row-major activations -> operand order + sums of 16 ------------------------------------------------
// One thread per 16-byte piece (8 values); rows M .. Mpad-1 are written as zeros.
__global__ __launch_bounds__(256) void int4_stage_x_kernel(const uint16_t *__restrict__ x, StagedOut out, int M, int K) {
  const int pieces_per_row = K >> 3;
  const int idx = blockIdx.x * 256 + threadIdx.x;
  const int m = idx / pieces_per_row, pc = idx % pieces_per_row;
  if (m >= out.mpad) return;  // pieces_per_row is even: both lanes of a pair leave or stay
  u32x4_t raw = {0u, 0u, 0u, 0u};
  if (m < M) raw = *reinterpret_cast<const u32x4_t *>(x + static_cast<size_t>(m) * K + pc * 8);
  staged_store_piece(out, m, pc, raw);
}

// ---- launch geometry ---------------------------------------------------------------------------------------------------
template <int EPI>
int dispatch_staged(const StagedArgs &a, int groupsize, const Geometry &g, hipStream_t stream) {
  switch (groupsize) {
    case 32: return launch_group<32>(EPI, a, g, stream);
    case 64: return launch_group<64>(EPI, a, g, stream);
    case 128: return launch_group<128>(EPI, a, g, stream);
  }
  return E2H_ERR_BAD_GROUPSIZE;
}

int check_shape(int64_t m, int64_t n, int64_t k, int groupsize) {
  if (groupsize != 32 && groupsize != 64 && groupsize != 128) return E2H_ERR_BAD_GROUPSIZE;
  if (m < 1 || m > 64 || n < 16 || (n % 16) != 0 || k < 128 || n > INT32_MAX || k > INT32_MAX) return E2H_ERR_BAD_SHAPE;
  if ((k % 128) != 0) return E2H_ERR_BAD_INNER_K_TILES;
  if (n * k / 2 >= (int64_t{1} << 32) || (k / groupsize) * n * 4 >= (int64_t{1} << 32)) return E2H_ERR_BAD_SHAPE;
  return E2H_OK;
}

// fills the shape part of the arguments and picks the geometry; false where there is none
bool plan(StagedArgs *a, Geometry *g, const void *staged, int64_t m, int64_t n, int64_t k, int groupsize, int epi) {
  a->M = static_cast<int>(m);
  a->Mpad = staged_mpad(m);
  a->N = static_cast<int>(n);
  a->K = static_cast<int>(k);
  a->frag = static_cast<const uint8_t *>(staged);
  a->sums = reinterpret_cast<const float *>(a->frag + static_cast<size_t>(a->Mpad) * k * 2);
  const int tiles16 = static_cast<int>(n / 16), kt = static_cast<int>(k / 128);
  const bool gate = epi == kStGate;
  // Above 32 rows: four row tiles per workgroup, so that the weights are read once, or two workgroups of two row tiles each while the weights
  // are small enough for L2 to hand them out twice and too small to fill the chip (64 rows, group size 128, us, one / two: 1024 x 2048 6.9 / 5.3,
  // 6144 x 4096 with the rotation 13.0 / 10.9, 2 x 5504 x 2048 gated 12.0 / 11.5, 4096 x 4096 with its norm 13.5 / 13.0; 12288 x 4096
  // 15.0 / 14.3 but 13.4 / 13.8 at 33 rows, 4096 x 11008 with its norm 19.2 / 19.7, 10240 x 8192 26.3 / 29.0, 2 x 11008 x 4096 24.7 / 27.4).
  const int halves = a->M > 32 && n * k * (gate ? 2 : 1) <= (int64_t{1} << 25) ? 2 : 1;
  const int mt = a->M <= 16 ? 1 : a->M <= 32 || halves == 2 ? 2 : 4;
  const int want_t = options().staged_tiles, want_s = options().staged_slices;  // experiments: force a geometry
  // The geometry with the least cost; the weights of the cost were fitted to a sweep over T and S, with workgroups of eight waves throughout, at 1 .. 64 rows of the shapes above and
  // 12288 / 4096 / 32000 x 4096: the chosen geometry was within 6 % of the best one there, and the 7B, 13B and 34B shapes have kept theirs.  One round of 256 workgroups with many tiles
  // beats two rounds with few (of eight waves: w1|w3 22016 x 8192, 1 row: T = 12 43.6 us, T = 8 46.0; 32000 x 4096: T = 8 14.6, T = 6 19.0); K slices pay
  // while a round is not full (w2 4096 x 11008, 32 rows: T = 4, S = 4 10.1 us, the best with S = 1 15.6).  What a slice costs the norm that
  // adds it grows with rows and columns: fitted with the norm's time, in the same form, to 1 .. 64 rows of 1024 x 2048 .. 8192 x 22016 at every group size, where
  // the choice was within 0.2 % of the best one on average and 6 % at most (one unit per slice whatever its size: 2.6 %, 31 %; 8192 x 8192 at
  // group size 128 and 32 rows 19.9 us, now 18.6; 4096 x 4096 at group size 64 and 64 rows 15.5, now 13.7).
  double best_cost = -1;
  for (int s = 1; s <= (epi == kStPartial ? 8 : 1) && s <= kt; s *= 2) {
    if (want_s && epi == kStPartial && s != want_s) continue;
    for (int t : {1, 2, 3, 4, 6, 8, 12}) {
      if (t > max_tiles(groupsize, mt, gate) || (gate && t % 2) || (want_t && !gate && t != want_t)) continue;
      const int tc = gate ? t / 2 : t;
      const long wgs = static_cast<long>((tiles16 + tc - 1) / tc) * s * halves;
      const long rounds = (wgs + kCUs - 1) / kCUs;
      const double chunks = static_cast<double>(kt) / s / 8;
      // per workgroup: a fixed part, per chunk its weight tiles (at 64 rows their matrix work) and the operands from L2;
      // per slice: what the norm pays to add it.  Beyond one round: workgroups of four waves, two on a CU, so that one's start and end run under
      // the other's chunks and the fixed part counts once (us, eight waves / four: w1|w3 22016 x 8192 at 64 rows, group size 64 86 / 78, 2 x 13824 x 5120 at 32 rows
      // 26.8 / 25.2, head 32000 x 4096 at 64 rows 31.3 / 29.3, 32000 x 8192 59 / 55; in one round eight are faster: 12288 x 4096 at 64 rows 14.7 / 16.6).
      const double work = chunks * (t * (mt == 4 ? 2.0 : 1.0) + 1.2 * mt);
      const double cost = (rounds > 1 ? 4 + rounds * work : 6 + work) + s * (0.5 + 0.6 * mt * halves * n / 4096);
      if (best_cost < 0 || cost < best_cost) {
        best_cost = cost;
        *g = Geometry{t, s, mt, halves, rounds > 1 ? 4 : 8};
      }
    }
  }
  if (best_cost < 0) return false;
  const int tc = gate ? g->t / 2 : g->t;
  a->col_blocks = (tiles16 + tc - 1) / tc;
  return true;
}

}  // namespace
}  // namespace e2h

using namespace e2h;

extern "C" int64_t e2h_int4_staged_bytes(int64_t m, int64_t k) {
  if (m < 1 || m > 64 || k < 128 || (k % 128) != 0) return E2H_ERR_BAD_SHAPE;
  return staged_bytes(m, k);
}

extern "C" int e2h_int4_stage_x(const uint16_t *x, void *staged, int64_t m, int64_t k, void *stream) {
  if (!x || !staged) return E2H_ERR_NULL_POINTER;
  if (m < 1 || m > 64 || k < 128 || (k % 128) != 0 || k > (1 << 24)) return E2H_ERR_BAD_SHAPE;
  if (!aligned16(x) || !aligned16(staged)) return E2H_ERR_MISALIGNED;
  const StagedOut out = staged_out(staged, m, k);
  const int64_t threads = static_cast<int64_t>(out.mpad) * (k / 8);
  hipLaunchKernelGGL(int4_stage_x_kernel, dim3(static_cast<unsigned>((threads + 255) / 256)), dim3(256), 0, static_cast<hipStream_t>(stream), x,
                     out, static_cast<int>(m), static_cast<int>(k));
  return launch_status();
}

extern "C" int e2h_int4_mm_staged_supported(int64_t m, int64_t n, int64_t k, int groupsize, int epilogue) {
  if (check_shape(m, n, k, groupsize) != E2H_OK || epilogue < 0 || epilogue > 4) return 0;
  StagedArgs a = {};
  Geometry g;
  return plan(&a, &g, nullptr, m, n, k, groupsize, epilogue) ? 1 : 0;
}

extern "C" int e2h_int4_mm_staged(const void *staged, const int32_t *packed, const uint16_t *scales_and_zeros, uint16_t *y, int64_t m,
                                  int64_t n, int64_t k, int groupsize, void *stream) {
  if (!staged || !packed || !scales_and_zeros || !y) return E2H_ERR_NULL_POINTER;
  const int rc = check_shape(m, n, k, groupsize);
  if (rc != E2H_OK) return rc;
  if (!aligned16(staged) || !aligned16(packed) || !aligned16(scales_and_zeros) || (reinterpret_cast<uintptr_t>(y) & 1u)) return E2H_ERR_MISALIGNED;
  StagedArgs a = {};
  Geometry g;
  if (!plan(&a, &g, staged, m, n, k, groupsize, kStPlain)) return E2H_ERR_BAD_SHAPE;
  a.wp = reinterpret_cast<const uint32_t *>(packed);
  a.sz = reinterpret_cast<const uint32_t *>(scales_and_zeros);
  a.y = y;
  return dispatch_staged<kStPlain>(a, groupsize, g, static_cast<hipStream_t>(stream));
}

extern "C" int64_t e2h_int4_mm_staged_argmax_scratch_bytes(int64_t m, int64_t n, int64_t k, int groupsize) {
  const int rc = check_shape(m, n, k, groupsize);
  if (rc != E2H_OK) return rc;
  StagedArgs a = {};
  Geometry g;
  if (!plan(&a, &g, nullptr, m, n, k, groupsize, kStArgmax)) return E2H_ERR_BAD_SHAPE;
  return static_cast<int64_t>(a.col_blocks) * m * 8;
}

extern "C" int e2h_int4_mm_staged_argmax(const void *staged, const int32_t *packed, const uint16_t *scales_and_zeros, void *scratch,
                                         int64_t *tokens, int64_t m, int64_t n, int64_t k, int groupsize, void *stream) {
  if (!staged || !packed || !scales_and_zeros || !scratch || !tokens) return E2H_ERR_NULL_POINTER;
  const int rc = check_shape(m, n, k, groupsize);
  if (rc != E2H_OK) return rc;
  if (!aligned16(staged) || !aligned16(packed) || !aligned16(scales_and_zeros) || (reinterpret_cast<uintptr_t>(scratch) & 7u) ||
      (reinterpret_cast<uintptr_t>(tokens) & 7u))
    return E2H_ERR_MISALIGNED;
  StagedArgs a = {};
  Geometry g;
  if (!plan(&a, &g, staged, m, n, k, groupsize, kStArgmax)) return E2H_ERR_BAD_SHAPE;
  a.wp = reinterpret_cast<const uint32_t *>(packed);
  a.sz = reinterpret_cast<const uint32_t *>(scales_and_zeros);
  a.cand = static_cast<unsigned long long *>(scratch);
  const int rc2 = dispatch_staged<kStArgmax>(a, groupsize, g, static_cast<hipStream_t>(stream));
  if (rc2 != E2H_OK) return rc2;
  hipLaunchKernelGGL(argmax_candidates_kernel, dim3(static_cast<unsigned>(m)), dim3(64), 0, static_cast<hipStream_t>(stream), a.cand,
                     a.col_blocks, a.M, tokens);
  return launch_status();
}

extern "C" int e2h_int4_mm_staged_partial_slices(int64_t m, int64_t n, int64_t k, int groupsize) {
  const int rc = check_shape(m, n, k, groupsize);
  if (rc != E2H_OK) return rc;
  StagedArgs a = {};
  Geometry g;
  if (!plan(&a, &g, nullptr, m, n, k, groupsize, kStPartial)) return E2H_ERR_BAD_SHAPE;
  return g.slices;
}

extern "C" int e2h_int4_mm_staged_partials(const void *staged, const int32_t *packed, const uint16_t *scales_and_zeros, float *partials,
                                           int64_t m, int64_t n, int64_t k, int groupsize, int slices, void *stream) {
  if (!staged || !packed || !scales_and_zeros || !partials) return E2H_ERR_NULL_POINTER;
  const int rc = check_shape(m, n, k, groupsize);
  if (rc != E2H_OK) return rc;
  if (!aligned16(staged) || !aligned16(packed) || !aligned16(scales_and_zeros) || (reinterpret_cast<uintptr_t>(partials) & 3u)) return E2H_ERR_MISALIGNED;
  StagedArgs a = {};
  Geometry g;
  if (!plan(&a, &g, staged, m, n, k, groupsize, kStPartial)) return E2H_ERR_BAD_SHAPE;
  if (slices != g.slices) return E2H_ERR_BAD_SHAPE;
  a.wp = reinterpret_cast<const uint32_t *>(packed);
  a.sz = reinterpret_cast<const uint32_t *>(scales_and_zeros);
  a.partials = partials;
  return dispatch_staged<kStPartial>(a, groupsize, g, static_cast<hipStream_t>(stream));
}

extern "C" int e2h_int4_mm_staged_silu_gate(const void *staged, const int32_t *packed_gate, const uint16_t *sz_gate, const int32_t *packed_up,
                                            const uint16_t *sz_up, uint16_t *y, void *staged_out_buf, int64_t m, int64_t n, int64_t k,
                                            int groupsize, void *stream) {
  if (!staged || !packed_gate || !sz_gate || !packed_up || !sz_up || (!y && !staged_out_buf)) return E2H_ERR_NULL_POINTER;
  const int rc = check_shape(m, n, k, groupsize);
  if (rc != E2H_OK) return rc;
  if (staged_out_buf && (n % 128) != 0) return E2H_ERR_BAD_SHAPE;  // the result is the next linear's K
  if (!aligned16(staged) || !aligned16(packed_gate) || !aligned16(sz_gate) || !aligned16(packed_up) || !aligned16(sz_up) ||
      (reinterpret_cast<uintptr_t>(y) & 1u) || !aligned16(staged_out_buf))
    return E2H_ERR_MISALIGNED;
  StagedArgs a = {};
  Geometry g;
  if (!plan(&a, &g, staged, m, n, k, groupsize, kStGate)) return E2H_ERR_BAD_SHAPE;
  a.wp = reinterpret_cast<const uint32_t *>(packed_gate);
  a.sz = reinterpret_cast<const uint32_t *>(sz_gate);
  a.wp2 = reinterpret_cast<const uint32_t *>(packed_up);
  a.sz2 = reinterpret_cast<const uint32_t *>(sz_up);
  a.y = y;
  a.out = staged_out(staged_out_buf, m, n);
  return dispatch_staged<kStGate>(a, groupsize, g, static_cast<hipStream_t>(stream));
}

extern "C" int e2h_int4_mm_staged_rope_kv(const void *staged, const int32_t *packed, const uint16_t *scales_and_zeros, const uint16_t *freqs_cis,
                                          uint16_t *q_out, uint16_t *k_cache, uint16_t *v_cache, const int64_t *input_pos, int64_t batch,
                                          int64_t n_head, int64_t n_kv_head, int64_t head_dim, int64_t cache_len, int64_t k, int groupsize,
                                          void *stream) {
  if (!staged || !packed || !scales_and_zeros || !freqs_cis || !q_out || !k_cache || !v_cache || !input_pos) return E2H_ERR_NULL_POINTER;
  if (n_head < 1 || n_kv_head < 1 || head_dim < 2 || (head_dim % 2) != 0 || cache_len < 1 || cache_len > INT32_MAX) return E2H_ERR_BAD_SHAPE;
  const int64_t n = (n_head + 2 * n_kv_head) * head_dim;
  const int rc = check_shape(batch, n, k, groupsize);
  if (rc != E2H_OK) return rc;
  if (!aligned16(staged) || !aligned16(packed) || !aligned16(scales_and_zeros) || (reinterpret_cast<uintptr_t>(freqs_cis) & 3u) ||
      (reinterpret_cast<uintptr_t>(q_out) & 1u) || (reinterpret_cast<uintptr_t>(k_cache) & 1u) || (reinterpret_cast<uintptr_t>(v_cache) & 1u) ||
      (reinterpret_cast<uintptr_t>(input_pos) & 7u))
    return E2H_ERR_MISALIGNED;
  StagedArgs a = {};
  Geometry g;
  if (!plan(&a, &g, staged, batch, n, k, groupsize, kStRope)) return E2H_ERR_BAD_SHAPE;
  a.wp = reinterpret_cast<const uint32_t *>(packed);
  a.sz = reinterpret_cast<const uint32_t *>(scales_and_zeros);
  a.rope = StagedRope{freqs_cis, q_out, k_cache, v_cache, input_pos, static_cast<int>(n_head), static_cast<int>(n_kv_head),
                      static_cast<int>(cache_len), static_cast<int>(head_dim)};
  return dispatch_staged<kStRope>(a, groupsize, g, static_cast<hipStream_t>(stream));
}
