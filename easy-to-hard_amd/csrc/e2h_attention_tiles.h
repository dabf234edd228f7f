// Softmax attention of 128 queries of one head over a list of keys: the loop that the prompt kernels share.
//
// Four waves of 32 queries, key tiles of 64.  Both products on v_mfma_f32_16x16x32_bf16 in transposed form: S^T = K Q^T puts one query into each
// lane column (lane 16 b + c holds keys 4 b .. 4 b + 3 of query c), so statistics are in-lane sums plus two shuffles, and the weights are the second operand of
// O^T = V^T P^T without moving, over the key order 4 b .. 4 b + 3, 16 + 4 b .. 16 + 4 b + 3 of each 32.
// What bounds it: the vector work between the products (scores, maxima, exponents, rounding) takes one and a half times as long as they do (8192 tokens, window 2048: matrix pipelines
// busy 36 %, vector units 56 %; 64 x 768 tokens 24 and 44 %), and waves wait for a third of their time and more.  (Measured with masks taken key by key and the next
// tile's loads waited for before V is read; without either 526 us have become 493 and 667 have become 646, 8 x 1024 tokens 185 and 174.)  Two workgroups share a CU (64 KB of LDS each), so that one computes
// under the other's products and waits.  32 queries per wave rather than 16, so that a fragment of K or V read from LDS feeds two or four products (with 16 the
// LDS took longer than the products); K and V reach LDS by loads that write it directly, two stages, one barrier per tile, and V's
// fragments leave it through the transposing read (written transposed by two-byte stores, V cost as much LDS time as both products' reads).
#pragma once

#include "e2h_common.h"

namespace e2h {
namespace attention {

constexpr int kQueries = 128, kKeys = 64;
constexpr float kMaskedScore = -__builtin_inff(), kLog2E = 1.4426950408889634f;
template <int D>
constexpr int kLdsBytes = 2 * 2 * kKeys * D * 2;

struct Keys {  // virtual index n -> key position: the kept first ones, then the window
  int first, kept, start, count;
  __device__ int at(int n) const { return n < kept ? first + n : start + (n - kept); }
};

struct Rule {  // which keys a query sees
  int first, window, keep;
  __device__ bool sees(int i, int j) const { return j <= i && j >= first && (i - j < window || j - first < keep); }
};

#if defined(__HIP_DEVICE_COMPILE__)
typedef __attribute__((address_space(3))) void lds_void_t;
typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4_t lds_s16x4_t;

__device__ __forceinline__ uint32_t pack_bf16_pair(float lo, float hi) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, bf16x2));
}

// The transposing read.  __restrict__ is what tells the compiler that loads into LDS under way do not write here: without it, it waits for
// all of them before the first such read of a tile, which are the next tile's.
__device__ __forceinline__ s16x4_t read_turned(const uint8_t *__restrict__ at) { return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t *)at); }

// Workgroup -> (sequence, key head), query head of its group, block of queries counted from the last one.  Workgroups are dealt out to the eight XCDs in turn.
// Where the (sequence, key head) pairs, or else the heads, divide by eight, each XCD walks its own ones, all blocks of one after each other and those with the most
// keys first, so that its L2 holds their keys and every XCD has the same work; otherwise the blocks with the most keys go first.
struct Place {
  int pair, rep, back;
};
__device__ __forceinline__ Place place(int id, int pairs, int reps, int blocks) {
  if (pairs % 8 == 0) {
    const int slot = id >> 3;
    return {(id & 7) + 8 * (slot / (reps * blocks)), slot % reps, slot / reps % blocks};
  }
  const int heads = pairs * reps;
  const int head = heads % 8 == 0 ? (id & 7) + 8 * ((id >> 3) / blocks) : id % heads;
  return {head / reps, head % reps, heads % 8 == 0 ? (id >> 3) % blocks : id / heads};
}

// eight weights as value + remainder (SPLIT: float32 accuracy against bfloat16 values) or rounded
template <bool SPLIT>
__device__ __forceinline__ void weights(const float (&p)[8], bf16x8_t &hi, bf16x8_t &lo) {
  u32x4_t h, l = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (SPLIT) {
      const uint32_t a = __builtin_bit_cast(uint32_t, p[2 * i]) & 0xFFFF0000u, b = __builtin_bit_cast(uint32_t, p[2 * i + 1]) & 0xFFFF0000u;
      h[i] = (a >> 16) | b;
      l[i] = pack_bf16_pair(p[2 * i] - __builtin_bit_cast(float, a), p[2 * i + 1] - __builtin_bit_cast(float, b));
    } else {
      h[i] = pack_bf16_pair(p[2 * i], p[2 * i + 1]);
    }
  }
  hi = __builtin_bit_cast(bf16x8_t, h);
  lo = __builtin_bit_cast(bf16x8_t, l);
}

// The same result for one wave without LDS, fragments straight from memory, scores taken relative to the largest one before anything is multiplied: for scores of any
// size.  Two walks over the keys, the first for the largest scores.
template <int D>
__device__ __forceinline__ void attend_far(const bf16x8_t (&qf)[2][D / 32], const int (&pos)[2], const Keys &kl, const Rule &rule, float sc, const uint16_t *kc, const uint16_t *vc,
                                           f32x4_t (&o)[2][D / 16], float (&m)[2], float (&l)[2]) {
  constexpr int KS = D / 32, VT = D / 16;
  const int lane = threadIdx.x & 63, c = lane & 15, b4 = lane >> 4;
  const auto key = [&](int n) { return kl.at(n < kl.count ? n : kl.count - 1); };
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    m[i] = kMaskedScore;
    l[i] = 0.f;
#pragma unroll
    for (int v = 0; v < VT; ++v) o[i][v] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int walk = 0; walk < 2; ++walk) {
      const float top = m[i] > kMaskedScore ? m[i] : 0.f;
#pragma unroll 1
      for (int n0 = 0; n0 < kl.count; n0 += 32) {
        float p[8];  // keys n0 + 16 (e / 4) + 4 b + e % 4
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
          f32x4_t st = {0.f, 0.f, 0.f, 0.f};
          const uint16_t *row = kc + static_cast<size_t>(key(n0 + 16 * kt + c)) * D + 8 * b4;
#pragma unroll
          for (int s = 0; s < KS; ++s) st = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8_t *>(row + 32 * s), qf[i][s], st, 0, 0, 0);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int n = n0 + 16 * kt + 4 * b4 + e;
            p[4 * kt + e] = n < kl.count && rule.sees(pos[i], kl.at(n)) ? st[e] : kMaskedScore;
          }
        }
        if (walk == 0) {
#pragma unroll
          for (int e = 0; e < 8; ++e) m[i] = fmaxf(m[i], p[e]);
          continue;
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          p[e] = __builtin_amdgcn_exp2f((p[e] - top) * sc);
          l[i] += p[e];
        }
        bf16x8_t wh, wl;
        weights<false>(p, wh, wl);
#pragma unroll
        for (int v = 0; v < VT; ++v) {
          u32x4_t a;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int n = n0 + 16 * (e >> 1) + 4 * b4 + 2 * (e & 1);
            a[e] = vc[static_cast<size_t>(key(n)) * D + 16 * v + c] | static_cast<uint32_t>(vc[static_cast<size_t>(key(n + 1)) * D + 16 * v + c]) << 16;
          }
          o[i][v] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), wh, o[i][v], 0, 0, 0);
        }
      }
      m[i] = fmaxf(m[i], __shfl_xor(m[i], 16));
      m[i] = fmaxf(m[i], __shfl_xor(m[i], 32));
    }
  }
}

// qf[i][s]: dimensions 32 s + 8 b .. + 7 of query 16 i + c of the wave (lane 16 b + c), at position pos[i]; lo, hi: the wave's smallest and largest position.
// kc, vc: [rows, D], 16-byte aligned.  Results, lane (b, c): o[i][v] = weighted sums of value columns 16 v + 4 b .. + 3 of query 16 i + c in units of 2^(its
// largest score times sc), m[i] that score (no key seen: minus infinity, and units of 1), l[i] this lane's share of the sum of weights.
// ANY: scores may have any size (with SPLIT there are no registers left for it).
template <int D, bool SPLIT, bool ANY>
__device__ __forceinline__ void attend(const bf16x8_t (&qf)[2][D / 32], const int (&pos)[2], int lo, int hi, const Keys &kl, const Rule &rule, float sc, const uint16_t *kc,
                                       const uint16_t *vc, uint32_t rows, uint8_t *lds, f32x4_t (&o)[2][D / 16], float (&m)[2], float (&l)[2]) {
  constexpr int KS = D / 32, VT = D / 16, kRow = D * 2, kOperand = kKeys * kRow, kStage = 2 * kOperand;
  constexpr int kPieces = D / 8, kBlockRows = 64 / kPieces, kBlocks = kKeys / kBlockRows / 4;  // 1 KB blocks of a wave and operand
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = lane & 15, b4 = lane >> 4;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    m[i] = kMaskedScore;
    l[i] = 0.f;
#pragma unroll
    for (int v = 0; v < VT; ++v) o[i][v] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  if (kl.count <= 0) return;  // the whole workgroup
  const __amdgpu_buffer_rsrc_t kr = make_rsrc(kc, rows * kRow), vr = make_rsrc(vc, rows * kRow);

  // Loads: lane l brings the piece that belongs at position l % kPieces of row l / kPieces of a block.  A row's 16-byte pieces of K stand at piece ^ row (16 rows read
  // one piece from 16 different bank groups), the 32-byte segments of V at segment ^ row (the transposing read takes one segment of 16 rows).
  const int brow = lane / kPieces, at = lane % kPieces;
  auto load = [&](int n0, uint32_t stage) {
#pragma unroll
    for (int i = 0; i < kBlocks; ++i) {
      const int row = (wave + 4 * i) * kBlockRows + brow, n = n0 + row, j = kl.at(n < kl.count ? n : kl.count - 1);
      const int kf = D == 128 ? row & 15 : (row >> 1) & 7, vf = D == 128 ? row & 7 : (row >> 1) & 3;
      const uint32_t base = static_cast<uint32_t>(j) * kRow;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(kr, (lds_void_t *)(lds + stage + (wave + 4 * i) * 1024), 16, base + ((at ^ kf) << 4), 0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(vr, (lds_void_t *)(lds + stage + kOperand + (wave + 4 * i) * 1024), 16, base + ((((at >> 1) ^ vf) << 5) | ((at & 1) << 4)), 0, 0, 0);
    }
  };
  uint32_t k_at[KS], v_at[VT];  // K: row c of a tile of 16, piece 4 s + b; V: rows 4 b + c / 4, bytes 8 (c % 4) of segment v
  const int vrow = 4 * b4 + (c >> 2), kf = D == 128 ? c : (c >> 1) & 7, vf = D == 128 ? vrow & 7 : (vrow >> 1) & 3;
#pragma unroll
  for (int s = 0; s < KS; ++s) k_at[s] = static_cast<uint32_t>(c * kRow + (((4 * s + b4) ^ kf) << 4));
#pragma unroll
  for (int v = 0; v < VT; ++v) v_at[v] = static_cast<uint32_t>(kOperand + vrow * kRow + ((v ^ vf) << 5) + 8 * (c & 3));

  load(0, 0);
  uint32_t stage = 0;
  for (int n0 = 0; n0 < kl.count; n0 += kKeys, stage ^= kStage) {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");  // this tile is in, and everybody is done with the other stage
    if (n0 + kKeys < kl.count) load(n0 + kKeys, stage ^ kStage);
    const int last = n0 + kKeys < kl.count ? n0 + kKeys - 1 : kl.count - 1, j0 = kl.at(n0), j1 = kl.at(last);
    // none of the wave's queries sees a key of the tile; uniform
    if (j0 > hi || (n0 >= kl.kept && j1 <= lo - rule.window)) continue;
    f32x4_t st[2][4];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
      st[0][kt] = st[1][kt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const bf16x8_t kfrag = *reinterpret_cast<const bf16x8_t *>(lds + stage + k_at[s] + kt * 16 * kRow);
#pragma unroll
        for (int i = 0; i < 2; ++i) st[i][kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kfrag, qf[i][s], st[i][kt], 0, 0, 0);
      }
    }
    // a tile inside every query's window needs no masks: whole, behind the kept keys, not beyond the first query, not out of the last one's window
    if (n0 >= kl.kept && n0 + kKeys <= kl.count && j1 <= lo && hi - j0 < rule.window && j0 >= rule.first) {
    } else if (n0 >= kl.kept && j0 - rule.first >= rule.keep) {
      // one run of keys, none of them kept: key t of the lane's (t = 16 kt + e) is `from` - t back from the query, and seen if that is in one range.
      // 100 instructions for a tile instead of 1000, of 700 in all: prompts shorter than the window have a tile or two of these in five.
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int from = pos[i] - (j0 + 4 * b4), end = pos[i] - rule.first + 1 < rule.window ? pos[i] - rule.first + 1 : rule.window;
        const int behind = from - (kl.count - n0 - 4 * b4) + 1, begin = behind > 0 ? behind : 0;
        const uint32_t span = end > begin ? static_cast<uint32_t>(end - begin) : 0u;
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
          for (int e = 0; e < 4; ++e) st[i][kt][e] = static_cast<uint32_t>(from - begin - (16 * kt + e)) < span ? st[i][kt][e] : kMaskedScore;
      }
    } else {
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int n = n0 + 16 * kt + 4 * b4 + e, j = n < kl.count ? kl.at(n) : INT32_MAX;
#pragma unroll
          for (int i = 0; i < 2; ++i)
            if (!rule.sees(pos[i], j)) st[i][kt][e] = kMaskedScore;
        }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      float mx = st[i][0][0];
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int e = 0; e < 4; ++e) mx = fmaxf(mx, st[i][kt][e]);
      mx = fmaxf(mx, __shfl_xor(mx, 16));
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      const float m_new = fmaxf(m[i], mx);
      // while a query has seen no key its maximum is the mask value, which no finite score reaches: exponents are then taken against 0, where masked scores give 0
      const float ref = m_new > kMaskedScore ? m_new * sc : 0.f;
      // sums enter and leave the branch as whole registers: element by element they would be copied once per tile
#pragma unroll
      for (int v = 0; v < VT; ++v) asm volatile("" : "+v"(o[i][v]));
      if (__builtin_amdgcn_ballot_w64(m_new > m[i])) {  // a larger score somewhere: uniform
        const float corr = __builtin_amdgcn_exp2f(__builtin_fmaf(m[i], sc, -ref));
        l[i] *= corr;
#pragma unroll
        for (int v = 0; v < VT; ++v)
#pragma unroll
          for (int e = 0; e < 4; ++e) o[i][v][e] *= corr;
        m[i] = m_new;
      }
#pragma unroll
      for (int v = 0; v < VT; ++v) asm volatile("" : "+v"(o[i][v]));
      float sum = 0.f;
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          st[i][kt][e] = __builtin_amdgcn_exp2f(__builtin_fmaf(st[i][kt][e], sc, -ref));
          sum += st[i][kt][e];
        }
      l[i] += sum;
    }
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      bf16x8_t wh[2], wl[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        float p[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) p[e] = st[i][2 * half + (e >> 2)][e & 3];
        weights<SPLIT>(p, wh[i], wl[i]);
      }
#pragma unroll
      for (int v = 0; v < VT; ++v) {
        const s16x4_t v0 = read_turned(lds + stage + v_at[v] + half * 32 * kRow), v1 = read_turned(lds + stage + v_at[v] + (half * 32 + 16) * kRow);
        const u32x2_t a = __builtin_bit_cast(u32x2_t, v0), b = __builtin_bit_cast(u32x2_t, v1);
        const bf16x8_t vfrag = __builtin_bit_cast(bf16x8_t, u32x4_t{a[0], a[1], b[0], b[1]});
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          o[i][v] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vfrag, wh[i], o[i][v], 0, 0, 0);
          if (SPLIT) o[i][v] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vfrag, wl[i], o[i][v], 0, 0, 0);
        }
      }
    }
  }
  if constexpr (!ANY) return;
  // An exponent above is one multiply-add against a rounded reference, 2^-24 of the largest score's own exponent off.  Where that is beyond 4096, or sums have left float32's range
  // on the way (the largest score may have been farther from zero before), the wave starts over without it.
  bool far = false;
#pragma unroll
  for (int i = 0; i < 2; ++i) far |= (m[i] > kMaskedScore && __builtin_fabsf(m[i] * sc) > 4096.f) || !__builtin_isfinite(l[i]);
  if (__builtin_expect(__builtin_amdgcn_ballot_w64(far) != 0, 0)) attend_far<D>(qf, pos, kl, rule, sc, kc, vc, o, m, l);
}
#endif

}  // namespace attention
}  // namespace e2h
