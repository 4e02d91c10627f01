// Pooled block probabilities of a query-aware head, and what they share with the last-query scores (sp_scores.hip): the
// layout of a K tile in LDS and the 32x32 accumulators' rows.
#pragma once
#include "sp_common.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

#define LQ_ROWS 128          // query rows (= block size)
#define LQ_TILE 128          // keys per tile
// Row maxima are kept in base-2 units (max logit * log2 e), so a probability is one fused multiply-add and one
// hardware exp2.  "No logit seen yet" is a large finite negative number, not -inf: then max, difference and exp2
// need no special case (exp2(-inf - finite) = 0 for masked logits, exp2(0) * 0 for an empty history).
#define LQ_LOG2E 1.4426950408889634f
#define LQ_NO_MAX (-1.0e30f)

__device__ static __forceinline__ int lq_row_of(int wave, int lane, int r) {
  return wave * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
}

typedef float lq_floatx2 __attribute__((ext_vector_type(2)));
typedef __bf16 lq_bf16x2 __attribute__((ext_vector_type(2)));

// 32 KiB (D = 128) or 16 KiB: 256-byte lines of 16 chunks of 16 bytes, position p of line l holding chunk p ^ ((l >> SWZ) & 15)
// of the line.  A line is a key's 128 channels, or the 64 channels of keys 2 l and 2 l + 1.
#define LQ_KSW_BYTES(D) (LQ_TILE * (D) * 2)

typedef __attribute__((address_space(3))) void* lq_lds_ptr;
typedef const __attribute__((address_space(1))) void* lq_gbl_ptr;

// byte offset in LDS of 16-byte chunk c of key r, for a lane whose line swizzle ((line >> SWZ) & 15) is known
template <int D>
__device__ static __forceinline__ int lq_line(int r) { return D == 128 ? r : r >> 1; }
template <int D>
__device__ static __forceinline__ int lq_chunk(int r, int c) { return D == 128 ? c : (r & 1) * 8 + c; }

// ---- pooled block probabilities of query-aware heads (attention_sharing.py:350-360) -------------------------------
// probs[h][r][c] = softmax over c <= r of  bf16(qbar[r][h] / sqrt d) . kbar[c][kv head of h],  zero for c > r.
// The same two passes as the last-query scores, over 128-row tiles of the pooled queries against 128-row tiles of
// the pooled keys: pass 1 the row maxima and sums (transposed product, a lane owns one query), pass 2 the logits
// again (a lane owns key columns: coalesced rows of the output), normalised in the exponent.  One workgroup per (row
// tile, head); the K tile goes straight from global memory into LDS, XOR-swizzled; heads that are not query-aware
// leave at once.
#define BPM_THREADS 256

// 32 segments of 1 KiB (4 lines of pooled keys each; 16 segments for D = 64): instruction `it` of wave w (0..3) fills
// segment 4 it + w
template <int D, int PARTS>
__device__ static __forceinline__ void bpm_issue_k(const sp_bf16* kb_head, int64_t row_stride, int nb, int c_tile, char* ks,
                                                   int part, int wave, int lane) {
  static_assert(D / 16 % PARTS == 0, "");
#pragma unroll
  for (int i = 0; i < D / 16 / PARTS; ++i) {
    const int it = i * PARTS + part;
    const int seg = it * 4 + wave;
    const int line = seg * 4 + (lane >> 4);
    const int cl = (lane & 15) ^ (line & 15);
    int key = c_tile * LQ_TILE + (D == 128 ? line : 2 * line + (cl >> 3));
    if (key > nb - 1) key = nb - 1;  // rows past the end are clamped onto the last pooled key (masked later)
    __builtin_amdgcn_global_load_lds((lq_gbl_ptr)(kb_head + (int64_t)key * row_stride + (D == 128 ? cl : cl & 7) * 8),
                                     (lq_lds_ptr)(ks + seg * 1024), 16, 0, 0);
  }
}

// elements r, r + 1 of an accumulator rounded to bf16 (hardware conversion, round to nearest even)
__device__ static __forceinline__ void bpm_round_pair(floatx16& v, int r) {
  lq_floatx2 f;
  f[0] = v[r];
  f[1] = v[r + 1];
  const uint32_t pk = __builtin_bit_cast(uint32_t, __builtin_convertvector(f, lq_bf16x2));
  v[r] = __uint_as_float(pk << 16);
  v[r + 1] = __uint_as_float(pk & 0xffff0000u);
}

template <int D>
struct BpmLds {
  __attribute__((aligned(1024))) char ks[LQ_KSW_BYTES(D)];
  float2 rstat[LQ_ROWS];
};

// 128-row tile rt of head h, by PARTS sets of BPM_THREADS threads: all of them stage the keys and take turns at the key
// columns of pass 2; pass 1, whose sums run in one order, is the first set's.  Every thread of the workgroup calls it.
template <int D, int PARTS>
__device__ static __forceinline__ void bpm_rows(BpmLds<D>& lds, const sp_bf16* qbar /* [nb][hq][D] */,
                                                const sp_bf16* kbar /* [nb][hkv][D] */, int rt, int h, int hq, int hkv, int nb,
                                                uint32_t flags, float inv_sqrt_d, float* probs /* [hq][nb][nb] */) {
  char* const Ks = lds.ks;
  float2* const rstat = lds.rstat;
  const int kvh = h / (hq / hkv);
  const int part = threadIdx.x / BPM_THREADS, wave = (threadIdx.x >> 6) & 3, lane = threadIdx.x & 63;
  const int lq = lane & 31, hi = lane >> 5;
  const sp_bf16* kb_head = kbar + (int64_t)kvh * D;
  const int64_t k_stride = (int64_t)hkv * D;
  // the lane's operand row: pooled query rt * 128 + 32 wave + lq (clamped), scaled and rounded as the reference's
  // avg_q / sqrt(d) in bf16
  bf16x8 qa[D / 16];
  {
    int row = rt * LQ_ROWS + wave * 32 + lq;
    if (row > nb - 1) row = nb - 1;
    const sp_bf16* src = qbar + ((int64_t)row * hq + h) * D + 8 * hi;
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) {
      uint4 raw = *reinterpret_cast<const uint4*>(src + 16 * ks);
      uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t lo = sp_f32_to_bf16(__uint_as_float(w[j] << 16) * inv_sqrt_d);
        const uint32_t hi16 = sp_f32_to_bf16(__uint_as_float(w[j] & 0xffff0000u) * inv_sqrt_d);
        w[j] = lo | (hi16 << 16);
      }
      raw = make_uint4(w[0], w[1], w[2], w[3]);
      qa[ks] = __builtin_bit_cast(bf16x8, raw);
    }
  }
  const int row_off = lq_line<D>(lq) * 256, swz = lq_line<D>(lq) & 15;

  // ---- pass 1: row maximum (base-2 units) and sum, transposed product: the lane's query is row 32 wave + lq ----
  {
    float m = LQ_NO_MAX, l = 0.f;
    const int my_row = rt * LQ_ROWS + wave * 32 + lq;
    for (int ct = 0; ct <= rt; ++ct) {
      __syncthreads();
      bpm_issue_k<D, PARTS>(kb_head, k_stride, nb, ct, Ks, part, wave, lane);
      __builtin_amdgcn_s_waitcnt(0x0F70);
      __syncthreads();
#pragma unroll 1
      for (int half = 0; half < 2; ++half) {
        // (half a tile beyond the last key would leave maximum and sum as they are)
        if ((PARTS > 1 && part != 0) || ct * LQ_TILE + 64 * half >= nb) break;
        floatx16 acc[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const char* src = Ks + (2 * half + j) * 32 * D * 2 + row_off;
          floatx16 c = {0};
#pragma unroll
          for (int ks = 0; ks < D / 16; ++ks) {
            const uint4 raw = *reinterpret_cast<const uint4*>(src + ((lq_chunk<D>(lq, 2 * ks + hi) ^ swz) << 4));
            c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, raw), qa[ks], c, 0, 0, 0);
          }
          acc[j] = c;
        }
        if (flags & SP_FLAG_LOGITS_BF16) {
#pragma unroll
          for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; r += 2) bpm_round_pair(acc[j], r);
        }
        if (ct == rt) {  // the diagonal tile: keys beyond the row's own block (and beyond the last block) are masked
#pragma unroll
          for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              const int key = ct * LQ_TILE + 64 * half + 32 * j + 8 * (r >> 2) + 4 * hi + (r & 3);
              if (key > my_row || key >= nb) acc[j][r] = -INFINITY;
            }
        }
        float tmax = acc[0][0];
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r) tmax = fmaxf(tmax, acc[j][r]);
        const float mn = fmaxf(m, tmax * LQ_LOG2E);
        float add[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r) add[r & 3] += __builtin_amdgcn_exp2f(__builtin_fmaf(acc[j][r], LQ_LOG2E, -mn));
        l = __builtin_fmaf(l, __builtin_amdgcn_exp2f(m - mn), (add[0] + add[1]) + (add[2] + add[3]));
        m = mn;
      }
    }
    const float m2 = __shfl_xor(m, 32, SP_WAVE), l2 = __shfl_xor(l, 32, SP_WAVE);
    const float mn = fmaxf(m, m2);
    const float a = (hi ? l2 : l) * __builtin_amdgcn_exp2f((hi ? m2 : m) - mn);
    const float b = (hi ? l : l2) * __builtin_amdgcn_exp2f((hi ? m : m2) - mn);
    // max + log2(sum): a probability is then exp2(logit * log2 e - that)
    if (hi == 0 && part == 0) rstat[wave * 32 + lq] = make_float2(mn + __builtin_amdgcn_logf(a + b), 0.f);
  }
  __syncthreads();
  float rm[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) rm[r] = rstat[lq_row_of(wave, lane, r)].x;

  // ---- pass 2: probabilities; acc[nt][r] = S[row 32 wave + 8 (r / 4) + 4 hi + r % 4][key 32 nt + lq] ----
  for (int ct = 0; ct <= rt; ++ct) {
    if (rt > 0) {  // (a single tile is still there)
      __syncthreads();
      bpm_issue_k<D, PARTS>(kb_head, k_stride, nb, ct, Ks, part, wave, lane);
      __builtin_amdgcn_s_waitcnt(0x0F70);
      __syncthreads();
    }
#pragma unroll 1
    for (int nt = part; nt < 4 && ct * LQ_TILE + 32 * nt < nb; nt += PARTS) {
      const char* src = Ks + nt * 32 * D * 2 + row_off;
      floatx16 c = {0};
#pragma unroll
      for (int ks = 0; ks < D / 16; ++ks) {
        const uint4 raw = *reinterpret_cast<const uint4*>(src + ((lq_chunk<D>(lq, 2 * ks + hi) ^ swz) << 4));
        c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qa[ks], __builtin_bit_cast(bf16x8, raw), c, 0, 0, 0);
      }
      if (flags & SP_FLAG_LOGITS_BF16) {
#pragma unroll
        for (int r = 0; r < 16; r += 2) bpm_round_pair(c, r);
      }
      const int key = ct * LQ_TILE + 32 * nt + lq;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = rt * LQ_ROWS + lq_row_of(wave, lane, r);
        float pv = __builtin_amdgcn_exp2f(__builtin_fmaf(c[r], LQ_LOG2E, -rm[r]));
        if (key > row) pv = 0.f;
        if (row < nb && key < nb) probs[((int64_t)h * nb + row) * nb + key] = pv;
      }
    }
  }
  // the rest of the rows: zero beyond the diagonal tile
  {
    const int c0 = (rt + 1) * LQ_TILE;
    for (int i = 0; i < LQ_ROWS; ++i) {
      const int row = rt * LQ_ROWS + i;
      if (row >= nb) break;
      float* out = probs + ((int64_t)h * nb + row) * nb;
      for (int c = c0 + (int)threadIdx.x; c < nb; c += BPM_THREADS * PARTS) out[c] = 0.f;
    }
  }
}
