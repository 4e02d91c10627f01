// Decode step: one query token per head against the whole KV cache (GQA, no mask), bf16 in / bf16 out, fp32
// softmax.  Replaces the flash_attn_func call of the reference's decode branch (shareprefill_attn.py:146-155).
//
// HBM-bound: K and V are read exactly once (2 * n * hkv * d * 2 bytes); everything else has to stay out of the
// way.  The cache of one kv head is split into chunks; one workgroup streams a chunk for all query heads of the
// group (so the group's `g` heads share every K / V byte), keeps an online softmax, and leaves an unnormalised
// partial (o, m, l); a second tiny kernel merges the partials in a fixed order.  A batch of sequences is one more grid
// axis.  Groups of up to 16 heads take the ring kernel further below; what follows is for the others.
//
// Both products run on the matrix core with the group's heads as a (mostly empty) 32-wide operand -- the MFMAs
// are free here, the point is to keep the vector ALU out of the inner loop:
//   S^T[keys x heads] = K . Q^T    A = K rows from LDS, B = the queries in registers (columns >= g are zero)
//   O[heads x d]     += P . V      A = P (bf16, from LDS), B = V read from its row-major LDS tile with the
//                                  transposing LDS load (ds_read_b64_tr_b16), which hands every lane four
//                                  consecutive keys of one channel.
#include "sp_common.h"

#include <mutex>
#include <type_traits>

#define DC_THREADS 256
#define DC_TILE 128   // keys per tile
#define DC_D 128
#define DC_GMAX 32    // query heads per kv head (the 32-wide operand of the MFMAs); kernels are built for <= 8, 16, 32
#define DC_PITCH 136  // bf16 elements per LDS row of 128 (272 bytes: conflict-free 128-bit reads)

typedef uint32_t dc_u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 dc_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 dc_bf16x4 __attribute__((ext_vector_type(4)));
typedef float dc_floatx16 __attribute__((ext_vector_type(16)));
typedef float dc_floatx2 __attribute__((ext_vector_type(2)));
typedef __bf16 dc_bf16x2 __attribute__((ext_vector_type(2)));
typedef float dc_floatx4 __attribute__((ext_vector_type(4), aligned(8)));  // (partials: 8-byte aligned workspace)

__device__ static __forceinline__ uint32_t dc_pack2(float a, float b) {
  dc_floatx2 f;
  f[0] = a;
  f[1] = b;
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, dc_bf16x2));
}

// A tile is 128 rows of D = 64 or 128 channels in chunks of 16 bytes: thread t fetches chunk t % (D / 8) of rows t / (D / 8),
// + 2048 / D, ...; rows past the end are clamped.  d < D (a smaller head): the chunks beyond the row's d channels are zeros put in on the way
// into LDS -- the tile there is the row zero-padded to D channels, which changes no product -- and the loads for them read the
// row's first chunk: a load that only some lanes make is waited for on the spot, and that was each of a tile's sixteen (64
// channels, us: 131072 keys 98.4 -> 52.6, 8 caches of 4001 24.9 -> 17.2; with half the tile's width besides).
// (FULL: d == D, nothing to pad)
template <int D, bool FULL>
__device__ static __forceinline__ void dc_fetch(const sp_bf16* __restrict__ x, int64_t n, int64_t stride_n, int64_t kb,
                                               int t, int d, dc_u32x4 (&r)[D / 16]) {
  constexpr int CHUNKS = D / 8;
  const int chunk = FULL || t % CHUNKS * 8 < d ? t % CHUNKS : 0;
#pragma unroll
  for (int i = 0; i < D / 16; ++i) {
    int64_t key = kb + i * (DC_THREADS / CHUNKS) + t / CHUNKS;
    if (key > n - 1) key = n - 1;
    r[i] = *reinterpret_cast<const dc_u32x4*>(x + key * stride_n + chunk * 8);
  }
}

template <int D, bool FULL>
__device__ static __forceinline__ void dc_store(sp_bf16* tile, int t, int d, const dc_u32x4 (&r)[D / 16]) {
  constexpr int CHUNKS = D / 8;
  const bool real = FULL || t % CHUNKS * 8 < d;
#pragma unroll
  for (int i = 0; i < D / 16; ++i)
    *reinterpret_cast<dc_u32x4*>(tile + (i * (DC_THREADS / CHUNKS) + t / CHUNKS) * (D + 8) + t % CHUNKS * 8) =
        real ? r[i] : (dc_u32x4){0, 0, 0, 0};
}

// The probabilities enter P.V as bf16, relative to the running max, so it matters where that max starts anew: it does so
// at every chunk of tiles_per_chunk tiles (those of one sequence alone, dc_launch) also where a workgroup of a batch walks
// several chunks, whose results meet in fp32 as they would in the merging kernel.  A running max over the whole share of a
// workgroup left 8 caches of 4001 tokens 2.20e-3 from the attention in 64 bits, one sequence at a time 2.16e-3, this the same.
//
// grid (splits, hkv, batch); partial layout: o [batch][hkv][splits][g][128] fp32, ml [batch][hkv][splits][g] float2 (m
// in log2 units, l).  A cache that is one chunk (splits == 1) needs no merging: the result goes straight to `out`.
// G8 = groups of 8 heads the instance handles (g <= 8 * G8): accumulator rows r < 4 * G8 can belong to real heads
struct DcStrides {
  int64_t q_b, q_h, k_b, k_n, k_h, v_b, v_n, v_h;
};
template <int D, int G8, bool FULL>
__global__ __launch_bounds__(DC_THREADS, 2) void sp_decode_partial_kernel(
    const sp_bf16* __restrict__ q, const sp_bf16* __restrict__ k, const sp_bf16* __restrict__ v, int64_t n, int g,
    int d, DcStrides st, float scale_log2, int64_t keys_per_split, int tiles_per_chunk, float* __restrict__ o_part,
    float2* __restrict__ ml_part, sp_bf16* __restrict__ out) {
  constexpr int PITCH = D + 8, KS = D / 16, CT = D / 32;  // K and V rows in LDS, channel steps of S, channel tiles of O
  __shared__ __attribute__((aligned(16))) sp_bf16 Ks[DC_TILE * PITCH];
  __shared__ __attribute__((aligned(16))) sp_bf16 Vs[DC_TILE * PITCH];
  constexpr int GM = 8 * G8;
  __shared__ __attribute__((aligned(16))) sp_bf16 Ps[GM * DC_PITCH];  // probabilities [head][key]
  __shared__ float wmax[4][GM], wsum[4][GM], alpha_s[GM];
  const int split = blockIdx.x, kvh = blockIdx.y, splits = gridDim.x;
  const int64_t bh = (int64_t)blockIdx.z * gridDim.y + kvh;  // (sequence, kv head)
  const int64_t sk_n = st.k_n, sv_n = st.v_n;
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int lh = lane & 31, hi = lane >> 5;  // operand column / row inside a 32-wide tile, lane half
  const bool head_ok = lh < g;               // this lane's S^T column is a real head
  const sp_bf16* kh = k + blockIdx.z * st.k_b + kvh * st.k_h;
  const sp_bf16* vh = v + blockIdx.z * st.v_b + kvh * st.v_h;

  // B operand of S^T = K . Q^T: column lh = head, k-step ks covers channels 16ks + 8hi .. +7
  dc_bf16x8 qb[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const bool real = head_ok && (FULL || 16 * ks + 8 * hi < d);
    const dc_u32x4 raw = *reinterpret_cast<const dc_u32x4*>(q + blockIdx.z * st.q_b + (int64_t)(kvh * g + (head_ok ? lh : 0)) * st.q_h +
                                                           (real ? 16 * ks + 8 * hi : 0));
    qb[ks] = __builtin_bit_cast(dc_bf16x8, real ? raw : (dc_u32x4){0, 0, 0, 0});
  }

  const int64_t key_begin = (int64_t)split * keys_per_split;
  int64_t key_end = key_begin + keys_per_split;
  if (key_end > n) key_end = n;

  dc_floatx16 o = {0};                   // rows = heads 8(r/4) + 4hi + r%4 (only r < 4 G8 can be real), col = channel 32*wave + lh
  float m_run = -INFINITY, l_run = 0.f;  // of head lh (every wave keeps the same copy)
  // ... of the chunk at hand; what the workgroup's chunks in front of it came to, on a running max of its own
  float o_sum[4 * G8] = {0.f}, m_sum = -INFINITY, l_sum = 0.f;
  bool folded = false;                                                                          // (uniform)
  int tiles_left = tiles_per_chunk - (int)(key_begin / DC_TILE % tiles_per_chunk);  // of the chunk
  dc_u32x4 kr[D / 16], vr[D / 16];
  if (key_begin < key_end) {
    dc_fetch<D, FULL>(kh, n, sk_n, key_begin, t, d, kr);
    dc_fetch<D, FULL>(vh, n, sv_n, key_begin, t, d, vr);
  }
  for (int64_t kb = key_begin; kb < key_end; kb += DC_TILE) {
    __syncthreads();  // the previous tile's operand reads are done
    dc_store<D, FULL>(Ks, t, d, kr);
    dc_store<D, FULL>(Vs, t, d, vr);
    __syncthreads();
    if (kb + DC_TILE < key_end) {  // next tile on its way while this one is used
      dc_fetch<D, FULL>(kh, n, sk_n, kb + DC_TILE, t, d, kr);
      dc_fetch<D, FULL>(vh, n, sv_n, kb + DC_TILE, t, d, vr);
    }
    // ---- S^T for this wave's 32 keys: acc[r] = logit(key 32*wave + 8(r/4) + 4hi + r%4, head lh) ----
    dc_floatx16 acc = {0};
    {
      const sp_bf16* arow = Ks + (32 * wave + lh) * PITCH + 8 * hi;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const dc_u32x4 raw = *reinterpret_cast<const dc_u32x4*>(arow + 16 * ks);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(dc_bf16x8, raw), qb[ks], acc, 0, 0, 0);
      }
    }
    const int valid = (int)((key_end - kb) < DC_TILE ? (key_end - kb) : DC_TILE);
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int key = 32 * wave + 8 * (r >> 2) + 4 * hi + (r & 3);
      acc[r] = key < valid ? acc[r] * scale_log2 : -INFINITY;
      mx = fmaxf(mx, acc[r]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 32, SP_WAVE));
    if (head_ok && hi == 0) wmax[wave][lh] = mx;
    __syncthreads();
    float m_new = m_run, alpha = 1.f;
    if (head_ok) {
      m_new = fmaxf(fmaxf(fmaxf(wmax[0][lh], wmax[1][lh]), fmaxf(wmax[2][lh], wmax[3][lh])), m_run);
      const float base = m_new == -INFINITY ? 0.f : m_new;  // (no key so far has a finite logit: every weight is exp2(-inf) = 0)
      alpha = __builtin_amdgcn_exp2f(m_run - base);         // 0 on the first tile
      float ls = 0.f;
      sp_bf16* prow = Ps + lh * DC_PITCH + 32 * wave + 4 * hi;
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        const float p0 = __builtin_amdgcn_exp2f(acc[4 * r4 + 0] - base), p1 = __builtin_amdgcn_exp2f(acc[4 * r4 + 1] - base);
        const float p2 = __builtin_amdgcn_exp2f(acc[4 * r4 + 2] - base), p3 = __builtin_amdgcn_exp2f(acc[4 * r4 + 3] - base);
        ls += (p0 + p1) + (p2 + p3);
        *reinterpret_cast<uint2*>(prow + 8 * r4) = make_uint2(dc_pack2(p0, p1), dc_pack2(p2, p3));
      }
      ls += __shfl_xor(ls, 32, SP_WAVE);
      if (hi == 0) {
        wsum[wave][lh] = ls;
        if (wave == 0) alpha_s[lh] = alpha;
      }
    }
    __syncthreads();
    if (head_ok) {
      l_run = l_run * alpha + ((wsum[0][lh] + wsum[1][lh]) + (wsum[2][lh] + wsum[3][lh]));
      m_run = m_new;
    }
    // ---- O += P . V for this wave's 32 channels; only accumulator rows of real heads need the rescale ----
    if (wave < CT) {
#pragma unroll
      for (int r = 0; r < 4 * G8; ++r) {
        const int h = 8 * (r >> 2) + 4 * hi + (r & 3);
        if (h < g) o[r] *= alpha_s[h];
      }
      const sp_bf16* prow = Ps + lh * DC_PITCH + 8 * hi;
      // transposing read: the 16 lanes of a block address 4 key rows x 16 channels (4 lanes x 8 bytes per row) and
      // each lane receives 4 consecutive keys of its channel
      const sp_bf16* vtr = Vs + (8 * hi + ((lane & 15) >> 2)) * PITCH + 32 * wave + 16 * ((lane >> 4) & 1) +
                           4 * (lane & 3);
#pragma unroll
      for (int kk = 0; kk < 8; ++kk) {
        dc_u32x4 praw = {0, 0, 0, 0};
        if (head_ok) praw = *reinterpret_cast<const dc_u32x4*>(prow + 16 * kk);
        const dc_bf16x4 b0 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
            (__attribute__((address_space(3))) dc_bf16x4*)(vtr + (16 * kk) * PITCH));
        const dc_bf16x4 b1 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
            (__attribute__((address_space(3))) dc_bf16x4*)(vtr + (16 * kk + 4) * PITCH));
        dc_bf16x8 bv;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          bv[j] = b0[j];
          bv[4 + j] = b1[j];
        }
        o = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(dc_bf16x8, praw), bv, o, 0, 0, 0);
      }
    }
    const bool last = kb + DC_TILE >= key_end;
    if (--tiles_left == 0 || last) {  // (uniform)
      tiles_left = tiles_per_chunk;
      if (folded || !last) {
        folded = true;
        const float m = fmaxf(m_sum, m_run), base = m == -INFINITY ? 0.f : m;
        const float before = __builtin_amdgcn_exp2f(m_sum - base), here = __builtin_amdgcn_exp2f(m_run - base);
        l_sum = l_sum * before + l_run * here;
        m_sum = m;
#pragma unroll
        for (int r = 0; r < 4 * G8; ++r) {  // (lane h holds head h's factors)
          const int h = 8 * (r >> 2) + 4 * hi + (r & 3);
          o_sum[r] = o_sum[r] * __shfl(before, h, SP_WAVE) + o[r] * __shfl(here, h, SP_WAVE);
        }
        o = (dc_floatx16){0};
        m_run = -INFINITY;
        l_run = 0.f;
      }
    }
  }
  if (folded) {
#pragma unroll
    for (int r = 0; r < 4 * G8; ++r) o[r] = o_sum[r];
    m_run = m_sum;
    l_run = l_sum;
  }

  if (splits == 1) {  // (uniform)
    __syncthreads();  // the last tile's reads of wsum are done
    if (wave == 0 && hi == 0 && head_ok) wsum[0][lh] = l_run;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 4 * G8; ++r) {
      const int h = 8 * (r >> 2) + 4 * hi + (r & 3), c = 32 * wave + lh;
      if (wave < CT && h < g && c < d) out[(bh * g + h) * d + c] = sp_f32_to_bf16(o[r] / wsum[0][h]);
    }
    return;
  }
  float* op = o_part + ((bh * splits + split) * g) * DC_D;
#pragma unroll
  for (int r = 0; r < 4 * G8; ++r) {
    const int h = 8 * (r >> 2) + 4 * hi + (r & 3);
    if (wave < CT && h < g) op[h * DC_D + 32 * wave + lh] = o[r];
  }
  if (wave == 0 && hi == 0 && head_ok) ml_part[(bh * splits + split) * g + lh] = make_float2(m_run, l_run);
}

// Merges the chunk partials of one query head: eight groups of 32 threads take every eighth chunk (a thread four
// channels, 16-byte loads), the groups meet in LDS in a fixed order.  What it costs is latency -- a launch and a chain of
// loads as deep as a group has chunks (64 chunks at 131072 keys and 8 kv heads: eight instead of sixty-four).
#define DC_MAX_SPLITS 512
#define DC_COMBINE_GROUPS 8
__global__ __launch_bounds__(32 * DC_COMBINE_GROUPS) void sp_decode_combine_kernel(
    const float* __restrict__ o_part, const float2* __restrict__ ml_part, int g, int splits, int d,
    sp_bf16* __restrict__ out) {
  constexpr int THREADS = 32 * DC_COMBINE_GROUPS;
  __shared__ float w_s[DC_MAX_SPLITS];  // weight of chunk s: exp2(m_s - m), 0 for an empty chunk
  __shared__ float red[THREADS / SP_WAVE];
  __shared__ __attribute__((aligned(16))) float o_s[DC_COMBINE_GROUPS][DC_D];
  const int64_t head = blockIdx.x, bh = head / g;  // (sequence, query head), (sequence, kv head)
  const int h = (int)(head % g), t = threadIdx.x, grp = t >> 5, c4 = (t & 31) * 4;
  const float2* ml = ml_part + bh * splits * g + h;
  // (a smaller head's instance leaves the channels behind its own unwritten, which are not read: those threads' sums are dropped below)
  const float* op = o_part + (bh * splits * g + h) * DC_D + (c4 < d ? c4 : 0);
  // every chunk's statistics once, kept in registers between the two passes (splits <= 2 THREADS)
  float2 mine[DC_MAX_SPLITS / THREADS];
  float m = -INFINITY;
#pragma unroll
  for (int j = 0; j < DC_MAX_SPLITS / THREADS; ++j) {
    mine[j] = t + j * THREADS < splits ? ml[(int64_t)(t + j * THREADS) * g] : make_float2(-INFINITY, 0.f);
    m = fmaxf(m, mine[j].x);
  }
  m = sp_wave_max(m);
  if ((t & 63) == 0) red[t >> 6] = m;
  __syncthreads();
  m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  __syncthreads();
  float l = 0.f;
#pragma unroll
  for (int j = 0; j < DC_MAX_SPLITS / THREADS; ++j) {
    const float w = mine[j].x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mine[j].x - m);
    if (t + j * THREADS < splits) w_s[t + j * THREADS] = w;
    l += mine[j].y * w;
  }
  l = sp_wave_sum(l);
  if ((t & 63) == 0) red[t >> 6] = l;
  __syncthreads();
  float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 8
  for (int s = grp; s < splits; s += DC_COMBINE_GROUPS) {
    const dc_floatx4 x = *reinterpret_cast<const dc_floatx4*>(op + (int64_t)s * g * DC_D);
    const float w = w_s[s];
    o.x += x[0] * w, o.y += x[1] * w, o.z += x[2] * w, o.w += x[3] * w;
  }
  *reinterpret_cast<float4*>(&o_s[grp][c4]) = o;
  __syncthreads();
  if (t < d) {
    float acc = 0.f;
#pragma unroll
    for (int j = 0; j < DC_COMBINE_GROUPS; ++j) acc += o_s[j][t];
    out[head * d + t] = sp_f32_to_bf16(acc / ((red[0] + red[1]) + (red[2] + red[3])));
  }
}

#define DC_MAX_GRID_Z 65535

// ---- up to 16 query heads per kv head --------------------------------------------------------------------------
// The waves of a workgroup take 32 keys each in turn, every wave with a running max and a ring of operands in LDS of its own that is
// filled by direct loads, no barrier between them, and meet in LDS at the end.
//   S^T[16 keys x 16 heads] = K . Q^T
//   O^T[16 channels x 16 heads] += V^T . P^T    V^T by the transposing LDS read; S^T leaves a lane with keys 4g .. 4g+3 of either
//                                               16-key tile, which is what two such reads deliver.
// P enters the product as two bf16 values, its rounding and what that leaves: outputs are 1.67e-3 from the attention in 64 bits, all of it
// their own rounding, where one bf16 value and a running max per chunk of the cache left 2.16e-3.
// Two ways to fill the chip (ds_plan):
//   * a workgroup takes ALL keys of a kv head and a slice of V's channels, so that nothing has to be merged across workgroups and there
//     is one launch.  Every slice forms the logits again, on CUs that would idle otherwise, from K's rows in the L2 that the slices share.
//     For caches of some hundred keys, where launches and latency are all there is, and for batches.
//   * all channels and a split of the keys, merged by the second kernel.
// Bound: HBM at 5.85 TB/s of a batch (16 caches of 8000 tokens 100 -> 89 us), the waves' chain of steps otherwise.  K's rows straight from
// memory into the operand registers (16 rows x 64 bytes an instruction) took 50 cycles an instruction, whole rows by way of LDS take
// 16 (1025 keys 11.3 -> 6.9 us); a ring one step deeper changes nothing.  us, GPU time in replayed graphs: 200 keys 8.0 -> 3.5, 1025
// 8.8 -> 6.9, 16 caches of 1025 22.7 -> 15.4, 131072 keys 97.9 -> 97.2; called one by one from Python, arguments in memory included, 200 keys
// 10.1 -> 9.0, 1025 14.0 -> 9.2, 2048 14.2 -> 12.7.
#define DS_GMAX 16
#define DS_KEYS 32  // keys of a wave's step
typedef float ds_floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t ds_u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void* ds_lds_ptr;

// CT_: channel tiles of 16 a slice has.  As many waves and steps of the ring as fit the LDS that the workgroup may have.
template <int D_, int CT_, int WAVES_, int KIB>
struct DsShape {
  static constexpr int D = D_, CT = CT_, WAVES = WAVES_;
  static constexpr int K_BYTES = DS_KEYS * D * 2, V_BYTES = DS_KEYS * CT * 32, STEP_BYTES = K_BYTES + V_BYTES;
  static constexpr int NB = KIB * 1024 / (WAVES * STEP_BYTES) < 4 ? KIB * 1024 / (WAVES * STEP_BYTES) : 4;
  static constexpr int LOADS = STEP_BYTES / 1024;  // of a step
  static constexpr int LDS_BYTES = WAVES * NB * STEP_BYTES;
  static_assert(NB >= 2 && LDS_BYTES >= WAVES * DS_GMAX * (16 * CT + 4) * 4, "");
};
// one to a CU
template <int D, int CT>
using DsWide = DsShape<D, CT, D == 64 || CT == 1 ? 8 : CT == 2 ? 7 : CT == 4 ? 6 : 4, 152>;
// two to a CU, and four, each taking all channels of a (sequence, kv head): for more of those than CUs (ds_plan)
template <int D>
using DsPair = DsShape<D, D / 16, D == 64 ? 4 : 2, 72>;
template <int D>
using DsQuad = DsShape<D, D / 16, D == 64 ? 2 : 1, 40>;
struct DsArgs {
  const sp_bf16 *q, *k, *v;
  int n_keys, g, hkv, d, batch;
  uint32_t hkv_mul;  // i / hkv = (i * hkv_mul) >> 16
  DcStrides st;
  float scale_log2;
  int keys_per_split;
  float* o_part;
  float2* ml_part;
  sp_bf16* out;
};

__device__ static __forceinline__ float ds_quad_max(float v) {  // over the lanes l, l ^ 16, l ^ 32, l ^ 48 that share a head
  uint32_t u = __builtin_bit_cast(uint32_t, v);
  const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  v = fmaxf(__builtin_bit_cast(float, (uint32_t)a[0]), __builtin_bit_cast(float, (uint32_t)a[1]));
  u = __builtin_bit_cast(uint32_t, v);
  const auto b = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return fmaxf(__builtin_bit_cast(float, (uint32_t)b[0]), __builtin_bit_cast(float, (uint32_t)b[1]));
}
__device__ static __forceinline__ float ds_quad_sum(float v) {
  uint32_t u = __builtin_bit_cast(uint32_t, v);
  const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  v = __builtin_bit_cast(float, (uint32_t)a[0]) + __builtin_bit_cast(float, (uint32_t)a[1]);
  u = __builtin_bit_cast(uint32_t, v);
  const auto b = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __builtin_bit_cast(float, (uint32_t)b[0]) + __builtin_bit_cast(float, (uint32_t)b[1]);
}

// LDS reads the compiler does not track: it would wait for every direct-to-LDS load in flight before each
__device__ static __forceinline__ dc_u32x4 ds_read_k(uint32_t addr) {
  dc_u32x4 r;
  asm volatile("ds_read_b128 %0, %1" : "=v"(r) : "v"(addr));
  return r;
}
template <int IMM>
__device__ static __forceinline__ ds_u32x2 ds_read_v(uint32_t addr) {
  ds_u32x2 r;
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "n"(IMM));
  return r;
}

// V for the product with the probabilities' second part: infinities become the largest value of their sign.  An infinite value has met its
// weight in the first product; the second part is zero or of either sign, and 0 * inf or inf - inf would make a NaN of the sum.  (Finite
// values are what they were, a NaN has made its sum NaN in the first product.)  Two instructions a register, issued under the first
// products: steps take 0.6 % longer in the median, 3 % at most (64 and fewer channels, 300 to 1025 keys); a second walk of the keys only
// where a sum came out NaN made the plain one slower (2 to 16 %).
__device__ static __forceinline__ dc_u32x4 ds_finite(dc_u32x4 v) {
  typedef short s16x8 __attribute__((ext_vector_type(8)));
  typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));
  const s16x8 pos = __builtin_elementwise_min(__builtin_bit_cast(s16x8, v), (s16x8)(short)0x7f7f);
  return __builtin_bit_cast(dc_u32x4, __builtin_elementwise_min(__builtin_bit_cast(u16x8, pos), (u16x8)(unsigned short)0xff7f));
}

// Steps in LDS: K [32 keys][D], V [32 keys][16 CT channels] in 16-byte chunks, swizzled by the row: K's chunks for reads of one chunk
// of 16 rows, V's pairs of chunks for the transposing reads of a pair of 8 rows (256 bytes, all banks, either way).
template <int D>
__device__ static __forceinline__ int ds_swz_k(int row) {
  return D == 128 ? row & 15 : (row >> 1) & 7;
}
template <int CT>
__device__ static __forceinline__ int ds_swz_v(int row) {
  return CT == 1 ? 0 : (row / (8 / CT)) & (CT - 1);
}

// grid (hkv, splits, batch) of splits of the keys where a slice is all channels; otherwise (8, slices, (sequence, kv head) / 8), which
// places the slices of a kv head on one XCD: they read the same keys (4 caches of 2048 keys, 4 kv heads: 13.0 us across two XCDs)
// FULL: d == D; a smaller head's rows read as zero-padded: its loads behind the row's end read the row's first chunk instead, K's are
// dropped from the operands and V's channels there are not written
template <class Shape, bool FULL>
__device__ static __forceinline__ void ds_workgroup(const DsArgs& a) {
  constexpr int D = Shape::D, CT = Shape::CT;
  const DcStrides& st = a.st;
  const int g = a.g, hkv = a.hkv, d = a.d;
  constexpr int KS = D / 32, CW = 16 * CT, WAVES = Shape::WAVES, NB = Shape::NB;  // channel steps of S, channels of the slice
  constexpr int KC = D / 8, VC = CW / 8;                                          // chunks of a row
  constexpr int KI = Shape::K_BYTES / 1024, VI = Shape::V_BYTES / 1024;           // instructions of a step
  constexpr int KR = SP_WAVE / KC, VR = SP_WAVE / VC;                             // rows of an instruction
  __shared__ __attribute__((aligned(1024))) char ds_lds[Shape::LDS_BYTES];
  __shared__ float m_s[WAVES][DS_GMAX], l_s[WAVES][DS_GMAX];
  const int slice = CW == D ? 0 : blockIdx.y, split = CW == D ? blockIdx.y : 0, splits = CW == D ? gridDim.y : 1;
  int kvh = blockIdx.x;
  int64_t b = blockIdx.z;
  if constexpr (CW < D) {
    const uint32_t i = blockIdx.z * 8 + blockIdx.x;  // (sequence, kv head)
    b = (i * a.hkv_mul) >> 16;
    kvh = i - (uint32_t)b * hkv;
    if (b >= a.batch || (!FULL && slice * CW >= d)) return;  // (uniform)
  }
  const int64_t bh = b * hkv + kvh;
  const int begin = split * a.keys_per_split, n = a.n_keys - begin < a.keys_per_split ? a.n_keys - begin : a.keys_per_split;
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int lq = lane & 15, gr = lane >> 4;  // head (or key row, channel) in a 16-wide tile, lane group
  dc_bf16x8 qb[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const bool real = lq < g && (FULL || 32 * ks + 8 * gr < d);
    const dc_u32x4 raw = *reinterpret_cast<const dc_u32x4*>(a.q + b * st.q_b + (int64_t)(kvh * g + (lq < g ? lq : 0)) * st.q_h +
                                                           (FULL || real ? 32 * ks + 8 * gr : 0));
    qb[ks] = __builtin_bit_cast(dc_bf16x8, real ? raw : (dc_u32x4){0, 0, 0, 0});
  }
  const char* const kh = (const char*)(a.k + b * st.k_b + kvh * st.k_h + begin * st.k_n);
  const char* const vh = (const char*)(a.v + b * st.v_b + kvh * st.v_h + begin * st.v_n);
  const uint32_t k_row = (uint32_t)st.k_n * 2u, v_row = (uint32_t)st.v_n * 2u;  // bytes
  const uint32_t ring = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)ds_lds + wave * NB * Shape::STEP_BYTES;

  // A step's loads: instruction i fills 1 KiB (lane j its chunk j) with KR or VR rows.  The step is a buffer of its own; only the one
  // that reaches past the cache clamps its rows onto the last key (masked below).
  auto fetch = [&](int buf, int kb) {
    const int rows = n - kb < DS_KEYS ? n - kb : DS_KEYS;
    auto step = [&](const char* x, uint32_t row_bytes) {
      return __builtin_amdgcn_make_buffer_rsrc((void*)(x + (uint64_t)(uint32_t)kb * row_bytes), 0, (int)((uint32_t)(rows - 1) * row_bytes + 2u * d), 0x00027000);
    };
    const __amdgpu_buffer_rsrc_t ksrc = step(kh, k_row), vsrc = step(vh, v_row);
    const uint32_t at = ring + buf * Shape::STEP_BYTES;
    auto within = [&](int chunk) { return 16u * (uint32_t)(FULL || 8 * chunk < d ? chunk : 0); };
    auto k_off = [&](int row) { return within((lane % KC) ^ ds_swz_k<D>(row)); };
    auto v_off = [&](int row) { return within(slice * VC + ((lane % VC) ^ (2 * ds_swz_v<CT>(row)))); };
    if (rows == DS_KEYS) {
#pragma unroll
      for (int i = 0; i < KI; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(ksrc, (ds_lds_ptr)(uintptr_t)(at + i * 1024), 16,
                                                 (int)((lane / KC) * k_row + k_off(i * KR + lane / KC)), (int)(i * KR * k_row), 0, 0);
#pragma unroll
      for (int i = 0; i < VI; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(vsrc, (ds_lds_ptr)(uintptr_t)(at + Shape::K_BYTES + i * 1024), 16,
                                                 (int)((lane / VC) * v_row + v_off(i * VR + lane / VC)), (int)(i * VR * v_row), 0, 0);
    } else {
#pragma unroll 1
      for (int i = 0; i < KI; ++i) {
        const int row = i * KR + lane / KC;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(ksrc, (ds_lds_ptr)(uintptr_t)(at + i * 1024), 16,
                                                 (int)((uint32_t)(row < rows ? row : rows - 1) * k_row + k_off(row)), 0, 0, 0);
      }
#pragma unroll 1
      for (int i = 0; i < VI; ++i) {
        const int row = i * VR + lane / VC;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(vsrc, (ds_lds_ptr)(uintptr_t)(at + Shape::K_BYTES + i * 1024), 16,
                                                 (int)((uint32_t)(row < rows ? row : rows - 1) * v_row + v_off(row)), 0, 0, 0);
      }
    }
  };
  constexpr int STRIDE = WAVES * DS_KEYS;
  const int kb0 = wave * DS_KEYS;
#pragma unroll
  for (int i = 0; i < NB - 1; ++i)
    if (kb0 + i * STRIDE < n) fetch(i, kb0 + i * STRIDE);

  ds_floatx4 o[CT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) o[ct] = (ds_floatx4){0, 0, 0, 0};
  float m = -INFINITY, l = 0.f;  // of head lq; l: this lane group's keys
  const uint32_t k_at = ring + lq * (D * 2);
  const int v_key = 4 * gr + (lq >> 2);  // row of the transposing read; 16 rows further the swizzle is the same
  const uint32_t v_at = ring + Shape::K_BYTES + v_key * (CT * 32) + 8 * (lq & 3);
  int buf = 0;
  for (int kb = kb0; kb < n; kb += STRIDE) {
    // the step's loads have landed, those of the NB - 2 behind it stay in flight (loads return in order)
    if (kb + (NB - 2) * STRIDE < n)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NB - 2) * Shape::LOADS) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    // (the place that is filled here was read in the step before: those reads' results have been used)
    if (kb + (NB - 1) * STRIDE < n) fetch(buf == 0 ? NB - 1 : buf - 1, kb + (NB - 1) * STRIDE);
    const uint32_t off = buf * Shape::STEP_BYTES;
    dc_u32x4 kr[2][KS];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        kr[i][ks] = ds_read_k(k_at + off + i * 16 * (D * 2) + (((4 * ks + gr) ^ ds_swz_k<D>(lq)) << 4));
    if constexpr (KS == 4)
      asm volatile("s_waitcnt lgkmcnt(0)"
                   : "+v"(kr[0][0]), "+v"(kr[0][1]), "+v"(kr[0][2]), "+v"(kr[0][3]), "+v"(kr[1][0]), "+v"(kr[1][1]), "+v"(kr[1][2]), "+v"(kr[1][3]));
    else
      asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(kr[0][0]), "+v"(kr[0][1]), "+v"(kr[1][0]), "+v"(kr[1][1]));
    if constexpr (!FULL) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        if (32 * ks + 8 * gr >= d) kr[0][ks] = kr[1][ks] = (dc_u32x4){0, 0, 0, 0};
    }
    ds_u32x2 vr[CT][2];  // on their way under the logits
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      const uint32_t at = v_at + off + ((ct ^ ds_swz_v<CT>(v_key)) << 5);
      vr[ct][0] = ds_read_v<0>(at);
      vr[ct][1] = ds_read_v<16 * CT * 32>(at);
    }
    ds_floatx4 s[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      s[i] = (ds_floatx4){0, 0, 0, 0};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        s[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(dc_bf16x8, kr[i][ks]), qb[ks], s[i], 0, 0, 0);
    }
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        s[i][j] = kb + 16 * i + 4 * gr + j < n ? s[i][j] * a.scale_log2 : -INFINITY;
        mx = fmaxf(mx, s[i][j]);
      }
    const float m_new = fmaxf(m, ds_quad_max(mx));
    const float base = m_new == -INFINITY ? 0.f : m_new;   // (no key so far has a finite logit: every weight is exp2(-inf) = 0)
    const float alpha = __builtin_amdgcn_exp2f(m - base);  // 0 in the first step
    float add = 0.f;
    uint32_t hi[4], lo[4];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 4; j += 2) {
        const float p0 = __builtin_amdgcn_exp2f(s[i][j] - base), p1 = __builtin_amdgcn_exp2f(s[i][j + 1] - base);
        const uint32_t w = dc_pack2(p0, p1);
        hi[2 * i + j / 2] = w;
        lo[2 * i + j / 2] = dc_pack2(p0 - __uint_as_float(w << 16), p1 - __uint_as_float(w & 0xffff0000u));
        add += p0 + p1;
      }
    l = l * alpha + add;
    m = m_new;
    const dc_bf16x8 ph = __builtin_bit_cast(dc_bf16x8, (dc_u32x4){hi[0], hi[1], hi[2], hi[3]});
    const dc_bf16x8 pl = __builtin_bit_cast(dc_bf16x8, (dc_u32x4){lo[0], lo[1], lo[2], lo[3]});
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(vr[ct][0]), "+v"(vr[ct][1]));
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      o[ct] *= alpha;
      o[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(dc_bf16x8, __builtin_shufflevector(vr[ct][0], vr[ct][1], 0, 1, 2, 3)), ph, o[ct], 0, 0, 0);
    }
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
      o[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(dc_bf16x8, ds_finite(__builtin_shufflevector(vr[ct][0], vr[ct][1], 0, 1, 2, 3))), pl, o[ct], 0, 0, 0);
    buf = buf + 1 == NB ? 0 : buf + 1;
  }
  l = ds_quad_sum(l);
  __syncthreads();  // the rings are free
  auto o_s = reinterpret_cast<float(*)[DS_GMAX][CW + 4]>(ds_lds);
  if (lq < g) {
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) *reinterpret_cast<ds_floatx4*>(&o_s[wave][lq][16 * ct + 4 * gr]) = o[ct];
    if (gr == 0) {
      m_s[wave][lq] = m;
      l_s[wave][lq] = l;
    }
  }
  __syncthreads();
  for (int i = t; i < g * (CW / 4); i += WAVES * SP_WAVE) {
    const int h = i / (CW / 4), c = i % (CW / 4) * 4;
    if (!FULL && slice * CW + c >= d) continue;
    float top = -INFINITY, sum = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) top = fmaxf(top, m_s[w][h]);
    ds_floatx4 acc = {0, 0, 0, 0};
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      // (a wave without keys, or without a finite logit: 0)
      const float f = m_s[w][h] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_s[w][h] - top);
      sum += l_s[w][h] * f;
      acc += *reinterpret_cast<const ds_floatx4*>(&o_s[w][h][c]) * f;
    }
    if (splits > 1) {  // (uniform) the merging kernel goes on
      const int64_t at = (bh * splits + split) * g + h;
      *reinterpret_cast<dc_floatx4*>(a.o_part + at * DC_D + c) = acc;
      if (c == 0) a.ml_part[at] = make_float2(top, sum);
      continue;
    }
    const float inv = 1.0f / sum;
    *reinterpret_cast<uint2*>(a.out + (bh * g + h) * d + slice * CW + c) =
        make_uint2(dc_pack2(acc[0] * inv, acc[1] * inv), dc_pack2(acc[2] * inv, acc[3] * inv));
  }
}
// (the arguments one by one: as one struct they came in one more round of scalar loads, 0.04 us of a step)
#define DS_PARAMS                                                                                                                        \
  const sp_bf16 *__restrict__ q, const sp_bf16 *__restrict__ k, const sp_bf16 *__restrict__ v, int n_keys, int g, int hkv, int d,        \
      int batch, uint32_t hkv_mul, DcStrides st, float scale_log2, int keys_per_split, float *__restrict__ o_part,                       \
      float2 *__restrict__ ml_part, sp_bf16 *__restrict__ out
#define DS_ARGS {q, k, v, n_keys, g, hkv, d, batch, hkv_mul, st, scale_log2, keys_per_split, o_part, ml_part, out}
template <int D, int CT, bool FULL>
__global__ __launch_bounds__((DsWide<D, CT>::WAVES * SP_WAVE)) void sp_decode_ring_kernel(DS_PARAMS) {
  ds_workgroup<DsWide<D, CT>, FULL>(DS_ARGS);
}
template <int D, bool FULL>
__global__ __launch_bounds__((DsPair<D>::WAVES * SP_WAVE)) void sp_decode_ring_pair_kernel(DS_PARAMS) {
  ds_workgroup<DsPair<D>, FULL>(DS_ARGS);
}
template <int D, bool FULL>
__global__ __launch_bounds__((DsQuad<D>::WAVES * SP_WAVE)) void sp_decode_ring_quad_kernel(DS_PARAMS) {
  ds_workgroup<DsQuad<D>, FULL>(DS_ARGS);
}

// How a call of the ring kernel is cut: slices of ct channel tiles (all of them: 16 ct = d) or splits of the keys
enum DsFill { DS_WIDE, DS_PAIR, DS_QUAD };
struct DsPlan {
  int ct, splits;
  DsFill fill;  // (other than DS_WIDE: all channels, no splits)
};

template <int D, int CT, bool FULL>
static int ds_launch(const void* q, const void* k, const void* v, int32_t batch, int64_t n, int32_t hq, int32_t hkv, int32_t d, const DcStrides& st,
                     float scale_log2, const DsPlan& plan, int splits, int keys_per_split, float* o_part, float2* ml_part, void* out, hipStream_t s) {
  const int slices = D / 16 / CT;
  auto launch = [&](dim3 grid, int64_t b0, int32_t count) {
    auto go = [&](auto kernel, int waves) {
      hipLaunchKernelGGL(kernel, grid, dim3(waves * SP_WAVE), 0, s, (const sp_bf16*)q + b0 * st.q_b, (const sp_bf16*)k + b0 * st.k_b,
                         (const sp_bf16*)v + b0 * st.v_b, (int)n, hq / hkv, (int)hkv, (int)d, (int)count, (uint32_t)sp_ceil_div(65536, hkv), st,
                         scale_log2, keys_per_split, o_part, ml_part, (sp_bf16*)out + b0 * hq * d);
    };
    if constexpr (CT * 16 == D) {
      if (plan.fill == DS_PAIR) return go(sp_decode_ring_pair_kernel<D, FULL>, DsPair<D>::WAVES);
      if (plan.fill == DS_QUAD) return go(sp_decode_ring_quad_kernel<D, FULL>, DsQuad<D>::WAVES);
    }
    go(sp_decode_ring_kernel<D, CT, FULL>, DsWide<D, CT>::WAVES);
  };
  if (slices > 1)  // (at most 256 workgroups)
    launch(dim3(8, slices, (unsigned)sp_ceil_div((int64_t)batch * hkv, 8)), 0, batch);
  else
    for (int64_t b0 = 0; b0 < batch; b0 += DC_MAX_GRID_Z) {  // (a batch of more sequences than a grid's z axis is not split)
      const int32_t count = (int32_t)(batch - b0 < DC_MAX_GRID_Z ? batch - b0 : DC_MAX_GRID_Z);
      launch(dim3(hkv, splits, (unsigned)count), b0, count);
    }
  SP_LAUNCH_CHECK();
  return SP_OK;
}

// ---- host -------------------------------------------------------------------------------------------------
// Chunks per (sequence, kv head): about two workgroups per CU over the whole batch, which is what the kernel's LDS
// lets a CU hold, and no chunk below one tile of keys.
static_assert(DC_MAX_GRID_Z >= 512, "");  // (the number of chunks is 1 before a batch needs a second launch)
static int dc_cut(int32_t batch, int64_t n, int32_t hkv) {
  const int64_t tiles = sp_ceil_div(n, DC_TILE);
  int64_t want = sp_ceil_div(512, (int64_t)hkv * batch);
  if (want > tiles) want = tiles;
  if (want < 1) want = 1;
  if (want > DC_MAX_SPLITS) want = DC_MAX_SPLITS;
  return (int)want;
}

// Splits per (sequence, kv head) at most, and what the workspace is sized for.  A cache of up to two tiles is one: no partials.
#define DC_ONE_LAUNCH_TILES 2
static int dc_splits(int32_t batch, int64_t n, int32_t hkv) {
  return n <= DC_ONE_LAUNCH_TILES * DC_TILE ? 1 : dc_cut(batch, n, hkv);
}

// How a call of the ring kernel is cut: slices of the channels in one launch, or splits of the keys and the merging launch -- the
// cheaper by the times they were measured to take with caches that come from memory (replayed graphs over 600 MB of caches; 28 / 4 and
// 32 / 8 heads of 128, 14 / 2 and 32 / 8 of 64 channels, 600 to 4001 keys, 1 to 16 sequences; within some 10 %).  ns:
//   3600 a launch with its first and last step, 3400 the merging one;
//   a key takes a workgroup 5.2 to 8.6 by the slice's width (64 channels 3.8 to 4.1) and a third of what it takes from memory beside the
//   others, or, where that is more, what it takes from memory, at 5.85 TB/s.
// More (sequence, kv head) pairs than CUs are not cut.  Up to 512 of them two workgroups a CU take them in one round; beyond, short caches
// go four to a CU, whose ends pass under each other's loads, and long ones, which keep the memory busy either way, one.  us, one to a CU / so,
// 32 / 8 heads: 264 pairs of 300 keys 16.7 / 13.0, of 4001 126 / 114; 640 of 100 13.8 / 10.9, of 300 26.7 / 22.4, of 2048 114 (two 130, four
// 118); 1536 of 500 71.7 (four 74.2); 4096 of 100 63.7 / 43.7, without groups of 200 92.2 / 74.2; 96 channels 4096 of 500 149 / 138; 64 channels
// 640 of 100 10.3 / 6.5, 4096 of 300 73.3 / 57.5, 2048 of 700 68.7 / 66.7, 1536 of 2048 132 (four 144; with one wave to a workgroup, which
// nine fit of, 138, and 2 to 5 % behind the streaming kernel at 100 keys).
// A launch's host time, 3300, counts half: whether the host or the GPU bounds a step is the caller's.  us, one launch / two: 1025 keys
// 9.1 / 8.5 (called one by one 9.5 / 12.9), 2048 14.3 / 8.7; 4 sequences of 1025 9.8 / 10.3, of 2048 16.0 / 12.4; 8 of 700 8.7 / 11.1, of
// 4001 32.9 / 29.4; 16 of 2000 26.0 / 29.5.
#define DS_QUAD_KEYS 400  // of 128 channels: what is read counts, a padded head's rows are as long as they are
static DsPlan ds_plan(int32_t batch, int64_t n, int32_t hkv, int32_t d, int32_t real_d) {
  const int64_t bh = (int64_t)batch * hkv;
  const int full = d / 16;  // channel tiles
  auto cost = [&](int ct, int64_t heads /* kv heads' keys in flight */, int64_t wgs, int64_t keys) {
    const int64_t alone = d == 64 ? (ct == 1 ? 3800 : 4100) : ct == 1 ? 5200 : ct == 2 ? 5600 : ct == 4 ? 6200 : 8600;  // (ps a key)
    const int64_t memory = heads * 4 * d * 1000 / 5850;
    const int64_t shared = alone + (memory < alone ? memory : alone) / 3;
    return 3600 + sp_ceil_div(wgs, 256) * keys * (memory > shared ? memory : shared) / 1000;
  };
  DsPlan best = {full, 1, DS_WIDE};
  int64_t least = INT64_MAX;
  for (int ct = 1; ct <= full; ct *= 2) {
    const int64_t wgs = bh * (full / ct);
    if (ct < full && wgs > 256) continue;
    const int64_t c = cost(ct, bh < 256 ? bh : 256, wgs, n);
    if (c < least) least = c, best.ct = ct;
  }
  const int room = dc_splits(batch, n, hkv);  // (what the workspace is sized for; 1: there is none)
  const int64_t splits = 256 / bh < room ? 256 / bh : room;
  if (splits > 1) {
    const int64_t keys = sp_ceil_div(sp_ceil_div(n, splits), DC_TILE) * DC_TILE, wgs = bh * sp_ceil_div(n, keys);
    if (cost(full, wgs, wgs, keys) + 3400 + 1650 < least) best = {full, (int)splits, DS_WIDE};
  }
  if (bh > 256) best.fill = bh <= 512 ? DS_PAIR : n * (d == 64 ? 64 : real_d) <= DS_QUAD_KEYS * 128 ? DS_QUAD : DS_WIDE;
  return best;
}

static size_t dc_partial_bytes(int32_t batch, int64_t n, int32_t hq, int32_t hkv) {
  if (batch <= 0 || n <= 0 || hq <= 0 || hkv <= 0) return 0;
  return (size_t)dc_splits(batch, n, hkv) * batch * hq * (DC_D * sizeof(float) + sizeof(float2));
}

// a batch whose caches are one chunk each leaves no partials (at 65535 sequences of 32 heads they would be 1.1 GB)
extern "C" size_t sp_decode_batch_workspace_bytes(int32_t batch, int64_t n, int32_t hq, int32_t hkv) {
  if (batch <= 0 || n <= 0 || hq <= 0 || hkv <= 0 || dc_splits(batch, n, hkv) == 1) return 0;
  return dc_partial_bytes(batch, n, hq, hkv);
}

extern "C" size_t sp_decode_workspace_bytes(int64_t n, int32_t hq, int32_t hkv) {
  return dc_partial_bytes(1, n, hq, hkv);
}

// argument checks shared by the two entry points
static int dc_check(const char* who, const void* q, const void* k, const void* v, int32_t batch, int64_t n, int32_t hq,
                    int32_t hkv, int32_t d, const DcStrides& st, float softmax_scale, const void* out) {
  SP_REQUIRE(q && k && v && out, SP_ERR_INVALID_ARGUMENT, "%s: null pointer", who);
  SP_REQUIRE(n > 0 && hq > 0 && hkv > 0 && hq % hkv == 0, SP_ERR_INVALID_ARGUMENT, "%s: bad shape n=%lld hq=%d hkv=%d",
             who, (long long)n, hq, hkv);
  SP_REQUIRE(batch > 0, SP_ERR_UNSUPPORTED, "%s: batch %d", who, batch);
  SP_REQUIRE(softmax_scale > 0.f, SP_ERR_INVALID_ARGUMENT, "%s: softmax_scale must be > 0", who);
  SP_REQUIRE(d >= 8 && d <= DC_D && d % 8 == 0, SP_ERR_UNSUPPORTED,
             "%s: head_dim %d unsupported (a multiple of 8 up to 128)", who, d);
  SP_REQUIRE(hq / hkv <= DC_GMAX, SP_ERR_UNSUPPORTED, "%s: more than %d query heads per kv head", who, DC_GMAX);
  // q, k and v are read with 16-byte loads
  SP_REQUIRE(st.q_h % 8 == 0 && st.q_b % 8 == 0 && ((uintptr_t)q % 16) == 0, SP_ERR_UNSUPPORTED,
             "%s: q must be 16-byte aligned with strides multiple of 8", who);
  SP_REQUIRE(st.k_n % 8 == 0 && st.k_h % 8 == 0 && st.k_b % 8 == 0 && st.v_n % 8 == 0 && st.v_h % 8 == 0 &&
                 st.v_b % 8 == 0 && ((uintptr_t)k % 16) == 0 && ((uintptr_t)v % 16) == 0,
             SP_ERR_UNSUPPORTED, "%s: k/v must be 16-byte aligned with strides multiple of 8", who);
  return SP_OK;
}

// both kernels; `partials` holds sp_decode_batch_workspace_bytes(batch, n, hq, hkv) bytes, of which the second kernel reads only what
// the first has written (nothing has to be cleared; heads of up to 64 channels write the first 64 of a partial's 128)
static int dc_launch(const void* q, const void* k, const void* v, int32_t batch, int64_t n, int32_t hq, int32_t hkv,
                     int32_t d, const DcStrides& st, float softmax_scale, void* out, void* partials, hipStream_t s) {
  const int g = hq / hkv;
  // (8-byte stores; offsets inside 32 keys and the token count have 32 bits)
  if (g <= DS_GMAX && n < (1 << 30) && (uintptr_t)out % 8 == 0 && st.k_n >= 0 && st.v_n >= 0 && st.k_n < (1 << 25) && st.v_n < (1 << 25)) {
    const float scale_log2 = softmax_scale * 1.4426950408889634f;
    const DsPlan plan = ds_plan(batch, n, hkv, d > 64 ? 128 : 64, d);
    const int keys_per_split = (int)(sp_ceil_div(sp_ceil_div(n, plan.splits), DC_TILE) * DC_TILE);
    const int splits = (int)sp_ceil_div(n, keys_per_split);  // (none without keys)
    float* o_part = (float*)partials;
    float2* ml_part = (float2*)(o_part + (size_t)splits * batch * hq * DC_D);
    auto go = [&](auto launch) { return launch(q, k, v, batch, n, hq, hkv, d, st, scale_log2, plan, splits, keys_per_split, o_part, ml_part, out, s); };
    auto by_slice = [&](auto whole) {
      constexpr bool FULL = decltype(whole)::value;
      if (d > 64)
        return plan.ct == 8   ? go(ds_launch<128, 8, FULL>)
               : plan.ct == 4 ? go(ds_launch<128, 4, FULL>)
               : plan.ct == 2 ? go(ds_launch<128, 2, FULL>)
                              : go(ds_launch<128, 1, FULL>);
      return plan.ct == 4 ? go(ds_launch<64, 4, FULL>) : plan.ct == 2 ? go(ds_launch<64, 2, FULL>) : go(ds_launch<64, 1, FULL>);
    };
    const int rc = d == 64 || d == 128 ? by_slice(std::true_type{}) : by_slice(std::false_type{});
    if (rc || splits == 1) return rc;
    hipLaunchKernelGGL(sp_decode_combine_kernel, dim3((unsigned)((int64_t)batch * hq)), dim3(32 * DC_COMBINE_GROUPS), 0, s, o_part, ml_part, g, splits,
                       (int)d, (sp_bf16*)out);
    SP_LAUNCH_CHECK();
    return SP_OK;
  }
  const int splits = dc_splits(batch, n, hkv);
  const int64_t keys_per_split = sp_ceil_div(sp_ceil_div(n, splits), DC_TILE) * DC_TILE;
  const int tiles_per_chunk = (int)sp_ceil_div(sp_ceil_div(n, dc_cut(1, n, hkv)), DC_TILE);
  float* o_part = (float*)partials;
  float2* ml_part = (float2*)(o_part + (size_t)splits * batch * hq * DC_D);
  const float scale_log2 = softmax_scale * 1.4426950408889634f;
  // A grid's z axis ends at 65535 sequences.  (A batch that large has one workgroup per sequence and kv head: no partials.)
  auto launch = [&](auto kernel) {
    for (int64_t b0 = 0; b0 < batch; b0 += DC_MAX_GRID_Z)
      hipLaunchKernelGGL(kernel, dim3(splits, hkv, (unsigned)(batch - b0 < DC_MAX_GRID_Z ? batch - b0 : DC_MAX_GRID_Z)),
                         dim3(DC_THREADS), 0, s, (const sp_bf16*)q + b0 * st.q_b, (const sp_bf16*)k + b0 * st.k_b,
                         (const sp_bf16*)v + b0 * st.v_b, n, g, (int)d, st, scale_log2, keys_per_split, tiles_per_chunk,
                         o_part, ml_part, (sp_bf16*)out + b0 * hq * d);
  };
  auto by_width = [&](auto g8) {
    constexpr int G8 = decltype(g8)::value;
    // (whole rows of up to 16 heads come here only where the ring kernel cannot take them)
    constexpr bool WHOLE = G8 == 4;
    if (d > 64)
      d == 128 && WHOLE ? launch(sp_decode_partial_kernel<128, G8, WHOLE>) : launch(sp_decode_partial_kernel<128, G8, false>);
    else
      d == 64 && WHOLE ? launch(sp_decode_partial_kernel<64, G8, WHOLE>) : launch(sp_decode_partial_kernel<64, G8, false>);
  };
  if (g <= 8)
    by_width(std::integral_constant<int, 1>{});
  else if (g <= 16)
    by_width(std::integral_constant<int, 2>{});
  else
    by_width(std::integral_constant<int, 4>{});
  SP_LAUNCH_CHECK();
  if (splits == 1) return SP_OK;
  hipLaunchKernelGGL(sp_decode_combine_kernel, dim3((unsigned)((int64_t)batch * hq)), dim3(32 * DC_COMBINE_GROUPS), 0, s,
                     o_part, ml_part, g, splits, (int)d, (sp_bf16*)out);
  SP_LAUNCH_CHECK();
  return SP_OK;
}

extern "C" int sp_decode_attn_batch_bf16(const void* q, const void* k, const void* v, int32_t batch, int64_t n, int32_t hq,
                                         int32_t hkv, int32_t d, int64_t q_stride_b, int64_t q_stride_h,
                                         int64_t k_stride_b, int64_t k_stride_n, int64_t k_stride_h, int64_t v_stride_b,
                                         int64_t v_stride_n, int64_t v_stride_h, float softmax_scale, void* out,
                                         void* workspace, size_t workspace_bytes, sp_stream_t stream) {
  const DcStrides st = {q_stride_b, q_stride_h, k_stride_b, k_stride_n, k_stride_h, v_stride_b, v_stride_n, v_stride_h};
  int rc = dc_check("sp_decode_attn_batch_bf16", q, k, v, batch, n, hq, hkv, d, st, softmax_scale, out);
  if (rc) return rc;
  const size_t need = sp_decode_batch_workspace_bytes(batch, n, hq, hkv);
  SP_REQUIRE(need == 0 || workspace != nullptr, SP_ERR_INVALID_ARGUMENT, "sp_decode_attn_batch_bf16: null workspace");
  SP_REQUIRE(workspace_bytes >= need && ((uintptr_t)workspace % 8) == 0,
             SP_ERR_WORKSPACE, "sp_decode_attn_batch_bf16: workspace too small or misaligned");
  return dc_launch(q, k, v, batch, n, hq, hkv, d, st, softmax_scale, out, workspace, (hipStream_t)stream);
}

extern "C" int sp_decode_attn_batch_args_bf16(const sp_decode_batch_args* a) {
  SP_REQUIRE(a != nullptr, SP_ERR_INVALID_ARGUMENT, "sp_decode_attn_batch_args_bf16: null pointer");
  SP_REQUIRE(a->batch == (int32_t)a->batch && a->hq == (int32_t)a->hq && a->hkv == (int32_t)a->hkv && a->d == (int32_t)a->d,
             SP_ERR_INVALID_ARGUMENT, "sp_decode_attn_batch_args_bf16: a size beyond 32 bits");
  return sp_decode_attn_batch_bf16(a->q, a->k, a->v, (int32_t)a->batch, a->n, (int32_t)a->hq, (int32_t)a->hkv, (int32_t)a->d, a->q_stride_b,
                                   a->q_stride_h, a->k_stride_b, a->k_stride_n, a->k_stride_h, a->v_stride_b, a->v_stride_n, a->v_stride_h,
                                   (float)a->softmax_scale, a->out, a->workspace, (size_t)a->workspace_bytes, a->stream);
}

extern "C" int sp_decode_attn_bf16(const void* q, const void* k, const void* v, int64_t n, int32_t hq, int32_t hkv,
                                   int32_t d, int64_t q_stride_h, int64_t k_stride_n, int64_t k_stride_h,
                                   int64_t v_stride_n, int64_t v_stride_h, float softmax_scale, void* out,
                                   void* workspace, size_t workspace_bytes, sp_stream_t stream) {
  const DcStrides st = {0, q_stride_h, 0, k_stride_n, k_stride_h, 0, v_stride_n, v_stride_h};
  int rc = dc_check("sp_decode_attn_bf16", q, k, v, 1, n, hq, hkv, d, st, softmax_scale, out);
  if (rc) return rc;
  SP_REQUIRE(workspace != nullptr, SP_ERR_INVALID_ARGUMENT, "sp_decode_attn_bf16: null workspace");
  SP_REQUIRE(workspace_bytes >= sp_decode_workspace_bytes(n, hq, hkv) && ((uintptr_t)workspace % 8) == 0,
             SP_ERR_WORKSPACE, "sp_decode_attn_bf16: workspace too small or misaligned");
  return dc_launch(q, k, v, 1, n, hq, hkv, d, st, softmax_scale, out, workspace, (hipStream_t)stream);
}

// ---- the same step for callers that cannot allocate ---------------------------------------------------------------
// The chunk partials live in a file-scope device array instead of a caller's workspace.  Every GPU the library runs on
// holds its own copy of the array (at its own address) until the process ends; the array's name is only a host-side
// handle, so the device address is looked up once per device with hipGetSymbolAddress and that pointer is what the
// kernels get.
#define DC_STATIC_BYTES SP_DECODE_STATIC_SCRATCH_BYTES
#define DC_MAX_DEVICES 64
static __device__ __align__(256) unsigned char scratch[DC_STATIC_BYTES];
static void* dc_scratch_ptr[DC_MAX_DEVICES];  // device address of `scratch` per device, nullptr = not looked up yet
static std::mutex dc_scratch_mutex;

static int dc_static_scratch(void** ptr) {
  int dev = -1;
  SP_HIP(hipGetDevice(&dev));
  SP_REQUIRE(dev >= 0 && dev < DC_MAX_DEVICES, SP_ERR_UNSUPPORTED, "sp_decode_attn_static_bf16: device index %d", dev);
  std::lock_guard<std::mutex> lock(dc_scratch_mutex);
  if (dc_scratch_ptr[dev] == nullptr) {
    void* p = nullptr;
    SP_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    SP_REQUIRE(p != nullptr, SP_ERR_HIP, "sp_decode_attn_static_bf16: no device address for the scratch array");
    dc_scratch_ptr[dev] = p;
  }
  *ptr = dc_scratch_ptr[dev];
  return SP_OK;
}

extern "C" int sp_decode_attn_static_bf16(const void* q, const void* k, const void* v, int64_t n, int32_t hq,
                                          int32_t hkv, int32_t d, int64_t q_stride_h, int64_t k_stride_n,
                                          int64_t k_stride_h, int64_t v_stride_n, int64_t v_stride_h,
                                          float softmax_scale, void* out, sp_stream_t stream) {
  const DcStrides st = {0, q_stride_h, 0, k_stride_n, k_stride_h, 0, v_stride_n, v_stride_h};
  int rc = dc_check("sp_decode_attn_static_bf16", q, k, v, 1, n, hq, hkv, d, st, softmax_scale, out);
  if (rc) return rc;
  const size_t need = sp_decode_workspace_bytes(n, hq, hkv);
  SP_REQUIRE(need <= DC_STATIC_BYTES, SP_ERR_WORKSPACE,
             "sp_decode_attn_static_bf16: n=%lld hq=%d hkv=%d needs %zu bytes of partials, the built-in scratch holds "
             "%u; use sp_decode_attn_bf16 with a workspace",
             (long long)n, hq, hkv, need, (unsigned)DC_STATIC_BYTES);
  void* partials = nullptr;
  rc = dc_static_scratch(&partials);
  if (rc) return rc;
  return dc_launch(q, k, v, 1, n, hq, hkv, d, st, softmax_scale, out, partials, (hipStream_t)stream);
}
