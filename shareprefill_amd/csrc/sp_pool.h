// Block pooling as device code: the pooling kernel itself and the launches that pool beside their own work use it.
//
// One thread owns one 16-byte channel chunk (8 bf16) of one (block, head) and walks a quarter of the block's tokens; the
// four partial results meet in LDS in the fixed order ((p0+p1)+(p2+p3)), so a result does not depend on who computes it.
#pragma once
#include "sp_common.h"

#define POOL_CHUNKS 64  // 16-byte chunks per unit of POOL_CHUNKS * POOL_SPLIT threads (one wave wide)
#define POOL_SPLIT 4    // token sub-ranges per block (one per wave)
#define POOL_THREADS (POOL_CHUNKS * POOL_SPLIT)

// one element into the running value of pool type TYPE
template <int TYPE>
__device__ __forceinline__ void pool_take(float& acc, float v) {
  if (TYPE == SP_POOL_MAX) acc = fmaxf(acc, v);
  else if (TYPE == SP_POOL_MIN) acc = fminf(acc, v);
  else if (TYPE == SP_POOL_MAXABS) acc = fmaxf(acc, fabsf(v));
  else acc += v;
}
// two partial values of pool type TYPE
template <int TYPE>
__device__ __forceinline__ float pool_join(float a, float b) {
  if (TYPE == SP_POOL_MAX || TYPE == SP_POOL_MAXABS) return fmaxf(a, b);
  if (TYPE == SP_POOL_MIN) return fminf(a, b);
  return a + b;
}

// quarter `sub` of block [t_begin, t_begin + bs) of the chunk whose token 0 is at `base`
template <int TYPE>
__device__ __forceinline__ void pool_quarter(const sp_bf16* __restrict__ base, int64_t sx_n, int64_t t_begin, int64_t n,
                                             int bs, int sub, float (&acc)[8]) {
  const int64_t t_end = (t_begin + bs < n) ? t_begin + bs : n;
  const int per = bs / POOL_SPLIT;
  int64_t t = t_begin + (int64_t)sub * per;
  const int64_t t1 = t + per < t_end ? t + per : t_end;
  for (; t + 8 <= t1; t += 8) {
    uint4 v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = *reinterpret_cast<const uint4*>(base + (t + u) * sx_n);
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const uint32_t w[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        pool_take<TYPE>(acc[2 * j], __uint_as_float(w[j] << 16));
        pool_take<TYPE>(acc[2 * j + 1], __uint_as_float(w[j] & 0xffff0000u));
      }
    }
  }
  for (; t < t1; ++t) {
    uint4 v = *reinterpret_cast<const uint4*>(base + t * sx_n);
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      pool_take<TYPE>(acc[2 * j], __uint_as_float(w[j] << 16));
      pool_take<TYPE>(acc[2 * j + 1], __uint_as_float(w[j] & 0xffff0000u));
    }
  }
}

// the four quarters' results part[0..3][lane] of a block of cnt tokens -> the 8 pooled channels at dst
template <int TYPE>
__device__ __forceinline__ void pool_store(const float (*part)[POOL_CHUNKS][8], int lane, int cnt, int bs, int tail_mode,
                                           sp_bf16* __restrict__ dst) {
  uint32_t o[4];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    float s = pool_join<TYPE>(pool_join<TYPE>(part[0][lane][j], part[1][lane][j]),
                              pool_join<TYPE>(part[2][lane][j], part[3][lane][j]));
    float m;
    if (TYPE != SP_POOL_AVG) {
      m = s;
    } else if (tail_mode == SP_POOL_TAIL_RESCALE && cnt != bs) {
      m = sp_round_bf16(s / (float)bs);
      m = sp_round_bf16(m * (float)bs);
      m = m / (float)cnt;
    } else {
      m = s / (float)cnt;
    }
    uint32_t b = sp_f32_to_bf16(m);
    if (j & 1)
      o[j / 2] |= b << 16;
    else
      o[j / 2] = b;
  }
  *reinterpret_cast<uint4*>(dst) = make_uint4(o[0], o[1], o[2], o[3]);
}

struct PoolArgs {
  const sp_bf16* x;  // [n][h][d] by strides
  sp_bf16* y;        // [nb][h][d]
  int64_t n, sx_n, sx_h;
  int h, d, bs, tail_mode;
  const int32_t* head_enable;  // [h] or null
  int chunks_per_block, groups_per_block;
  int64_t units;  // blocks x groups of POOL_CHUNKS chunks
};

static inline PoolArgs pool_args(const void* x, void* y, int64_t n, int32_t h, int32_t d, int64_t sx_n, int64_t sx_h,
                                 int32_t bs, int32_t tail_mode, const int32_t* head_enable) {
  const int chunks = h * (d / 8), groups = (int)sp_ceil_div(chunks, POOL_CHUNKS);
  return PoolArgs{(const sp_bf16*)x, (sp_bf16*)y, n, sx_n, sx_h, h, d, bs, tail_mode, head_enable, chunks, groups,
                  sp_ceil_div(n, bs) * groups};
}

// unit `unit` by the POOL_THREADS threads t = 0 .. POOL_THREADS - 1 that call it; every thread of the workgroup calls it
// (it holds a barrier), also for a unit past the last one
template <int TYPE>
__device__ __forceinline__ void pool_unit(const PoolArgs& a, int64_t unit, int t, float (*part)[POOL_CHUNKS][8]) {
  const int lane = t % POOL_CHUNKS, sub = t / POOL_CHUNKS;
  const int64_t blk = unit / a.groups_per_block;
  const int chunk = (int)(unit % a.groups_per_block) * POOL_CHUNKS + lane;
  const int dchunks = a.d / 8;
  const bool active = unit < a.units && chunk < a.chunks_per_block;
  const int head = active ? chunk / dchunks : 0;
  const int d0 = active ? (chunk % dchunks) * 8 : 0;
  const bool enabled = active && (a.head_enable == nullptr || a.head_enable[head] != 0);
  const int64_t t_begin = blk * a.bs;
  const int64_t t_end = (t_begin + a.bs < a.n) ? t_begin + a.bs : a.n;
  // The reference's kernel loads the tokens of a ragged last block that lie beyond the sequence as zeros
  // (utils.py:168-179, other=0), so there a maximum is at least 0 and a minimum at most 0: the neutral start value
  // is 0 for that block, and for sums everywhere.
  const bool ragged = t_end - t_begin < a.bs;
  const float start = (TYPE == SP_POOL_MAX && !ragged) ? -INFINITY : (TYPE == SP_POOL_MIN && !ragged) ? INFINITY : 0.f;
  float acc[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) acc[j] = start;
  if (enabled) pool_quarter<TYPE>(a.x + (int64_t)head * a.sx_h + d0, a.sx_n, t_begin, a.n, a.bs, sub, acc);
#pragma unroll
  for (int j = 0; j < 8; ++j) part[sub][lane][j] = acc[j];
  __syncthreads();
  if (sub == 0 && enabled)
    pool_store<TYPE>(part, lane, (int)(t_end - t_begin), a.bs, a.tail_mode, a.y + (blk * a.h + head) * (int64_t)a.d + d0);
}
