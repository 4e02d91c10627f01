// The key-major copy of V that the persistent attention kernel reads, as device code: the repack launch itself and the launch
// that repacks beside its own work use it.
#pragma once
#include "sp_common.h"

#define RP_BS 128     // keys per tile
#define RP_D 128      // channels
#define RP_PITCH 136  // bf16 elements per LDS row
#define RP_LDS_BYTES (RP_BS * RP_PITCH * 2)

// position p (0..31) inside a group of 32 keys of the repacked V^T row holds key offset at_perm32(p):
// [0-3, 16-19, 4-7, 20-23, 8-11, 24-27, 12-15, 28-31]: lane group g of a wave owns rows 4g .. 4g+3 of both 16x16
// S^T accumulators of a half-tile, and its P^T operand is key slots 8g .. 8g+7
__host__ __device__ static inline int at_perm32(int p) { return 16 * ((p >> 2) & 1) + 4 * (p >> 3) + (p & 3); }

struct RepackArgs {
  const sp_bf16* v;  // [n][hkv][128] by strides
  sp_bf16* vt;       // [hkv][nb][128 channels][128 key slots]
  int64_t n, sv_n, sv_h;
  int nb, hkv;
};

// one tile by the THREADS threads of the workgroup; keys behind the sequence are zeros
template <int THREADS>
__device__ static __forceinline__ void repack_v_tile(const RepackArgs& a, int blk, int kvh, sp_bf16* tile /* LDS, RP_LDS_BYTES */) {
  constexpr int ROWS = THREADS / 16;  // rows at a time: a row is 16 chunks of 16 bytes
  const int t = threadIdx.x, chunk = t & 15;
#pragma unroll
  for (int it = 0; it < RP_BS / ROWS; ++it) {
    const int row = it * ROWS + (t >> 4);
    const int64_t key = (int64_t)blk * RP_BS + row;
    uint4 val = make_uint4(0, 0, 0, 0);
    if (key < a.n) val = *reinterpret_cast<const uint4*>(a.v + (int64_t)kvh * a.sv_h + key * a.sv_n + chunk * 8);
    *reinterpret_cast<uint4*>(&tile[row * RP_PITCH + chunk * 8]) = val;
  }
  __syncthreads();
  sp_bf16* dst = a.vt + (((int64_t)kvh * a.nb + blk) * RP_D) * RP_BS;
#pragma unroll
  for (int it = 0; it < RP_D / ROWS; ++it) {
    const int dd = it * ROWS + (t >> 4);  // output row = channel
    const int p0 = chunk * 8;             // 8 consecutive key slots
    uint32_t w[4];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int slot = p0 + j;
      const int key = (slot & ~31) + at_perm32(slot & 31);
      const uint32_t e = tile[key * RP_PITCH + dd];
      if (j & 1)
        w[j >> 1] |= e << 16;
      else
        w[j >> 1] = e;
    }
    *reinterpret_cast<uint4*>(dst + (int64_t)dd * RP_BS + p0) = make_uint4(w[0], w[1], w[2], w[3]);
  }
}

// host: what both launches refuse, and the arguments; vt holds workspace_bytes bytes
static int repack_args(RepackArgs* a, const char* who, const void* v, int64_t n, int32_t hkv, int32_t d, int64_t v_stride_n,
                       int64_t v_stride_h, int32_t bs, void* vt, size_t workspace_bytes) {
  SP_REQUIRE(v && vt, SP_ERR_INVALID_ARGUMENT, "%s: null pointer", who);
  SP_REQUIRE(n > 0 && hkv > 0, SP_ERR_INVALID_ARGUMENT, "%s: bad shape", who);
  SP_REQUIRE((bs == 128 || bs == 64 || bs == 32 || bs == 16) && d == RP_D, SP_ERR_UNSUPPORTED,
             "%s: block size %d / head_dim %d unsupported (16, 32, 64 or 128 / 128)", who, bs, d);
  SP_REQUIRE(v_stride_n % 8 == 0 && v_stride_h % 8 == 0 && ((uintptr_t)v % 16) == 0 && ((uintptr_t)vt % 16) == 0,
             SP_ERR_UNSUPPORTED, "%s: v must be 16-byte aligned, strides multiple of 8", who);
  const int64_t nb = sp_ceil_div(n, RP_BS);
  SP_REQUIRE(workspace_bytes >= (size_t)hkv * nb * RP_BS * RP_D * sizeof(sp_bf16), SP_ERR_WORKSPACE, "%s: workspace too small", who);
  SP_REQUIRE(nb * hkv < (1ll << 31), SP_ERR_UNSUPPORTED, "%s: grid too large", who);
  *a = RepackArgs{(const sp_bf16*)v, (sp_bf16*)vt, n, v_stride_n, v_stride_h, (int)nb, hkv};
  return SP_OK;
}
