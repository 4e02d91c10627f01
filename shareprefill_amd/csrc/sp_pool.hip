// Block pooling (HBM-bound): x[n][h][d] bf16 -> y[nb][h][d] bf16; averages and sums accumulate in fp32.
// Replaces the reference's bnhd_pool_kernel (shareprefill/attn/utils.py:131-208), all five of its pool types
// (avg 0, max 1, min 2, max of absolute values 3, sum 4); the selection itself only ever asks for the average
// (attention_sharing.py:194-196).
//
// One workgroup per unit of sp_pool.h: a wave reads 1 KiB of contiguous channels per token, and the four waves split the
// block's tokens.
#include "sp_pool.h"

template <int TYPE>
__global__ __launch_bounds__(POOL_THREADS) void sp_pool_kernel(PoolArgs a) {
  __shared__ float part[POOL_SPLIT][POOL_CHUNKS][8];
  pool_unit<TYPE>(a, blockIdx.x, threadIdx.x, part);
}

static int pool_launch(int pool_type, const void* x, void* y, int64_t n, int32_t h, int32_t d, int64_t x_stride_n,
                       int64_t x_stride_h, int32_t bs, int32_t tail_mode, const int32_t* head_enable,
                       sp_stream_t stream);

extern "C" int sp_pool_avg_bf16(const void* x, void* y, int64_t n, int32_t h, int32_t d, int64_t x_stride_n,
                                int64_t x_stride_h, int32_t bs, int32_t tail_mode, const int32_t* head_enable,
                                sp_stream_t stream) {
  return pool_launch(SP_POOL_AVG, x, y, n, h, d, x_stride_n, x_stride_h, bs, tail_mode, head_enable, stream);
}

extern "C" int sp_pool_bf16(const void* x, void* y, int64_t n, int32_t h, int32_t d, int64_t x_stride_n,
                            int64_t x_stride_h, int32_t bs, int32_t pool_type, sp_stream_t stream) {
  SP_REQUIRE(pool_type >= SP_POOL_AVG && pool_type <= SP_POOL_SUM, SP_ERR_INVALID_ARGUMENT,
             "sp_pool_bf16: unknown pool type %d", pool_type);
  return pool_launch(pool_type, x, y, n, h, d, x_stride_n, x_stride_h, bs, SP_POOL_TAIL_TRUE_LENGTH, nullptr, stream);
}

static int pool_launch(int pool_type, const void* x, void* y, int64_t n, int32_t h, int32_t d, int64_t x_stride_n,
                       int64_t x_stride_h, int32_t bs, int32_t tail_mode, const int32_t* head_enable,
                       sp_stream_t stream) {
  SP_REQUIRE(x && y, SP_ERR_INVALID_ARGUMENT, "sp_pool_avg_bf16 / sp_pool_bf16: null tensor pointer");
  SP_REQUIRE(n > 0 && h > 0 && d > 0, SP_ERR_INVALID_ARGUMENT, "sp_pool_avg_bf16 / sp_pool_bf16: n, h, d must be positive");
  SP_REQUIRE(d % 8 == 0, SP_ERR_UNSUPPORTED, "sp_pool_avg_bf16 / sp_pool_bf16: head_dim %d is not a multiple of 8", d);
  SP_REQUIRE(bs >= POOL_SPLIT && bs % POOL_SPLIT == 0, SP_ERR_UNSUPPORTED,
             "sp_pool_avg_bf16 / sp_pool_bf16: block size %d is not a multiple of %d", bs, POOL_SPLIT);
  SP_REQUIRE(x_stride_n % 8 == 0 && x_stride_h % 8 == 0 && ((uintptr_t)x % 16) == 0 && ((uintptr_t)y % 16) == 0,
             SP_ERR_UNSUPPORTED, "sp_pool_avg_bf16 / sp_pool_bf16: tensors must be 16-byte aligned with strides multiple of 8");
  SP_REQUIRE(tail_mode == SP_POOL_TAIL_TRUE_LENGTH || tail_mode == SP_POOL_TAIL_RESCALE, SP_ERR_INVALID_ARGUMENT,
             "sp_pool_avg_bf16 / sp_pool_bf16: unknown tail_mode %d", tail_mode);
  const PoolArgs a = pool_args(x, y, n, h, d, x_stride_n, x_stride_h, bs, tail_mode, head_enable);
  SP_REQUIRE(a.units < (1ll << 31), SP_ERR_UNSUPPORTED, "sp_pool_avg_bf16 / sp_pool_bf16: grid too large");
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)a.units), dim3(POOL_THREADS), 0, (hipStream_t)stream, a);
  };
  switch (pool_type) {
    case SP_POOL_MAX: launch(sp_pool_kernel<SP_POOL_MAX>); break;
    case SP_POOL_MIN: launch(sp_pool_kernel<SP_POOL_MIN>); break;
    case SP_POOL_MAXABS: launch(sp_pool_kernel<SP_POOL_MAXABS>); break;
    case SP_POOL_SUM: launch(sp_pool_kernel<SP_POOL_SUM>); break;
    default: launch(sp_pool_kernel<SP_POOL_AVG>); break;
  }
  SP_LAUNCH_CHECK();
  return SP_OK;
}
