// argmax.hip - per-row greedy token pick over a logits matrix, the step
// after the paged-attention path (rvllm: src/cuda/kernels/argmax.cu via
// argmax_wrapper, src/cuda/ops.rs:516-550, queued behind the forward at
// src/cuda/engine.rs:118-125).
//
// Semantics are those of the greedy scan in Sampler::sample_slice
// (src/sampler.rs:64-75): the first maximum wins (lowest index on ties),
// NaN is never a maximum, and a row with nothing above -inf gives 0.
//
// One workgroup per row: 1024 threads, so a few rows (a decode step's, far
// fewer than CUs) have enough loads in flight, four 16-byte ones a thread (a
// scalar loop if the row is not 16-byte aligned or a multiple of 4 long);
// 256 threads from 512 rows on, where the rows fill the chip. Each lane keeps
// its best (value, index), with strictly-greater updates so its own first
// maximum wins; a wave reduces by xor shuffles and the waves through LDS,
// preferring the larger value and, on equal values, the smaller index. Bound
// by the loads' latency for few rows (1 x 32000 6.4 -> 3.9 us, 1 x 151936 23.8
// -> 7.1, 64 x 151936 45.4 -> 9.9), by HBM for many (2000 x 32000 36.9 us).
#include "pool.h"

using rvkv_detail::fail;
using rvkv_detail::hip_fail;

namespace {

__device__ __forceinline__ void take(float &bv, uint32_t &bi, float v,
                                     uint32_t i) {
  if (v > bv || (v == bv && i < bi)) {
    bv = v;
    bi = i;
  }
}

template <bool VEC, int T>
__global__ void __launch_bounds__(T)
    argmax_kernel(const float *__restrict__ x, uint32_t row_len,
                  uint32_t *__restrict__ out) {
  const float *row = x + (size_t)blockIdx.x * row_len;
  float bv = -__builtin_inff();
  uint32_t bi = 0xffffffffu;
  if constexpr (VEC) {
    const float4 *r4 = reinterpret_cast<const float4 *>(row);
    const uint32_t n4 = row_len / 4;
    auto best4 = [&](const float4 v, uint32_t i) {
      if (v.x > bv) { bv = v.x; bi = i; }
      if (v.y > bv) { bv = v.y; bi = i + 1; }
      if (v.z > bv) { bv = v.z; bi = i + 2; }
      if (v.w > bv) { bv = v.w; bi = i + 3; }
    };
    uint32_t c = threadIdx.x;
    for (; c + 3 * T < n4; c += 4 * T) {
      const float4 v0 = r4[c], v1 = r4[c + T], v2 = r4[c + 2 * T],
                   v3 = r4[c + 3 * T];
      best4(v0, 4 * c);
      best4(v1, 4 * (c + T));
      best4(v2, 4 * (c + 2 * T));
      best4(v3, 4 * (c + 3 * T));
    }
    for (; c < n4; c += T) best4(r4[c], 4 * c);
  } else {
    for (uint32_t i = threadIdx.x; i < row_len; i += T) {
      const float v = row[i];
      if (v > bv) { bv = v; bi = i; }
    }
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const float ov = __shfl_xor(bv, o);
    const uint32_t oi = __shfl_xor(bi, o);
    take(bv, bi, ov, oi);
  }
  __shared__ float sv[T / 64];
  __shared__ uint32_t si[T / 64];
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    sv[wave] = bv;
    si[wave] = bi;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < T / 64; ++w) take(bv, bi, sv[w], si[w]);
    out[blockIdx.x] = bi == 0xffffffffu ? 0u : bi;
  }
}

}  // namespace

extern "C" {

int rvkv_argmax(const float *logits, uint32_t rows, uint32_t row_len,
                uint32_t *out, rvkv_stream stream) {
  const char *op = "argmax";
  if (rows == 0) return RVKV_OK;
  if (!logits || !out) return fail(RVKV_EINVAL, op, "NULL logits or out");
  if (row_len == 0) return fail(RVKV_EINVAL, op, "row_len must be positive");
  const hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const bool vec = row_len % 4 == 0 && (uintptr_t)logits % 16 == 0;
#define RVKV_ARGMAX(VEC, T)                                               \
  hipLaunchKernelGGL((argmax_kernel<VEC, T>), dim3(rows), dim3(T), 0, st, \
                     logits, row_len, out)
  if (rows < 512) {
    if (vec) RVKV_ARGMAX(true, 1024);
    else RVKV_ARGMAX(false, 1024);
  } else {
    if (vec) RVKV_ARGMAX(true, 256);
    else RVKV_ARGMAX(false, 256);
  }
#undef RVKV_ARGMAX
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? RVKV_OK : hip_fail(op, e);
}

}  // extern "C"
