// delta[b, h, q] = sum_d dO * O ahead of the 32-row backward kernels, for outputs whose rows are not 16-byte aligned (aligned
// ones are read by the dQ kernel itself).  One wavefront per row, an element per lane: bound by the 2-byte loads, 3 TB/s.
#include "attn_common.hpp"

namespace {

constexpr int GT = 256;  // threads

__global__ __launch_bounds__(GT) void attn_delta_kernel(const bf16_t* __restrict__ dout, int64_t ds0, int64_t ds1, int64_t ds2,
                                                        const bf16_t* __restrict__ o, int64_t os0, int64_t os1, int64_t os2,
                                                        float* __restrict__ delta, int B, int H, int S, int D) {
  const int lane = threadIdx.x & 63;
  const int64_t row = static_cast<int64_t>(blockIdx.x) * (GT / 64) + (threadIdx.x >> 6);
  const int64_t total = static_cast<int64_t>(B) * H * S;
  if (row >= total) return;
  const int s = static_cast<int>(row % S);
  const int h = static_cast<int>((row / S) % H);
  const int b = static_cast<int>(row / (static_cast<int64_t>(S) * H));
  const bf16_t* dp = dout + b * ds0 + h * ds1 + static_cast<int64_t>(s) * ds2;
  const bf16_t* op = o + b * os0 + h * os1 + static_cast<int64_t>(s) * os2;
  float acc = 0.f;
  for (int d = lane; d < D; d += 64) acc += to_f32<bf16_t>(dp[d]) * to_f32<bf16_t>(op[d]);
  acc = wave_sum(acc);
  if (lane == 0) delta[row] = acc;
}

}  // namespace

int mlts_attn_delta_bf16(const void* dout, const int64_t* dos, const void* o, const int64_t* os, float* delta, int B, int H, int S,
                         int D, hipStream_t st) {
  const int64_t rows = static_cast<int64_t>(B) * H * S;
  if (rows == 0) return MLTS_OK;
  MltsKernelTimer timer("attn_delta", st);
  const int64_t blocks = (rows + (GT / 64) - 1) / (GT / 64);
  hipLaunchKernelGGL(attn_delta_kernel, dim3((unsigned)blocks), dim3(GT), 0, st, static_cast<const bf16_t*>(dout), dos[0], dos[1],
                     dos[2], static_cast<const bf16_t*>(o), os[0], os[1], os[2], delta, B, H, S, D);
  return mlts_check_launch("mlts_attn_delta");
}
