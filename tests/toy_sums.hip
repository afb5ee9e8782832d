// The sums and maxima over a wave and a block that common.h gives to every kernel, in blocks that are not whole waves
// and under a condition on lanes.  One block; v and out: n floats, out [4, n].
#include "common.h"
#include "packed_call.h"

ZK_DEFINE_HOST_SIDE

__global__ void toy_sums_kernel(const float* __restrict__ v, float* __restrict__ out, int n) {
  __shared__ float scratch[16];
  const int i = threadIdx.x;
  out[i] = wave_sum(v[i]);
  out[n + i] = wave_max(v[i]);
  out[2 * n + i] = block_sum(v[i], scratch);
  out[3 * n + i] = block_sum(1.f, scratch);
}
__global__ __launch_bounds__(64) void toy_sums_under_kernel(const float* __restrict__ v, float* __restrict__ out, int n) {
  const int i = threadIdx.x;
  if (i % 3 == 0 && i < n) {             // some lanes of a whole wave
    out[i] = wave_sum(v[i]);
    out[n + i] = wave_max(v[i]);
  }
}

extern "C" int zk_toy_sums(const float* v, float* out, int n, int under, void* stream) {
  ZK_REQUIRE(n > 0 && n <= (under ? 64 : 1024), "zk_toy_sums: one block");
  if (under) toy_sums_under_kernel<<<1, 64, 0, (hipStream_t)stream>>>(v, out, n);
  else toy_sums_kernel<<<1, n, 0, (hipStream_t)stream>>>(v, out, n);
  return zk_launch_status("zk_toy_sums");
}
ZK_PACKED(zk_toy_sums)
