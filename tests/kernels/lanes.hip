// The moves between lanes of csrc/common.h, written out for every lane of a wave: for tests.
#include "common.h"

template <int O>
__device__ __forceinline__ void steps(const float* x, float* out, int n, int lane) {
  const float v = x[lane];
  out[(0 * 6 + n) * WAVE + lane] = lane_xor<O>(v);
  out[(1 * 6 + n) * WAVE + lane] = xor_sum<O>(v);
  out[(2 * 6 + n) * WAVE + lane] = xor_max<O>(v);
  out[(3 * 6 + n) * WAVE + lane] = lanes_sum<2 * O>(v);
  out[(4 * 6 + n) * WAVE + lane] = lanes_max<2 * O>(v);
  const double wide = lane_xor<O>((double)v * 1.0000000001);
  out[(5 * 6 + n) * WAVE + lane] = wide == (double)lane_xor<O>(v) * 1.0000000001 ? (float)lane_xor<O>(lane) : -1.f;
  out[(6 * 6 + n) * WAVE + lane] = of_lane(v, 2 * O - 1);
}

__global__ void lanes_kernel(const float* __restrict__ x, float* __restrict__ out) {
  const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
  x += wave * WAVE;
  out += wave * 7 * 6 * WAVE;
  steps<1>(x, out, 0, lane);
  steps<2>(x, out, 1, lane);
  steps<4>(x, out, 2, lane);
  steps<8>(x, out, 3, lane);
  steps<16>(x, out, 4, lane);
  steps<32>(x, out, 5, lane);
}

// x [waves, 64] -> out [waves, 7, 6, 64]; what the seven are says `steps`, the six are distances 1, 2, 4 .. 32.
extern "C" int test_lanes(const float* x, float* out, int waves, void* stream) {
  if (waves < 1 || waves > 16) return -1;
  lanes_kernel<<<1, waves * WAVE, 0, (hipStream_t)stream>>>(x, out);
  return hipGetLastError() == hipSuccess ? 0 : -2;
}
