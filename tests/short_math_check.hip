// Device check of the walk's short square root and reciprocal (sqrt_short,
// rcp_short in simplehydrology_amd/csrc/shy_kernels.hpp): over every float of
// [2^-100, 2^126) the result must be the correctly rounded one, by its definition:
// the midpoints to its two neighbours enclose the exact value.  A midpoint has 25
// bits, so its square and its product with a float are exact in double, and
// neither equals the value they are compared with.
#include "../simplehydrology_amd/csrc/shy_kernels.hpp"

namespace {
constexpr uint32_t kFirst = 27u << 23, kLast = 253u << 23;  // 2^-100, 2^126
constexpr int kPerThread = 64;
static_assert((kLast - kFirst) % (256 * kPerThread) == 0, "whole blocks");

__device__ double mid(float a, float b) { return 0.5 * ((double)a + (double)b); }

__global__ void check(unsigned long long* bad) {
  const uint32_t base = kFirst + blockIdx.x * (256u * kPerThread) + threadIdx.x;
  unsigned long long s = 0, r = 0;
  for (int i = 0; i < kPerThread; ++i) {
    const float x = __uint_as_float(base + 256u * i);
    const float q = shy::sqrt_short(x), y = shy::rcp_short(x);
    const uint32_t qb = __float_as_uint(q), yb = __float_as_uint(y);
    const double ql = mid(__uint_as_float(qb - 1), q), qh = mid(q, __uint_as_float(qb + 1));
    const double yl = mid(__uint_as_float(yb - 1), y), yh = mid(y, __uint_as_float(yb + 1));
    if (!(ql * ql < (double)x && (double)x < qh * qh)) ++s;
    if (!(yl * (double)x < 1.0 && 1.0 < yh * (double)x)) ++r;
  }
  if (s) atomicAdd(&bad[0], s);
  if (r) atomicAdd(&bad[1], r);
}
}  // namespace

// out[3] = {floats checked, wrong roots, wrong reciprocals}; 0 or a HIP error
extern "C" int short_math_check(unsigned long long* out) {
  unsigned long long* d = nullptr;
  hipError_t e = hipMalloc(&d, 2 * sizeof(*d));
  if (e != hipSuccess) return (int)e;
  const unsigned long long zero[2] = {0, 0};
  e = hipMemcpy(d, zero, sizeof(zero), hipMemcpyHostToDevice);
  if (e == hipSuccess) {
    check<<<(kLast - kFirst) / (256 * kPerThread), 256>>>(d);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipMemcpy(out + 1, d, sizeof(zero), hipMemcpyDeviceToHost);
  hipFree(d);
  out[0] = kLast - kFirst;
  return (int)e;
}
