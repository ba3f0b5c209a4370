// sl_sqrt_inv (csrc/common.hpp) against the correctly rounded square root and
// reciprocal, sqrtf(x) and 1.0f / sqrtf(x), at every float: where it returns
// true both have to carry the same bits, which rests on the rounding of
// v_rsq_f32 and on the compiler keeping its operations.  Built with the
// library's device flags.
//
//   sqrtinv_gpu     exit 0 when nothing accepted differs
// Prints the floats accepted; of those, the roots and reciprocals that differ;
// the floats of [2^-96, 2^96) refused, and those of them whose reciprocal the
// formula has wrong (what the refusal is for).
#include <cmath>
#include <cstdio>
#include <cstring>

#include "common.hpp"

namespace {

enum { kAccepted, kBadRoot, kBadInv, kRefused, kRefusedWrong, kCounts };

__global__ __launch_bounds__(256) void sweep_kernel(unsigned long long* __restrict__ counts) {
  unsigned long long c[kCounts] = {};
  const unsigned stride = gridDim.x * 256u;  // divides 2^32
  unsigned b = blockIdx.x * 256u + threadIdx.x;
  for (unsigned long long k = 0; k < (1ull << 32) / stride; ++k, b += stride) {
    const float x = __uint_as_float(b);
    float rho, inv;
    const bool ok = sl_sqrt_inv(x, rho, inv);
    const float r = sqrtf(x), i = 1.0f / r;
    const bool inside = x >= 0x1p-96f && x < 0x1p96f;
    c[kAccepted] += ok;
    c[kBadRoot] += ok && __float_as_uint(rho) != __float_as_uint(r);
    c[kBadInv] += ok && __float_as_uint(inv) != __float_as_uint(i);
    c[kRefused] += !ok && inside;
    c[kRefusedWrong] += !ok && inside && __float_as_uint(inv) != __float_as_uint(i);
  }
  for (int q = 0; q < kCounts; ++q)
    if (c[q]) atomicAdd(counts + q, c[q]);
}

bool ok(hipError_t e, const char* what) {
  if (e != hipSuccess) std::fprintf(stderr, "%s: %s\n", what, hipGetErrorString(e));
  return e == hipSuccess;
}

}  // namespace

int main() {
  unsigned long long* d = nullptr;
  unsigned long long h[kCounts] = {};
  if (!ok(hipMalloc(&d, sizeof(h)), "hipMalloc") ||
      !ok(hipMemcpy(d, h, sizeof(h), hipMemcpyHostToDevice), "copy"))
    return 1;
  hipLaunchKernelGGL(sweep_kernel, dim3(4096), dim3(256), 0, 0, d);
  if (!ok(hipGetLastError(), "launch") || !ok(hipMemcpy(h, d, sizeof(h), hipMemcpyDeviceToHost), "copy"))
    return 1;
  (void)hipFree(d);
  std::printf("accepted %llu roots_differ %llu reciprocals_differ %llu refused %llu "
              "refused_wrong %llu\n",
              h[kAccepted], h[kBadRoot], h[kBadInv], h[kRefused], h[kRefusedWrong]);
  return h[kBadRoot] || h[kBadInv] ? 1 : 0;
}
