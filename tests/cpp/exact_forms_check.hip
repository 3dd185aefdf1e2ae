// Device check of the correctly rounded fp32 forms of mcx_internal.h whose
// operands are not a small set (built by marching_cube_amd/build.py, run by
// tests/test_exact_forms_gpu.py), against IEEE division and square root:
//  * recip_rn(b) for all 2^23 significands of b;
//  * sqrt_rn(x) for all 2^24 floats of [1, 4);
//  * div_rn(a, b, recip_rn(b)) for every pair of significands whose quotient
//    lies so near the middle of two floats that the form's error could matter:
//    with A, B in [2^23, 2^24) the numerator's and denominator's significands
//    and M the result's, |2^s A - (2 M + 1) B| <= 16 (s = 25 where A < B, else
//    24).  For B = 2^t o (o odd) and a given difference d, A is the solution of
//    2^s A = B + d modulo 2 B: none unless 2^(t+1) divides B + d, else one
//    modulo o, found by halving (B + d) / 2^(t+1) modulo o s - t - 1 times.
// Prints "recip_mismatch R sqrt_mismatch S div_mismatch D pairs P"; exits 0
// when run.
#include <hip/hip_runtime.h>

#include <cstdio>

#include "mcx_internal.h"

namespace {

__global__ void check_recip(unsigned long long* cnt) {
  const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (1u << 23)) return;
  const float b = __uint_as_float(0x3f800000u | i);
  if (mcx::recip_rn(b) != 1.0f / b) atomicAdd(&cnt[0], 1ull);
}

__global__ void check_sqrt(unsigned long long* cnt) {
  const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (1u << 24)) return;
  const float x = __uint_as_float(0x3f800000u + i);
  if (mcx::sqrt_rn(x) != sqrtf(x)) atomicAdd(&cnt[1], 1ull);
}

__global__ void check_div(unsigned long long* cnt) {
  const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (1u << 23)) return;
  const long long B = (1ll << 23) + i;
  int t = 0;
  while (!((B >> t) & 1)) ++t;
  const long long o = B >> t;
  const float b = (float)B, r = mcx::recip_rn(b);
  unsigned long long pairs = 0, bad = 0;
  for (int above = 0; above < 2; ++above) {
    const int s = above ? 24 : 25;
    const long long lo = above ? B : 1ll << 23, hi = above ? 1ll << 24 : B;
    for (int d = -16; d <= 16; ++d) {
      const long long v = B + d;
      if (d == 0 || (v & ((1ll << (t + 1)) - 1))) continue;
      long long x = (v >> (t + 1)) % o;
      for (int k = 0; k < s - t - 1; ++k) x = x & 1 ? (x + o) >> 1 : x >> 1;
      for (long long A = x + (lo - x + o - 1) / o * o; A < hi; A += o) {
        ++pairs;
        if (mcx::div_rn((float)A, b, r) != (float)A / b) ++bad;
      }
    }
  }
  atomicAdd(&cnt[3], pairs);
  if (bad) atomicAdd(&cnt[2], bad);
}

}  // namespace

int main() {
  unsigned long long* d = nullptr;
  if (hipMalloc(&d, 4 * sizeof(unsigned long long)) != hipSuccess) return 2;
  if (hipMemset(d, 0, 4 * sizeof(unsigned long long)) != hipSuccess) return 2;
  hipLaunchKernelGGL(check_recip, dim3((1 << 23) / 256), dim3(256), 0, 0, d);
  hipLaunchKernelGGL(check_sqrt, dim3((1 << 24) / 256), dim3(256), 0, 0, d);
  hipLaunchKernelGGL(check_div, dim3((1 << 23) / 256), dim3(256), 0, 0, d);
  if (hipDeviceSynchronize() != hipSuccess) return 3;
  unsigned long long h[4] = {};
  if (hipMemcpy(h, d, sizeof(h), hipMemcpyDeviceToHost) != hipSuccess) return 3;
  std::printf("recip_mismatch %llu sqrt_mismatch %llu div_mismatch %llu pairs %llu\n", h[0], h[1],
              h[2], h[3]);
  return hipFree(d) == hipSuccess ? 0 : 4;
}
