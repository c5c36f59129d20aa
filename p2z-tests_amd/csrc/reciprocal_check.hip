// Checks the reference typing's reciprocals (p2z_lane.hpp) against the
// divisions that they stand for, on the GPU:
//   fast_rcp     every float with |x| in (2^-100, 2^100)
//   ref_rcp      every float
//   rcp_f64      the largest |1 - x rcp(x)| of the hardware's FP64 reciprocal,
//                over every 24-bit mantissa with the 29 bits below it all 0 and
//                all 1, and 2^30 pseudorandom mantissas
//   ref_inv_det  2^30 pseudorandom doubles with |x| in (2^-120, 2^120), and the
//                9 doubles around the reciprocal of each middle of two floats
//                (each 25-bit odd mantissa)
// Prints one line each: the operands checked, how many differ, or the error.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>

#include "p2z_lane.hpp"

namespace {

using p2z::fast_rcp;
using p2z::ref_inv_det;
using p2z::ref_rcp;

struct Result {
  unsigned long long checked, differ, error;  // error: bits of a double >= 0
};

constexpr int kThreads = 256, kBlocks = 8192;

__device__ inline bool same(float a, float b) {
  return __builtin_bit_cast(uint32_t, a) == __builtin_bit_cast(uint32_t, b) || (a != a && b != b);
}

__device__ inline uint64_t mix(uint64_t x) {  // splitmix64
  x += 0x9e3779b97f4a7c15u;
  x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9u;
  x = (x ^ (x >> 27)) * 0x94d049bb133111ebu;
  return x ^ (x >> 31);
}

__device__ inline void report(Result* r, unsigned long long checked, unsigned long long differ, double error) {
  atomicAdd(&r->checked, checked);
  if (differ) atomicAdd(&r->differ, differ);
  atomicMax(&r->error, __builtin_bit_cast(unsigned long long, error));
}

__global__ __launch_bounds__(kThreads) void k_floats(Result* fast, Result* any) {
  unsigned long long nf = 0, df = 0, na = 0, da = 0;
  const uint64_t step = (uint64_t)gridDim.x * kThreads;
  for (uint64_t i = (uint64_t)blockIdx.x * kThreads + threadIdx.x; i < (1ull << 32); i += step) {
    const float x = __builtin_bit_cast(float, (uint32_t)i);
    const float want = (float)(1. / (double)x);
    const float a = __builtin_fabsf(x);
    if (a > 0x1p-100f && a < 0x1p100f) {
      ++nf;
      df += !same(fast_rcp(x), want);
    }
    ++na;
    da += !same(ref_rcp(x), want);
  }
  report(fast, nf, df, 0.);
  report(any, na, da, 0.);
}

__device__ inline double mantissa(uint64_t m52) { return __builtin_bit_cast(double, 0x3ff0000000000000u | m52); }

__global__ __launch_bounds__(kThreads) void k_rcp_error(Result* r) {
  unsigned long long n = 0;
  double worst = 0.;
  auto check = [&](double x) {
    const double e = __builtin_fabs(__builtin_fma(-x, __builtin_amdgcn_rcp(x), 1.0));
    worst = e > worst ? e : worst;
    ++n;
  };
  const uint64_t step = (uint64_t)gridDim.x * kThreads, first = (uint64_t)blockIdx.x * kThreads + threadIdx.x;
  for (uint64_t i = first; i < (1ull << 23); i += step) {
    check(mantissa(i << 29));
    check(mantissa(i << 29 | 0x1fffffffu));
  }
  for (uint64_t i = first; i < (1ull << 30); i += step) check(mantissa(mix(i) >> 12));
  report(r, n, 0, worst);
}

__global__ __launch_bounds__(kThreads) void k_inv_det(Result* r) {
  unsigned long long n = 0, d = 0;
  auto check = [&](double x) {
    ++n;
    d += !same(ref_inv_det(x), (float)(1. / x));
  };
  const uint64_t step = (uint64_t)gridDim.x * kThreads, first = (uint64_t)blockIdx.x * kThreads + threadIdx.x;
  for (uint64_t i = first; i < (1ull << 30); i += step) {
    const uint64_t h = mix(i + (1ull << 40)), e = mix(h);
    const uint64_t bits = (1023 - 119 + e % 239) << 52 | h >> 12;  // exponents -119 .. 119
    check(__builtin_bit_cast(double, bits | (e >> 63) << 63));
  }
  for (uint64_t i = first; i < (1ull << 24); i += step) {
    const uint64_t x = __builtin_bit_cast(uint64_t, 1. / (double)(1ull << 24 | i | 1ull));
    for (int k = -4; k <= 4; ++k) check(__builtin_bit_cast(double, x + k));
  }
  report(r, n, d, 0.);
}

bool ok(hipError_t e, const char* what) {
  if (e != hipSuccess) std::fprintf(stderr, "%s: %s\n", what, hipGetErrorString(e));
  return e == hipSuccess;
}

}  // namespace

int main() {
  Result* dev = nullptr;
  Result r[4] = {};
  if (!ok(hipMalloc((void**)&dev, sizeof r), "hipMalloc")) return 1;
  if (!ok(hipMemcpy(dev, r, sizeof r, hipMemcpyHostToDevice), "hipMemcpy")) return 1;
  hipLaunchKernelGGL(k_floats, dim3(kBlocks), dim3(kThreads), 0, 0, dev, dev + 1);
  hipLaunchKernelGGL(k_rcp_error, dim3(kBlocks), dim3(kThreads), 0, 0, dev + 2);
  hipLaunchKernelGGL(k_inv_det, dim3(kBlocks), dim3(kThreads), 0, 0, dev + 3);
  if (!ok(hipGetLastError(), "launch")) return 1;
  if (!ok(hipMemcpy(r, dev, sizeof r, hipMemcpyDeviceToHost), "hipMemcpy")) return 1;
  if (!ok(hipFree(dev), "hipFree")) return 1;
  const char* names[4] = {"fast_rcp", "ref_rcp", "rcp_f64", "ref_inv_det"};
  for (int i = 0; i < 4; ++i)
    std::printf("%s checked %llu differ %llu error %.6g\n", names[i], r[i].checked, r[i].differ,
                __builtin_bit_cast(double, r[i].error));
  return 0;
}
