// Device-side comparisons for the GPU tests: functions of the library's kernels against the
// general forms that they stand for, and kernel forms that only very large jobs take.
#include <cstdint>

#include "mbir_host.h"
#include "mbir_selector.h"

using namespace mbir;

namespace {

__device__ inline uint32_t hash(uint64_t& s)  // splitmix64
{
  uint64_t z = (s += 0x9e3779b97f4a7c15ull);
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return (uint32_t)((z ^ (z >> 31)) >> 16);
}
// 2^e with e uniform in [lo, hi), times a random mantissa in [1, 2)
__device__ inline float draw(uint64_t& s, int lo, int hi)
{
  const uint32_t m = hash(s) & 0x7fffffu;
  const int e = lo + (int)(hash(s) % (uint32_t)(hi - lo));
  return ldexpf(__uint_as_float(0x3f800000u | m), e);
}

// every mantissa at every exponent of the range
__global__ void k_roots(unsigned long long* out)
{
  unsigned long long n = 0, bad = 0;
  for (uint32_t m = blockIdx.x * blockDim.x + threadIdx.x; m < (1u << 23); m += gridDim.x * blockDim.x)
    for (int e = -50; e < 50; ++e) {
      const float a = __uint_as_float((uint32_t)(127 + e) << 23 | m);
      if (!(a > kRejectLo && a < kRejectHi)) continue;
      ++n;
      bad += root_short(a) != sqrtf(a);
    }
  atomicAdd(out, n);
  atomicAdd(out + 1, bad);
}

__global__ void k_quotients(uint64_t seed, int per, unsigned long long* out)
{
  uint64_t s = seed + ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) * 0x632be59bd9b4e019ull;
  unsigned long long n = 0, bad = 0;
  for (int i = 0; i < per; ++i) {
    const float a = draw(s, -50, 50), b = draw(s, -50, 50);
    if (!(a > kRejectLo && b > kRejectLo)) continue;
    ++n;
    bad += quotient_short(a, b) != a / b;
  }
  atomicAdd(out, n);
  atomicAdd(out + 1, bad);
}

// Quotients next to the middle of two floats: for an odd d of 24 bits and a small odd r, the
// odd m of 25 bits with m d = r (mod 2^25) gives n = (m d - r) / 2^25, and n / d is m / 2^25
// less r / (2^25 d).
__global__ void k_midpoints(unsigned long long* out)
{
  unsigned long long n = 0, bad = 0;
  for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < (1u << 22); k += gridDim.x * blockDim.x) {
    const uint32_t d = (1u << 23) + 2 * k + 1;
    uint32_t inv = d;  // the inverse modulo 2^32: 3 bits, doubled
    for (int i = 0; i < 5; ++i) inv *= 2u - d * inv;
    for (int r = -15; r <= 15; r += 2) {
      const uint32_t m = ((uint32_t)r * inv) & 0x1ffffffu;
      if (m < (1u << 24)) continue;
      const uint64_t nn = ((uint64_t)m * d - (int64_t)r) >> 25;
      const float a = (float)nn, b = (float)d;
      ++n;
      bad += quotient_short(a, b) != a / b || (uint64_t)a != nn;
    }
  }
  atomicAdd(out, n);
  atomicAdd(out + 1, bad);
}

__global__ void k_factors(uint64_t seed, int per, unsigned long long* out)
{
  uint64_t s = seed + ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) * 0x632be59bd9b4e019ull;
  unsigned long long n = 0, bad = 0;
  for (int i = 0; i < per; ++i) {
    const float ea = draw(s, -60, 40), aw = draw(s, -50, 50), dT = draw(s, -49, 50);
    float lo = 1.f, hi = 1.f;
    const float f = rejected_factor(ea, aw, dT, lo, hi);
    if (!(lo > kRejectLo && hi < kRejectHi)) continue;
    ++n;
    bad += f != dT / (ea * sqrtf(aw));
  }
  atomicAdd(out, n);
  atomicAdd(out + 1, bad);
}

// T from 64 units below |e sqrt(w)| to 64 above, or far from it; counted are the entries that
// the square decides
__global__ void k_selector(uint64_t seed, int per, unsigned long long* out)
{
  uint64_t s = seed + ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) * 0x632be59bd9b4e019ull;
  unsigned long long n = 0, bad = 0;
  for (int i = 0; i < per; ++i) {
    const float w = draw(s, -148, 100);
    const float x = draw(s, -49, 70);  // about |e sqrt(w)|
    const float e = (hash(s) & 1 ? 1.f : -1.f) * (x / sqrtf(w));
    const float y = fabsf(e * sqrtf(w));
    const float T = hash(s) & 7 ? __uint_as_float(__float_as_uint(y) + hash(s) % 129 - 64)
                                : draw(s, -49, 70);
    bool near = false;
    const bool kept = kept_by_square(e, w, square_of(T), near);
    if (near) continue;
    ++n;
    bad += kept != kept_by_root(e, w, T);
  }
  atomicAdd(out, n);
  atomicAdd(out + 1, bad);
}

}  // namespace

// out[0] comparisons, out[1] differences; what: 0 roots, 1 quotients, 2 quotients next to the
// middle of two floats, 3 factors, 4 selector
extern "C" int checks_selector(int what, uint64_t seed, int per, unsigned long long* out)
{
  unsigned long long* d = nullptr;
  if (hipMalloc((void**)&d, 2 * sizeof(*d)) != hipSuccess) return -1;
  const dim3 grid(2048), block(256);
  hipError_t r = hipMemset(d, 0, 2 * sizeof(*d));
  if (r == hipSuccess) {
    switch (what) {
      case 0: hipLaunchKernelGGL(k_roots, grid, block, 0, 0, d); break;
      case 1: hipLaunchKernelGGL(k_quotients, grid, block, 0, 0, seed, per, d); break;
      case 2: hipLaunchKernelGGL(k_midpoints, grid, block, 0, 0, d); break;
      case 3: hipLaunchKernelGGL(k_factors, grid, block, 0, 0, seed, per, d); break;
      default: hipLaunchKernelGGL(k_selector, grid, block, 0, 0, seed, per, d); break;
    }
    r = hipGetLastError();
  }
  if (r == hipSuccess) r = hipMemcpy(out, d, 2 * sizeof(*d), hipMemcpyDeviceToHost);
  (void)hipFree(d);
  return r == hipSuccess ? 0 : -1;
}

// The projection of vol by 64-bit line addresses, whatever the volume's size
extern "C" int checks_project_wide(mbir_job* j, const float* vol, double* out)
{
  const size_t M = (size_t)j->g.N_theta * j->g.N_r * j->g.N_t;
  const size_t V = (size_t)j->g.N_z * j->g.N_x * j->g.N_y;
  float* dv = nullptr;
  double* dout = nullptr;
  hipError_t r = hipMalloc((void**)&dv, V * sizeof(float));
  if (r == hipSuccess) r = hipMalloc((void**)&dout, M * sizeof(double));
  if (r == hipSuccess) r = hipMemcpy(dv, vol, V * sizeof(float), hipMemcpyHostToDevice);
  if (r == hipSuccess) r = launch_forward_project(j->J, dv, dout, j->stream, 0);
  if (r == hipSuccess) r = hipStreamSynchronize(j->stream);
  if (r == hipSuccess) r = hipMemcpy(out, dout, M * sizeof(double), hipMemcpyDeviceToHost);
  if (dv) (void)hipFree(dv);
  if (dout) (void)hipFree(dout);
  return r == hipSuccess ? 0 : -1;
}
