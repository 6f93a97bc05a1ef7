// Test kernels (not part of the library): the exact instance's short forms of p2r_lane_math.inc against the general ones, by
// exhaustion on the GPU, since they start from hardware estimates.  Built to lib/libp2r_short_forms.so by the Makefile; run by
// tests/test_gpu_short_forms.py.  Each entry point adds its mismatches to counts[0] (device memory, zeroed by the
// caller); counts[1] counts what was compared.
#include <hip/hip_runtime.h>

#include "../p2r-tests_amd/csrc/p2r_lane.hpp"

namespace {
namespace ex = p2r::exact;
constexpr int kBlock = 256, kGrid = 4096;

__device__ uint32_t word(float v) { return __builtin_bit_cast(uint32_t, v); }
__device__ uint64_t word(double v) { return __builtin_bit_cast(uint64_t, v); }
__device__ uint64_t mix(uint64_t x) {  // splitmix64
  x += 0x9e3779b97f4a7c15ull;
  x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ull;
  x = (x ^ (x >> 27)) * 0x94d049bb133111ebull;
  return x ^ (x >> 31);
}
__device__ void add(unsigned long long* counts, unsigned long long bad, unsigned long long all) {
  atomicAdd(&counts[0], bad);
  atomicAdd(&counts[1], all);
}

// Every float with bits in [lo, hi]: which = 0 square root, 1 reciprocal, 2 sine and cosine (of both signs, where sure).
__global__ void floats_kernel(uint32_t lo, uint32_t hi, int which, unsigned long long* counts) {
#pragma clang fp contract(off)
  unsigned long long bad = 0, all = 0;
  for (uint64_t b = lo + (uint64_t)blockIdx.x * kBlock + threadIdx.x; b <= hi; b += (uint64_t)kGrid * kBlock) {
    const float x = __builtin_bit_cast(float, (uint32_t)b);
    if (which == 0) {
      bad += word(ex::s_sqrt(x)) != word(ex::m_sqrt(x));
      ++all;
    } else if (which == 1) {
      bad += word(ex::s_rcp(x)) != word(ex::m_rcp(x));
      ++all;
    } else {
      for (int neg = 0; neg < 2; ++neg) {
        const float v = neg ? -x : x;
        float s, c, ls, lc;
        uint32_t unsure = ~0u;
        ex::s_sincos(v, s, c, unsure);
        if (unsure < 2u * ex::kUnsure) continue;
        ex::m_sincos(v, ls, lc);
        bad += word(s) != word(ls) || word(c) != word(lc);
        ++all;
      }
    }
  }
  add(counts, bad, all);
}

// Every divisor significand, `per` quotients each: half with dividends next to a midpoint between two floats.
__global__ void quotients_kernel(int per, unsigned long long* counts) {
#pragma clang fp contract(off)
  unsigned long long bad = 0, all = 0;
  for (uint32_t m = blockIdx.x * kBlock + threadIdx.x; m < (1u << 23); m += kGrid * kBlock)
    for (int i = 0; i < per; ++i) {
      const uint64_t h = mix((uint64_t)m * per + i);
      // 2^-12 .. 2^12
      const float b = __builtin_bit_cast(float, ((115u + (uint32_t)(h >> 58) % 24u) << 23) | m);
      const float q = __builtin_bit_cast(float, (127u << 23) | ((uint32_t)h & 0x7fffffu));
      float a = __builtin_bit_cast(float, ((103u + (uint32_t)((h >> 48) % 48u)) << 23) | ((uint32_t)(h >> 23) & 0x7fffffu));
      if (i & 1) a = (float)((double)b * ((double)q + 0x1p-24));
      bad += word(ex::s_div(a, b, ex::s_rcp(b))) != word(ex::m_div(a, b));
      ++all;
    }
  add(counts, bad, all);
}

// FP64 reciprocals of products of floats: random significands and exponents of 2^-290 .. 2^250, and the special values.
__global__ void reciprocals64_kernel(uint64_t n, unsigned long long* counts) {
#pragma clang fp contract(off)
  unsigned long long bad = 0, all = 0;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (uint64_t)kGrid * kBlock) {
    const uint64_t h = mix(i);
    uint64_t bits = (h & 0x800fffffffffffffull) | ((733ull + mix(h) % 540ull) << 52);
    if (i < 4) bits = (i & 1 ? 0x8000000000000000ull : 0) | (i & 2 ? 0x7ff0000000000000ull : 0);  // +-0, +-infinity
    const double b = __builtin_bit_cast(double, bits);
    bad += word(ex::m_rcp64(b)) != word(1.0 / b);
    ++all;
  }
  add(counts, bad, all);
}
}  // namespace

extern "C" int short_forms_floats(uint32_t lo, uint32_t hi, int which, unsigned long long* counts, void* stream) {
  if (lo > hi || hi >= 0x7f800000u || which < 0 || which > 2 || !counts) return 1;
  floats_kernel<<<kGrid, kBlock, 0, static_cast<hipStream_t>(stream)>>>(lo, hi, which, counts);
  return hipGetLastError() != hipSuccess;
}
extern "C" int short_forms_quotients(int per, unsigned long long* counts, void* stream) {
  if (per < 1 || per > 4096 || !counts) return 1;
  quotients_kernel<<<kGrid, kBlock, 0, static_cast<hipStream_t>(stream)>>>(per, counts);
  return hipGetLastError() != hipSuccess;
}
extern "C" int short_forms_reciprocals64(uint64_t n, unsigned long long* counts, void* stream) {
  if (n < 1 || n > (1ull << 40) || !counts) return 1;
  reciprocals64_kernel<<<kGrid, kBlock, 0, static_cast<hipStream_t>(stream)>>>(n, counts);
  return hipGetLastError() != hipSuccess;
}
