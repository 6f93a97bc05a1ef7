// The exact instance's short forms on the host -- TEST HARNESS (built and run by tests/test_exact_forms_cpu.py).
//
// Instantiates p2r-tests_amd/csrc/p2r_lane_math.inc as p2r::exact does (contraction off; a wavefront of one lane; host
// values in place of the hardware estimates) and prints
//   "ulps <sin> <cos>": the largest error of s_sincos64 against long double in ulps of the FP64 result, over every STEP-th
//       float of 0 .. 2^12 and the floats nearest to multiples of pi/2;
//   "words <n>": of the same arguments and their negatives, those where a result that s_sincos is sure of is not the
//       rounding of the long double one;
//   "remainder <r>": the largest |r| - pi/4 there;
//   then per kind of track "<name> <short> <general> <library>": the square roots taken by the short and by the general form
//       and the library sine/cosine calls of one propagation.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <initializer_list>

#define __device__
#define __forceinline__ inline

#include "../p2r-tests_amd/csrc/p2r_types.hpp"

namespace {
int g_short = 0, g_general = 0, g_library = 0;
float counted_sqrt(float x) {
  ++g_general;
  return std::sqrt(x);
}
void counted_sincos(double x, double* s, double* c) {
  ++g_library;
  *s = std::sin(x);
  *c = std::cos(x);
}
}  // namespace

namespace ex {
inline float rcp_prio(float x) { return 1.0f / x; }
inline double rcp_prio(double x) { return 1.0 / x; }
inline float rsq_prio(float x) {
  ++g_short;
  return 1.0f / std::sqrt(x);
}
inline void opaque(float&) {}
inline void phase_boundary() {}
inline bool any_lane(bool v) { return v; }
using real = float;
using Trk = p2r::TrkT<real>;
using Hit = p2r::HitT<real>;
using Jac = p2r::JacT<real>;
using p2r::kNiter;
using p2r::sym;
#define P2R_EXACT 1
#define P2R_DOUBLE 0
#define sqrtf(x) counted_sqrt(x)
#define sincos(x, s, c) counted_sincos(x, s, c)
#define __builtin_amdgcn_div_fixup(y, b, a) ((a) / (b))
#include "../p2r-tests_amd/csrc/p2r_lane_math.inc"
#undef sqrtf
#undef sincos
#undef P2R_EXACT
#undef P2R_DOUBLE
}  // namespace ex

int main(int argc, char** argv) {
  using namespace ex;
  if (argc < 2) return 1;
  const uint32_t step = (uint32_t)std::atol(argv[1]);
  long double e_sin = 0, e_cos = 0, excess = -1;
  long wrong = 0;
  auto ulps = [](double got, long double want) {
    return std::fabs((long double)got - want) / std::ldexp(1.0L, std::ilogb(want) - 52);
  };
  auto check = [&](float x) {
    double sr, cr;
    uint32_t q;
    s_sincos64(x, sr, cr, q);
    // pi/2 = its first 46 bits, whose product with n and difference from x are exact, and the rest
    const long double n = (long double)(int32_t)(q - 0x4b400000u);
    const long double r = ((long double)x - n * 0x1.921fb54442dp+0L) - n * 5.3903028581581189681104586997606911e-15L;
    if (std::fabs(r) - 0.785398163397448309616L > excess) excess = std::fabs(r) - 0.785398163397448309616L;
    const long double s = std::sin(r), c = std::cos(r);
    if (r != 0) e_sin = std::fmax(e_sin, ulps(sr, s));
    e_cos = std::fmax(e_cos, ulps(cr, c));
    for (float v : {x, -x}) {
      float gs, gc;
      uint32_t unsure = ~0u;
      s_sincos(v, gs, gc, unsure);
      if (unsure < 2u * kUnsure) continue;
      long double ws = (q & 1) ? c : s, wc = (q & 1) ? s : c;
      if (q & 2) ws = -ws;
      if ((q + 1) & 2) wc = -wc;
      if (std::signbit(v) != std::signbit(x)) ws = -ws;
      const float fs = (float)ws, fc = (float)wc;
      wrong += std::memcmp(&gs, &fs, 4) != 0 || std::memcmp(&gc, &fc, 4) != 0;
    }
  };
  for (uint32_t b = 0; b <= 0x45800000u; b += step) {
    float x;
    std::memcpy(&x, &b, 4);
    check(x);
  }
  for (int k = 1; k <= 2607; ++k) {
    const float x = (float)(k * 1.5707963267948966);
    check(x);
    check(std::nextafter(x, 0.f));
    check(std::nextafter(x, 1e9f));
  }
  std::printf("ulps %.1Lf %.1Lf\nwords %ld\nremainder %.2Le\n", e_sin, e_cos, wrong, excess);

  auto propagate = [&](const char* name, int field, uint32_t bits) {
    Trk t, o;
    const float par[6] = {-12.8068466f, -7.7238250f, 38.1301422f, 0.2373203f, -2.6133728f, 0.3559412f};
    for (int i = 0; i < 6; ++i) t.par[i] = par[i];
    for (int i = 0; i < 21; ++i) t.cov[i] = 1e-4f;
    if (field >= 0) std::memcpy(&t.par[field], &bits, 4);
    g_short = g_general = g_library = 0;
    propagate_to_r(t, -87.5f, -17.f, -10.5f, o);
    std::printf("%s %d %d %d\n", name, g_short, g_general, g_library);
  };
  propagate("ordinary", -1, 0);
  propagate("x=0", 0, 0);
  propagate("y=-0", 1, 0x80000000u);
  propagate("x=2^13", 0, 0x46000000u);
  propagate("ipt=0", 3, 0);
  propagate("ipt=NaN", 3, 0x7fc00000u);
  propagate("phi=0", 4, 0);
  propagate("phi=-0", 4, 0x80000000u);
  propagate("phi=8192", 4, 0x46000000u);
  propagate("phi=NaN", 4, 0x7fc00000u);
  propagate("phi=unsure", 4, 0xc0259f7cu);
  propagate("theta=unsure", 5, 0x40096e02u);
  propagate("theta=0", 5, 0);
  return 0;
}
