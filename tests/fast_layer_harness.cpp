// The fast instance's regrouped layer (p2r_fast_layer.inc) on the host -- TEST HARNESS (built and run by
// tests/test_fast_layer_cpu.py).
//
// Instantiates p2r-tests_amd/csrc/p2r_lane_math.inc and p2r_fast_layer.inc with real = float as p2r::fast does (host
// values in place of the hardware estimates), and the formulas of p2r_lane_math.inc with real = double beside them.
// One layer of an ordinary track, with every input (x, y, z, 1/pt, phi, theta, k, hit x, y, z) and every pair of them
// set to 0, -0, +-infinity and NaN: prints each case in which an output is finite in one of the two and not in the
// other.  Then "max <parameters> <covariance>": the largest difference of the two over N ordinary tracks, in units of
// the propagated state's sigma.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>

#define __device__
#define __forceinline__ inline
#define __builtin_amdgcn_sqrtf(x) std::sqrt(x)
#define __builtin_amdgcn_rcpf(x) (1.0f / (x))

#include "../p2r-tests_amd/csrc/p2r_types.hpp"

namespace fst {
inline double rcp_est(double x) { return 1.0 / x; }
inline float rcp_prio(float x) { return 1.0f / x; }
inline float rsq_prio(float x) { return 1.0f / std::sqrt(std::fabs(x) < 1.17549435e-38f ? 0.0f : x); }  // as v_rsq_f32
inline void opaque(float&) {}
inline void phase_boundary() {}
using real = float;
using Trk = p2r::TrkT<real>;
using Hit = p2r::HitT<real>;
using Jac = p2r::JacT<real>;
using p2r::kNiter;
using p2r::sym;
#define P2R_EXACT 0
#define P2R_DOUBLE 0
#include "../p2r-tests_amd/csrc/p2r_lane_math.inc"
#include "../p2r-tests_amd/csrc/p2r_fast_layer.inc"
#undef P2R_EXACT
#undef P2R_DOUBLE
}  // namespace fst

namespace dbl {
inline void opaque(double&) {}
inline void phase_boundary() {}
using real = double;
using Trk = p2r::TrkT<real>;
using Hit = p2r::HitT<real>;
using Jac = p2r::JacT<real>;
using p2r::kNiter;
using p2r::sym;
#define P2R_EXACT 0
#define P2R_DOUBLE 1
#include "../p2r-tests_amd/csrc/p2r_lane_math.inc"
#undef P2R_EXACT
#undef P2R_DOUBLE
}  // namespace dbl

namespace {
struct Case {
  float in[10] = {-12.8068466f, -7.7238250f, 38.1301422f, 0.2373203f, -2.6133728f, 0.3559412f, -87.5222f, -17.0f, -10.5f, 50.0f};
};
const char* kName[10] = {"x", "y", "z", "ipt", "phi", "theta", "k", "hx", "hy", "hz"};

struct Out {
  double v[28];  // parameters, covariance, chi2
};
void inputs(const Case& c, float par[6], float cov[21]) {
  const float var[6] = {6.3e-7f, 7.5e-7f, 9.6e-8f, 2.5e-3f, 4.1e-4f, 2.3e-4f};
  for (int i = 0; i < 6; ++i) par[i] = c.in[i];
  for (int i = 0; i < 6; ++i)
    for (int j = 0; j <= i; ++j) cov[p2r::sym(i, j)] = (i == j ? 1.0f : 0.1f) * std::sqrt(var[i] * var[j]);
}
template <class T, class H> void track(const Case& c, T& t, H& h) {
  float par[6], cov[21];
  inputs(c, par, cov);
  for (int i = 0; i < 6; ++i) t.par[i] = par[i];
  for (int i = 0; i < 21; ++i) t.cov[i] = cov[i];
  for (int i = 0; i < 3; ++i) h.pos[i] = c.in[7 + i];
  for (int i = 0; i < 6; ++i) h.cov[i] = 0;
  h.cov[0] = h.cov[2] = h.cov[5] = 1e-4f;
}
template <class T> Out result(const T& t, double chi2) {
  Out o;
  for (int i = 0; i < 6; ++i) o.v[i] = t.par[i];
  for (int i = 0; i < 21; ++i) o.v[6 + i] = t.cov[i];
  o.v[27] = chi2;
  return o;
}
Out fast_layer(const Case& c, fst::Trk* prop = nullptr) {
  fst::Trk t, o;
  fst::Hit h;
  track(c, t, h);
  const float rinv = fst::fast_propagate(t.par, t.cov, c.in[6], h.pos[0], h.pos[1], o);
  if (prop) *prop = o;
  const float chi2 = fst::fast_update(o, h, rinv);
  return result(o, chi2);
}
Out dbl_layer(const Case& c, dbl::Trk* prop = nullptr) {
  dbl::Trk t, o;
  dbl::Hit h;
  track(c, t, h);
  dbl::propagate_to_r(t, (double)c.in[6], h.pos[0], h.pos[1], o);
  if (prop) *prop = o;
  const double chi2 = dbl::kalman_update(o, h);
  return result(o, chi2);
}
}  // namespace

int main(int argc, char** argv) {
  if (argc < 2) return 1;
  const float special[] = {0.f, -0.f, INFINITY, -INFINITY, NAN};
  for (int a = 0; a < 10; ++a)
    for (int b = a; b < 10; ++b)
      for (float va : special)
        for (float vb : special) {
          Case c;
          c.in[a] = va;
          if (b != a) c.in[b] = vb;
          const Out f = fast_layer(c), d = dbl_layer(c);
          int differ = 0;
          for (int i = 0; i < 28; ++i) differ += std::isfinite(f.v[i]) != std::isfinite(d.v[i]);
          if (differ) std::printf("%s=%g %s=%g %d outputs\n", kName[a], va, kName[b], b != a ? vb : va, differ);
        }
  const long n = std::atol(argv[1]);
  uint64_t st = 0x2545F4914F6CDD1Dull;
  auto uniform = [&] {
    st ^= st << 13;
    st ^= st >> 7;
    st ^= st << 17;
    return (double)(st >> 11) * 0x1.0p-53;
  };
  double epar = 0, ecov = 0;
  for (long i = 0; i < n; ++i) {
    Case c;
    for (int f = 0; f < 6; ++f) c.in[f] *= (float)(0.9 + 0.2 * uniform());
    if (uniform() < 0.5) c.in[6] = -c.in[6];
    const double r = 17 + 3 * uniform(), phi = std::atan2(c.in[1], c.in[0]) + 0.1 * (uniform() - 0.5);
    c.in[7] = (float)(r * std::cos(phi));
    c.in[8] = (float)(r * std::sin(phi));
    fst::Trk f;
    dbl::Trk d;
    fast_layer(c, &f);
    dbl_layer(c, &d);
    for (int j = 0; j < 6; ++j) {
      epar = std::fmax(epar, std::fabs(f.par[j] - d.par[j]) / std::sqrt(d.cov[p2r::sym(j, j)]));
      for (int l = 0; l <= j; ++l)
        ecov = std::fmax(ecov, std::fabs(f.cov[p2r::sym(j, l)] - d.cov[p2r::sym(j, l)]) /
                                   std::sqrt(d.cov[p2r::sym(j, j)] * d.cov[p2r::sym(l, l)]));
    }
  }
  std::printf("max %.3e %.3e\n", epar, ecov);
  return 0;
}
