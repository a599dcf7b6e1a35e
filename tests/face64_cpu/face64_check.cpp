// The FP64 production forms of the cada3 and WENO5 face states and of the
// roots and reciprocals against the general forms of the same header, on the
// CPU.  Prints the worst error in units of its bound per group; exit status 1
// if one exceeds 1.
#include <cstdio>
#include <limits>
#include <random>

#include "../../amrvac_amd/csrc/fv_device.h"

using namespace fv;

static const double U53 = 0x1p-53;

// cada3 by the general form (cada3_side with IEEE quotients)
static void cada3_general(double rdel, const double* w, double& wL, double& wR) {
  const double eps = 1.4901161193847656e-08;
  const double dm = w[1] - w[0], d0 = w[2] - w[1], dp = w[3] - w[2];
  double l, r;
  cada3_side(dm / (d0 + copysign(eps, d0)), (d0 * d0 + dm * dm) * rdel, l);
  cada3_side(dp / (d0 + copysign(eps, d0)), (dp * dp + d0 * d0) * rdel, r);
  wL = w[1] + 0.5 * (l * d0);
  wR = w[2] - 0.5 * (r * d0);
}

static double scale4(const double* w) { return fabs(w[0]) + fabs(w[1]) + fabs(w[2]) + fabs(w[3]); }

int main() {
  std::mt19937_64 rng(20261203);
  std::uniform_real_distribution<double> U(-1.0, 1.0);
  const double inf = std::numeric_limits<double>::infinity(), nan = std::numeric_limits<double>::quiet_NaN();
  int bad = 0;
  auto report = [&](const char* what, double worst) {
    std::printf("%s: worst / bound %.3f\n", what, worst);
    if (!(worst <= 1.0)) bad = 1;
  };

  // ---- cada3: differences from far below the smoothness radius to far
  // above it, of one sign and of both, some exactly zero.  Bound: each form
  // rounds a dozen times at the size of the cells' values.
  fvc::FVParams fp{};
  const double rad = 0.1 / 64.0;
  for (int d = 0; d < 3; ++d) { fp.rdelinv[d] = 1.0 / (rad * rad); fp.cada3k[d] = 0.5e14 * fp.rdelinv[d]; }
  double worst = 0.0;
  for (int t = 0; t < 400000; ++t) {
    const double base = (t & 3) ? U(rng) : 0.0;
    double d[3];
    for (int k = 0; k < 3; ++k) d[k] = (t >> (2 + k)) % 7 == 0 ? 0.0 : U(rng) * std::pow(10.0, 6.0 * U(rng) - 5.0);
    double w[4] = {base, base + d[0], base + d[0] + d[1], base + d[0] + d[1] + d[2]};
    // the reference's blend between the two forms is 2e-14 wide: outside it
    // both take the same form
    const double dm = w[1] - w[0], d0 = w[2] - w[1], dp = w[3] - w[2];
    if (fabs((d0 * d0 + dm * dm) * fp.rdelinv[0] - 1.0) < 1e-12 || fabs((d0 * d0 + dp * dp) * fp.rdelinv[0] - 1.0) < 1e-12)
      continue;
    double l, r, lg, rg;
    cada3_face64(fp, 0, w[0], w[1], w[2], w[3], l, r);
    cada3_general(fp.rdelinv[0], w, lg, rg);
    const double bound = 32.0 * U53 * scale4(w) + 1e-300;
    worst = fmax(worst, fmax(fabs(l - lg), fabs(r - rg)) / bound);
  }
  report("cada3", worst);

  // ---- inside and at the ends of the blend: eta = 1 + k 1e-15.  There the
  // result moves by |lim - third| over 2e-14 of eta, and eta carries the
  // rounding of its three operations in each form (4 units of 2^-53 each).
  worst = 0.0;
  for (int k = -40; k <= 40; ++k)
    for (int t = 0; t < 500; ++t) {
      const double a = 3.141592653589793 * U(rng), s = rad * std::sqrt(1.0 + k * 1e-15);
      double w[4] = {0.0, s * std::cos(a), s * std::cos(a) + s * std::sin(a), 0.0};
      w[3] = w[2] + s * std::cos(a) * (t & 1 ? 1.0 : -1.0);
      double l, r, lg, rg;
      cada3_face64(fp, 0, w[0], w[1], w[2], w[3], l, r);
      cada3_general(fp.rdelinv[0], w, lg, rg);
      // both forms lie between third and lim, at most |x| + 2|d0| apart
      const double jump = 1.5 * s;
      const double bound = 0.5e14 * 8.0 * U53 * jump + 32.0 * U53 * scale4(w);
      worst = fmax(worst, fmax(fabs(l - lg), fabs(r - rg)) / bound);
    }
  report("cada3 blend", worst);

  // ---- WENO5 over sizes of the differences, with flat stretches and
  // jumps, beyond the range of the products too.  Bound: candidates and
  // weights round at the size of the cells' values.
  worst = 0.0;
  const double sizes[] = {1e-12, 1e-6, 1e-3, 1.0, 1e6, 1e30, 1e37, 1e45, 1e70};
  for (double sz : sizes)
    for (int t = 0; t < 40000; ++t) {
      double w[6];
      for (int k = 0; k < 6; ++k) w[k] = sz * (U(rng) + (t % 3 == 1 && k >= t % 6 ? 5.0 : 0.0));
      if (t % 5 == 2)
        for (int k = 1; k < 1 + t % 6; ++k) w[k] = w[0];
      double l, r, lg, rg;
      weno5_face64(w[0], w[1], w[2], w[3], w[4], w[5], l, r);
      weno5(w[0], w[1], w[2], w[3], w[4], w[5], lg, rg);
      double m = 0.0;
      for (double v : w) m = fmax(m, fabs(v));
      worst = fmax(worst, fmax(fabs(l - lg), fabs(r - rg)) / (256.0 * U53 * m));
    }
  report("weno5", worst);

  // ---- not finite in, not finite out, as the general forms
  worst = 0.0;
  for (int k = 0; k < 6; ++k)
    for (double v : {inf, -inf, nan}) {
      double w[6] = {1.0, 1.25, 1.5, 1.0, 0.5, 1.0}, l, r, lg, rg;
      w[k] = v;
      weno5_face64(w[0], w[1], w[2], w[3], w[4], w[5], l, r);
      weno5(w[0], w[1], w[2], w[3], w[4], w[5], lg, rg);
      if (std::isnan(l) != std::isnan(lg) || std::isnan(r) != std::isnan(rg)) worst = 2.0;
    }
  for (int k = 0; k < 4; ++k) {
    double w[4] = {1.0, 1.25, 1.5, 1.0}, l, r, lg, rg;
    w[k] = nan;
    cada3_face64(fp, 0, w[0], w[1], w[2], w[3], l, r);
    cada3_general(fp.rdelinv[0], w, lg, rg);
    if (std::isnan(l) != std::isnan(lg) || std::isnan(r) != std::isnan(rg)) worst = 2.0;
  }
  report("not finite", worst);

  // ---- roots and reciprocals: two units in the last place
  worst = 0.0;
  for (int t = 0; t < 200000; ++t) {
    const double a = std::pow(10.0, 60.0 * U(rng));
    double s, i;
    sqrt_rcp(a, s, i);
    worst = fmax(worst, fabs(s / std::sqrt(a) - 1.0) / (4.0 * U53));
    worst = fmax(worst, fabs(i * a - 1.0) / (6.0 * U53));
    worst = fmax(worst, fabs(sqrt_floor(a) / std::sqrt(a) - 1.0) / (4.0 * U53));
  }
  if (!(sqrt_floor(0.0) < 1e-140) || !(sqrt_floor(-1e-20) < 1e-140)) worst = 2.0;
  report("roots", worst);
  return bad;
}
