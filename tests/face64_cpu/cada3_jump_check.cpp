// The FP64 production form of the cada3 face states beside jumps far larger
// than the cell, against the general form of the same header, on the CPU: each
// side is held to the size of its own cell and slope, not to the jump's.
// Prints the worst error in units of its bound per group; exit status 1 if one
// exceeds 1.
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

int main() {
  std::mt19937_64 rng(20261206);
  std::uniform_real_distribution<double> U(-1.0, 1.0);
  const double inf = std::numeric_limits<double>::infinity();
  int bad = 0;
  auto report = [&](const char* what, double worst) {
    std::printf("%s: worst / bound %.3f\n", what, worst);
    if (!(worst <= 1.0)) bad = 1;
  };
  fvc::FVParams fp{};
  const double rad = 0.1 / 64.0;
  for (int d = 0; d < 3; ++d) { fp.rdelinv[d] = 1.0 / (rad * rad); fp.cada3k[d] = 0.5e14 * fp.rdelinv[d]; }

  // ---- two cells of size 1e-12 .. 1 with a difference up to their own size;
  // the cells beside them 1 .. 1e12 times as large (jumps far above the
  // smoothness radius: the limited form).  Each form rounds a dozen times at
  // the size of the cell and of d0.  The limited states lie between the cells.
  double worst = 0.0, out = 0.0;
  for (int t = 0; t < 400000; ++t) {
    const double s = std::pow(10.0, -6.0 + 6.0 * U(rng));
    double w[4];
    w[1] = s * (1.5 + 0.5 * U(rng));
    w[2] = w[1] + s * U(rng) * std::pow(10.0, -3.0 + 3.0 * U(rng));
    w[0] = w[1] + (t & 1 ? 1.0 : -1.0) * std::pow(10.0, 6.0 + 6.0 * U(rng));
    w[3] = w[2] + (t & 2 ? 1.0 : -1.0) * std::pow(10.0, 6.0 + 6.0 * U(rng));
    const double d0 = w[2] - w[1];
    double l, r, lg, rg;
    cada3_face64(fp, 0, w[0], w[1], w[2], w[3], l, r);
    cada3_general(fp.rdelinv[0], w, lg, rg);
    worst = fmax(worst, fabs(l - lg) / (32.0 * U53 * (fabs(w[1]) + fabs(d0))));
    worst = fmax(worst, fabs(r - rg) / (32.0 * U53 * (fabs(w[2]) + fabs(d0))));
    const double lo = fmin(w[1], w[2]), hi = fmax(w[1], w[2]), tol = 8.0 * U53 * hi;
    out = fmax(out, fmax(fmax(lo - l, l - hi), fmax(lo - r, r - hi)) / tol);
  }
  report("jumps", worst);
  report("between the cells", out);

  // ---- an infinite cell among the four (with its pressure, as the conversion
  // leaves it, or psi alone): what the general form gives, finite where that
  // is finite
  using P = Phys<3, 3, true, DIVB_GLM>;
  worst = 0.0;
  for (int k = 0; k < 4; ++k)
    for (int v = 0; v < P::NW; ++v)
      for (int t = 0; t < 400; ++t) {
        double st[4][P::NW], l[P::NW], r[P::NW];
        for (auto& cell : st)
          for (double& c : cell) c = 1.0 + U(rng);
        st[k][v] = t & 1 ? inf : -inf;
        if (v != P::PSI) st[k][P::E] = t & 2 ? inf : -inf;
        tvd_states<P, double, 0, LIM_CADA3, 1>(st, fp, l, r);
        for (int iw = 0; iw < P::NW; ++iw) {
          const double w[4] = {st[0][iw], st[1][iw], st[2][iw], st[3][iw]};
          double lg, rg;
          cada3_general(fp.rdelinv[0], w, lg, rg);
          if (std::isfinite(l[iw]) != std::isfinite(lg) || std::isfinite(r[iw]) != std::isfinite(rg)) worst = 2.0;
          const double b = 32.0 * U53 * (fabs(w[1]) + fabs(w[2]) + fabs(w[2] - w[1]));
          if (std::isfinite(lg)) worst = fmax(worst, fabs(l[iw] - lg) / b);
          if (std::isfinite(rg)) worst = fmax(worst, fabs(r[iw] - rg) / b);
        }
      }
  report("infinite neighbours", worst);
  return bad;
}
