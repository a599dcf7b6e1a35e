// The FP64 production HLL flux of supersonic faces, on the CPU: the side the
// flow comes from alone gives the flux, also where the other one is infinite.
// Prints the number of faces; exit status 1 at the first that differs.
#include <cstdio>
#include <limits>
#include <random>

#include "../../amrvac_amd/csrc/fv_device.h"

using namespace fv;

static std::mt19937_64 rng(20261207);
static long n = 0;

// P's faces with minmod: cells 0, 1 on one side, 2, 3 on the other, in flow at
// `dir` times eight sound speeds; v: the variable that is infinite in the cell
// behind the face
template <class P, int ID>
static int sides(int boundspeed) {
  std::uniform_real_distribution<double> U(-1.0, 1.0);
  const double inf = std::numeric_limits<double>::infinity();
  fvc::FVParams fp{};
  fp.gamma = 5.0 / 3.0;
  fp.inv_gamma_1 = 1.5;
  fp.gamma_1 = fp.gamma - 1.0;
  fp.tvdlfeps = 1.0;
  fp.boundspeed = boundspeed;
  for (int dir = -1; dir <= 1; dir += 2)
    for (int v : {P::RHO, P::E})
      for (int t = 0; t < 2000; ++t) {
        double st[4][P::NW], flux[2][P::NW];
        for (int c = 0; c < 4; ++c)
          for (int iw = 0; iw < P::NW; ++iw) st[c][iw] = 0.1 * U(rng);
        for (auto& c : st) {
          c[P::RHO] = 1.0 + 0.1 * U(rng);
          c[P::E] = 1.0 + 0.1 * U(rng);
          c[P::MOM + ID] = dir * (10.0 + U(rng));
        }
        // the slope that the used side keeps is the one away from the face
        const int use = dir > 0 ? 1 : 2, out = dir > 0 ? 0 : 3, behind = dir > 0 ? 2 : 1, far = dir > 0 ? 3 : 0;
        st[out][v] = st[use][v] - 1.0e-3;
        st[behind][v] = st[use][v] + 0.5;
        st[far][v] = st[behind][v] + 0.5;
        int crash = 0;
        face_flux<P, double, RIEM_HLL, ID, LIM_MINMOD, 2>(st, fp, 2.0, flux[0], crash);
        st[behind][v] = st[far][v] = inf;
        face_flux<P, double, RIEM_HLL, ID, LIM_MINMOD, 2>(st, fp, 2.0, flux[1], crash);
        // (without GLM the normal field's flux is the speeds' dissipation)
        for (int iw = 0; iw < P::NW; ++iw)
          if (P::MHD && !P::GLM && iw == P::MAG + ID ? !std::isfinite(flux[1][iw]) : !(flux[0][iw] == flux[1][iw])) {
            std::printf("differs: dir %d, infinite %d, flux %d: %a, %a\n", dir, v, iw, flux[0][iw], flux[1][iw]);
            return 1;
          }
        ++n;
      }
  return 0;
}

int main() {
  // the bound speeds from the faster of the two sides (cmaxleftright): the
  // others are not finite with one side
  int bad = sides<Phys<2, 2, false, DIVB_NONE>, 0>(0) + sides<Phys<3, 3, false, DIVB_NONE>, 2>(0);
  bad += sides<Phys<3, 3, true, DIVB_NONE>, 0>(0) + sides<Phys<3, 3, true, DIVB_GLM>, 1>(0);
  std::printf("%ld faces\n", n);
  return bad ? 1 : 0;
}
