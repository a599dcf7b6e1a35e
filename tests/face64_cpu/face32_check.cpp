// cada3_face32 against the limiter's definition in FP32, on the CPU: values
// equal bit for bit (NaN with NaN).  The definition rounds as the FP32 faces
// do: the squares' sum in one multiply-add, 1/d0 as a reciprocal, 1 -+ 1e-14
// as 1.  Exit status 1 at the first difference.
#include <hip/hip_runtime.h>
#include <algorithm>
inline float __builtin_amdgcn_fmed3f(float a, float b, float c) {
  return std::max(std::min(a, b), std::min(std::max(a, b), c));
}
#include <cstdio>
#include <cstring>
#include <limits>
#include <random>

#include "../../amrvac_amd/csrc/fv_device.h"

using namespace fv;

static float side(float th, float eta) {
  const float A = (2.0f + th) * float(1.0 / 3.0);
  if (eta <= 1.0f) return A;
  const float lim = fmax(0.0f, fmin(A, fmax(-0.5f * th, fmin(fmin(2.0f * th, A), 1.6f))));
  if (eta >= 1.0f) return lim;
  return eta + A;  // NaN
}

static float threshold(float r) {
  float s = 1.0f / r;
  while (s * r > 1.0f) s = std::nextafterf(s, 0.0f);
  while (std::nextafterf(s, HUGE_VALF) * r <= 1.0f) s = std::nextafterf(s, HUGE_VALF);
  return s;
}

int main() {
  std::mt19937_64 rng(20261205);
  std::uniform_real_distribution<float> U(-1.0f, 1.0f);
  const float inf = std::numeric_limits<float>::infinity(), nan = std::numeric_limits<float>::quiet_NaN();
  long n = 0;
  for (int m = 0; m < 4; ++m) {
    fvc::FVParams fp{};
    const double rad = 0.1 / (37.0 * (1 << (3 * m)));
    fp.rdelinv[0] = 1.0 / (rad * rad);
    fp.cada3t[0] = threshold((float)fp.rdelinv[0]);
    const float rdel = (float)fp.rdelinv[0], sr = std::sqrt(1.0f / rdel);
    for (int t = 0; t < 400000; ++t) {
      float w[4];
      w[1] = (t & 3) ? U(rng) : 0.0f;
      float d[3];
      for (int k = 0; k < 3; ++k) {
        d[k] = U(rng) * std::pow(10.0f, 6.0f * U(rng) - 5.0f);
        if ((t >> (2 + k)) % 7 == 0) d[k] = 0.0f;
        if ((t >> (3 + k)) % 5 == 0) d[k] = U(rng) * 1.5f * sr;  // about the smoothness radius
      }
      w[0] = w[1] - d[0];
      w[2] = w[1] + d[1];
      w[3] = w[2] + d[2];
      if (t % 997 == 0) w[(t / 997) % 4] = inf;
      if (t % 997 == 1) w[(t / 997) % 4] = -inf;
      if (t % 997 == 2) w[(t / 997) % 4] = nan;
      const float dm = w[1] - w[0], d0 = w[2] - w[1], dp = w[3] - w[2];
      const float inv = 1.0f / (d0 + copysign(1.4901161193847656e-08f, d0));
      const float gl = fma(0.5f, side(dm * inv, fma(dm, dm, d0 * d0) * rdel) * d0, w[1]);
      const float gr = fma(-0.5f, side(dp * inv, fma(dp, dp, d0 * d0) * rdel) * d0, w[2]);
      float l, r;
      cada3_face32<float>(fp, 0, w[0], w[1], w[2], w[3], l, r);
      auto same = [](float a, float b) { return a == b || (a != a && b != b); };
      if (!same(l, gl) || !same(r, gr)) {
        std::printf("differs: %a %a %a %a: %a %a, expected %a %a\n", w[0], w[1], w[2], w[3], l, r, gl, gr);
        return 1;
      }
      ++n;
    }
  }
  std::printf("%ld faces equal\n", n);
  return 0;
}
