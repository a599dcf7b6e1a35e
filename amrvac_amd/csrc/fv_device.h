// fv_device.h -- device-side physics, limiters and Riemann solvers of the
// finite-volume block update, templated on the physics (HD / ideal MHD with
// GLM or Linde div B control), the direction of the face (compile-time, so
// every per-variable array stays in registers) and the working precision R
// of reconstruction / fluxes / wave speeds.
//
// Each routine restates the reference routine cited beside it; operand
// order follows the reference's Fortran so that FP64 results agree with the
// reference to rounding.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#ifdef FV_EXACT
#define FV_NS fvx
#else
#define FV_NS fv
#endif

namespace fvc {
// scalar parameters of the scheme (kernel argument, by value)
struct FVParams {
  double gamma, gamma_1, inv_gamma_1;
  double glm_alpha;
  int glm_extended;
  double divbdiff;
  int limiter;
  int boundspeed;
  double tvdlfeps;
  double small_pressure, small_density;
  int check_small;
  int fix_small;       // fix_small_values (small_values_method 'error')
  double dx[3];
  double dxinv[3];     // 1/dx
  double rdelinv[3];   // 1/(cada3_radius*dx)^2, src/limiter/mod_limiter.t:254
  double cada3k[3];    // 1e14/2 times rdelinv: the slope of cada3's blend
  double cada3t[3];    // the largest FP32 number whose FP32 product with rdelinv is at most 1
  double invds2;       // sum_d 1/dx_d^2 (Linde)
  double mindx;        // minval(dxlevel) (GLM decay)
};

}  // namespace fvc

namespace FV_NS {
using fvc::FVParams;

// Arithmetic helpers.  The contraction-free build (FV_EXACT) keeps IEEE
// division / square root and the reference's MIN/MAX semantics, so that every
// operation rounds like the CPU restatement; the production builds use the
// hardware min/max and, in FP32, the single-instruction reciprocal and square
// root (about 1 ulp).  In FP64 they refine the hardware reciprocal and
// reciprocal square root (about 23 correct bits) by Newton / Goldschmidt
// steps to within an ulp or two, in half the instructions of the IEEE
// sequences; arguments are finite and positive (densities, sound speeds,
// wave-speed spans), or zero for the square root.
#ifdef FV_EXACT
constexpr bool kExact = true;
#else
constexpr bool kExact = false;
#endif

template <class R>
__device__ __forceinline__ R mn2(R a, R b) {
  if constexpr (kExact) return a < b ? a : b;
  else return fmin(a, b);
}
template <class R>
__device__ __forceinline__ R mx2(R a, R b) {
  if constexpr (kExact) return a > b ? a : b;
  else return fmax(a, b);
}
__device__ __forceinline__ double frcp(double a) {
  if constexpr (kExact) {
    return 1.0 / a;
  } else {
    double r = __builtin_amdgcn_rcp(a);
    double e = fma(-a, r, 1.0);  // relative error of r, about 2^-23
    r = fma(r, e, r);            // about 2^-46
    e = fma(-a, r, 1.0);
    return fma(r, e, r);
  }
}
__device__ __forceinline__ float frcp(float a) {
  if constexpr (kExact) return 1.0f / a;
  else return __builtin_amdgcn_rcpf(a);
}
__device__ __forceinline__ double fdiv(double a, double b) {
  if constexpr (kExact) return a / b;
  else return a * frcp(b);
}
__device__ __forceinline__ float fdiv(float a, float b) {
  if constexpr (kExact) return a / b;
  else return a * __builtin_amdgcn_rcpf(b);
}
__device__ __forceinline__ double fsqrt(double a) {
  if constexpr (kExact) {
    return sqrt(a);
  } else {
    // Goldschmidt: g -> sqrt(a), h -> 1/(2 sqrt(a)) from y = rsq(a)
    const double y = __builtin_amdgcn_rsq(a);
    double g = a * y, h = 0.5 * y;
    const double r = fma(-g, h, 0.5);
    g = fma(g, r, g);
    h = fma(h, r, h);
    const double d = fma(-g, g, a);
    g = fma(d, h, g);
    return a == 0.0 ? 0.0 : g;
  }
}
__device__ __forceinline__ float fsqrt(float a) {
  if constexpr (kExact) return sqrtf(a);
  else return __builtin_amdgcn_sqrtf(a);
}

// a / b for a divisor whose correctly rounded reciprocal is at hand: the
// remainder of the rounded product corrects it to the correctly rounded
// quotient (P. Markstein, IBM J. Res. Dev. 34, 1990), in 3 operations instead
// of the 11 of the IEEE sequence
__device__ __forceinline__ double div_by(double a, double b, double binv) {
  if constexpr (kExact) {
    return a / b;
  } else {
    const double q = a * binv;
    return fma(fma(-q, b, a), binv, q);
  }
}

// FP64 production arithmetic: the forms below that round differently from the
// reference's expressions (by an ulp or two) are taken by these kernels only;
// the bit-reproducible build and the FP32 faces keep the plain expressions.
template <class R>
constexpr bool kFast64 = !kExact && std::is_same<R, double>::value;

// sqrt(a) and 1/a of a positive a from one reciprocal square root, refined by
// Goldschmidt's iteration (g -> sqrt(a), h -> 1/(2 sqrt(a))) and a Newton step
// on 1/a: both within an ulp or two, in 15 issue slots instead of the 23 of fsqrt
// and frcp.
__device__ __forceinline__ void sqrt_rcp(double a, double& s, double& inv) {
  const double y = __builtin_amdgcn_rsq(a);
  double g = a * y, h = 0.5 * y;
  const double r = fma(-g, h, 0.5);
  g = fma(g, r, g);
  h = fma(h, r, h);
  s = fma(fma(-g, g, a), h, g);
  const double t = h + h;
  const double i = t * t;
  inv = fma(i, fma(-a, i, 1.0), i);
}
// sqrt of max(a, 1e-300), by the same iteration: the root of a difference that
// rounding may have made zero or negative; no test for zero (the root is then
// 1e-150)
__device__ __forceinline__ double sqrt_floor(double a) {
  a = fmax(a, 1.0e-300);
  const double y = __builtin_amdgcn_rsq(a);
  double g = a * y, h = 0.5 * y;
  const double r = fma(-g, h, 0.5);
  g = fma(g, r, g);
  h = fma(h, r, h);
  return fma(fma(-g, g, a), h, g);
}

// ---------------------------------------------------------------------------
// physics traits: variable indices as in hd_phys_init / mhd_phys_init
// (rho_, mom(:), e_, mag(:), psi_; src/hd/mod_hd_phys.t:217-228,
// src/mhd/mod_mhd_phys.t:478-503)
// ---------------------------------------------------------------------------
enum { DIVB_NONE = 0, DIVB_GLM = 1, DIVB_LINDE = 4 };
enum { RIEM_HLL = 1, RIEM_HLLC = 2, RIEM_HLLD = 3, RIEM_TVDLF = 5, RIEM_HANCOCK = 8 };
enum {
  LIM_MINMOD = 1, LIM_WOODWARD = 2, LIM_MCBETA = 3, LIM_SUPERBEE = 4,
  LIM_VANLEER = 5, LIM_ALBADA = 6, LIM_KOREN = 7, LIM_CADA = 8, LIM_CADA3 = 9, LIM_WENO5 = 16
};

template <int NDIM_, int NDIR_, bool MHD_, int DIVB_>
struct Phys {
  static constexpr int NDIM = NDIM_;
  static constexpr int NDIR = NDIR_;
  static constexpr bool MHD = MHD_;
  static constexpr bool GLM = MHD_ && DIVB_ == DIVB_GLM;
  static constexpr bool LINDE = MHD_ && DIVB_ == DIVB_LINDE;
  static constexpr int RHO = 0;
  static constexpr int MOM = 1;
  static constexpr int E = NDIR_ + 1;
  static constexpr int MAG = NDIR_ + 2;
  static constexpr int PSI = 2 * NDIR_ + 2;
  static constexpr int NW = MHD_ ? (2 * NDIR_ + 2 + (GLM ? 1 : 0)) : (NDIR_ + 2);
};

// ---------------------------------------------------------------------------
// conversions
// ---------------------------------------------------------------------------

// v1^2 + v2^2 (+ v3^2).  Which of the first two products the multiply-add takes
// in is written out: left to the compiler it is chosen for each place a
// conversion is inlined at, so that a cell and its copy in a neighbour's halo
// would get pressures that differ in the last bit.
template <int N>
__device__ __forceinline__ double sum_sq(const double* v) {
  if constexpr (kExact) {
    double s = v[0] * v[0];
#pragma unroll
    for (int d = 1; d < N; ++d) s = s + v[d] * v[d];
    return s;
  } else {
    double s = fma(v[0], v[0], v[1] * v[1]);
#pragma unroll
    for (int d = 2; d < N; ++d) s = fma(v[d], v[d], s);
    return s;
  }
}

// hd_to_primitive src/hd/mod_hd_phys.t:703-734,
// mhd_to_primitive_origin src/mhd/mod_mhd_phys.t:1741-1765 (always FP64:
// the pressure recovery from total energy cancels at low beta)
template <class P>
__device__ __forceinline__ void to_prim(const double* c, double* w, const FVParams& fp) {
#pragma unroll
  for (int iw = 0; iw < P::NW; ++iw) w[iw] = c[iw];
  const double inv_rho = 1.0 / w[P::RHO];
#pragma unroll
  for (int d = 0; d < P::NDIR; ++d) w[P::MOM + d] = w[P::MOM + d] * inv_rho;
  const double vsq = sum_sq<P::NDIR>(w + P::MOM);
  if constexpr (!P::MHD) {
    w[P::E] = (fp.gamma - 1.0) * (w[P::E] - 0.5 * w[P::RHO] * vsq);
  } else {
    const double bsq = sum_sq<P::NDIR>(w + P::MAG);
    w[P::E] = fp.gamma_1 * (w[P::E] - 0.5 * (w[P::RHO] * vsq + bsq));
  }
}

// phys_check_w on a conserved FP64 cell (hd_check_w src/hd/mod_hd_phys.t:
// 648-674, mhd_check_w_origin src/mhd/mod_mhd_phys.t:1452-1473 with small_e
// = small_pressure/(gamma-1)).  With fix_small_values and the default
// small_values_method 'error' a flagged cell sets crash
// (src/mod_small_values.t:25-87).
template <class P>
__device__ __forceinline__ bool small_cons(const double* c, const FVParams& fp) {
  if (c[P::RHO] < fp.small_density) return true;
  double msq = c[P::MOM] * c[P::MOM];
#pragma unroll
  for (int d = 1; d < P::NDIR; ++d) msq = msq + c[P::MOM + d] * c[P::MOM + d];
  if constexpr (!P::MHD) {
    return (fp.gamma - 1.0) * (c[P::E] - 0.5 * msq / c[P::RHO]) < fp.small_pressure;
  } else {
    double bsq = c[P::MAG] * c[P::MAG];
#pragma unroll
    for (int d = 1; d < P::NDIR; ++d) bsq = bsq + c[P::MAG + d] * c[P::MAG + d];
    return c[P::E] - 0.5 * (msq / c[P::RHO] + bsq) < fp.small_pressure * fp.inv_gamma_1;
  }
}

// hd_to_conserved src/hd/mod_hd_phys.t:677-700,
// mhd_to_conserved_origin src/mhd/mod_mhd_phys.t:1562-1579
// FUSE_P: the pressure's product is the fused one (Fused)
template <class P, class R, bool FUSE_P = false>
__device__ __forceinline__ void to_cons(R* w, R inv_gamma_1) {
  R vsq = w[P::MOM] * w[P::MOM];
#pragma unroll
  for (int d = 1; d < P::NDIR; ++d) vsq = vsq + w[P::MOM + d] * w[P::MOM + d];
  if constexpr (!P::MHD) {
    w[P::E] = w[P::E] * inv_gamma_1 + R(0.5) * vsq * w[P::RHO];
  } else {
    R bsq = w[P::MAG] * w[P::MAG];
#pragma unroll
    for (int d = 1; d < P::NDIR; ++d) bsq = bsq + w[P::MAG + d] * w[P::MAG + d];
    if constexpr (FUSE_P) {
      w[P::E] = fma(w[P::E], inv_gamma_1, R(0.5) * (vsq * w[P::RHO] + bsq));
    } else {
      w[P::E] = w[P::E] * inv_gamma_1 + R(0.5) * (vsq * w[P::RHO] + bsq);
    }
  }
#pragma unroll
  for (int d = 0; d < P::NDIR; ++d) w[P::MOM + d] = w[P::RHO] * w[P::MOM + d];
}

// hd_get_flux src/hd/mod_hd_phys.t:1097-1146,
// mhd_get_flux src/mhd/mod_mhd_phys.t:3810-3889 (GLM :3868-3874)
// PIN_BN: in b.v the normal field's product is not the fused one (Fused)
template <class P, class R, int ID, bool PIN_BN = false>
__device__ __forceinline__ void phys_flux(const R* wC, const R* w, R ch, R* f) {
  const R vn = w[P::MOM + ID];
  if constexpr (!P::MHD) {
    f[P::RHO] = vn * w[P::RHO];
#pragma unroll
    for (int d = 0; d < P::NDIR; ++d) f[P::MOM + d] = vn * wC[P::MOM + d];
    f[P::MOM + ID] = f[P::MOM + ID] + w[P::E];
    f[P::E] = vn * (wC[P::E] + w[P::E]);
  } else {
    const R bn = w[P::MAG + ID];
    f[P::RHO] = vn * w[P::RHO];
#pragma unroll
    for (int d = 0; d < P::NDIR; ++d) f[P::MOM + d] = wC[P::MOM + ID] * w[P::MOM + d] - bn * w[P::MAG + d];
    R bsq = w[P::MAG] * w[P::MAG];
#pragma unroll
    for (int d = 1; d < P::NDIR; ++d) bsq = bsq + w[P::MAG + d] * w[P::MAG + d];
    const R ptotal = w[P::E] + R(0.5) * bsq;
    f[P::MOM + ID] = f[P::MOM + ID] + ptotal;
    R bv = w[P::MAG] * w[P::MOM];
    if constexpr (PIN_BN && ID < 2) {
      constexpr int O = 1 - ID;
      bv = fma(w[P::MAG + O], w[P::MOM + O], bn * vn);
#pragma unroll
      for (int d = 2; d < P::NDIR; ++d) bv = fma(w[P::MAG + d], w[P::MOM + d], bv);
    } else {
#pragma unroll
      for (int d = 1; d < P::NDIR; ++d) bv = bv + w[P::MAG + d] * w[P::MOM + d];
    }
    f[P::E] = vn * (wC[P::E] + ptotal) - bn * bv;
#pragma unroll
    for (int d = 0; d < P::NDIR; ++d) f[P::MAG + d] = vn * w[P::MAG + d] - bn * w[P::MOM + d];
    if constexpr (P::GLM) {
      f[P::MAG + ID] = w[P::PSI];
      f[P::PSI] = ch * ch * w[P::MAG + ID];
    }
  }
}

// mhd_get_csound_prim src/mhd/mod_mhd_phys.t:3329-3379 (no B0, no Hall)
template <class P, class R, int ID>
__device__ __forceinline__ R fast_speed(const R* w, R gamma) {
  const R inv_rho = frcp(w[P::RHO]);
  const R cs = gamma * w[P::E] * inv_rho;
  R b2 = w[P::MAG] * w[P::MAG];
#pragma unroll
  for (int d = 1; d < P::NDIR; ++d) b2 = b2 + w[P::MAG + d] * w[P::MAG + d];
  const R cfast2 = b2 * inv_rho + cs;
  const R bn = w[P::MAG + ID];
  R av = cfast2 * cfast2 - R(4) * cs * (bn * bn) * inv_rho;
  if (av < R(0)) av = R(0);
  return fsqrt(R(0.5) * (cfast2 + fsqrt(av)));
}

// hd_get_cbounds src/hd/mod_hd_phys.t:891-1001,
// mhd_get_cbounds src/mhd/mod_mhd_phys.t:3037-3127
template <class P, class R, int ID, bool WANT_CMIN, bool PIN = false>
__device__ __forceinline__ void cbounds(const R* wLC, const R* wRC, const R* wLp, const R* wRp,
                                        const FVParams& fp, R& cmax, R& cmin, int& crash) {
  const R g = R(fp.gamma);
  constexpr int MN = P::MOM + ID;
  if constexpr (kFast64<R>) {
    if (fp.boundspeed == 1) {
      // Einfeldt with the squared speeds it needs (no root of the fast speed)
      // and each side's sqrt(rho) and 1/rho from one reciprocal square root
      auto c2 = [&](const R* w, R inv_rho) {
        const R cs = g * w[P::E] * inv_rho;
        if constexpr (!P::MHD) {
          return cs;
        } else {
          R b2 = w[P::MAG] * w[P::MAG];
#pragma unroll
          for (int d = 1; d < P::NDIR; ++d) b2 = b2 + w[P::MAG + d] * w[P::MAG + d];
          const R cf2 = b2 * inv_rho + cs;
          const R bn = w[P::MAG + ID];
          return R(0.5) * (cf2 + sqrt_floor(cf2 * cf2 - R(4) * cs * (bn * bn) * inv_rho));
        }
      };
      R sL, sR, iL, iR;
      sqrt_rcp(wLp[P::RHO], sL, iL);
      sqrt_rcp(wRp[P::RHO], sR, iR);
      const R t = frcp(sL + sR);
      const R umean = (wLp[MN] * sL + wRp[MN] * sR) * t;
      const R dv = (wRp[MN] - wLp[MN]) * t;
      const R dmean = fsqrt((sL * c2(wLp, iL) + sR * c2(wRp, iR)) * t + R(0.5) * sL * sR * (dv * dv));
      if constexpr (WANT_CMIN) {
        cmin = umean - dmean;
        cmax = umean + dmean;
      } else {
        cmax = fabs(umean) + dmean;
      }
      return;
    }
  }
  if constexpr (!P::MHD) {
    if (fp.boundspeed == 1) {
      const R tmp1 = fsqrt(wLp[P::RHO]);
      const R tmp2 = fsqrt(wRp[P::RHO]);
      const R tmp3 = frcp(tmp1 + tmp2);
      const R umean = (wLp[MN] * tmp1 + wRp[MN] * tmp2) * tmp3;
      const R csL = fdiv(g * wLp[P::E], wLp[P::RHO]);
      const R csR = fdiv(g * wRp[P::E], wRp[P::RHO]);
      const R dv = wRp[MN] - wLp[MN];
      R dmean = (tmp1 * csL + tmp2 * csR) * tmp3 + R(0.5) * tmp1 * tmp2 * (tmp3 * tmp3) * (dv * dv);
      dmean = fsqrt(dmean);
      if constexpr (WANT_CMIN) {
        cmin = umean - dmean;
        cmax = umean + dmean;
      } else {
        cmax = fabs(umean) + dmean;
      }
    } else if (fp.boundspeed == 2) {
      // conserved mean, hd_get_csound2 -> hd_get_pthermal (:1021-1064)
      const R rho = R(0.5) * (wLC[P::RHO] + wRC[P::RHO]);
      const R mn = R(0.5) * (wLC[MN] + wRC[MN]);
      R msq = R(0);
#pragma unroll
      for (int d = 0; d < P::NDIR; ++d) {
        const R m = R(0.5) * (wLC[P::MOM + d] + wRC[P::MOM + d]);
        msq = msq + m * m;
      }
      const R e = R(0.5) * (wLC[P::E] + wRC[P::E]);
      const R tmp1 = fdiv(mn, rho);
      R pth = (g - R(1)) * (e - fdiv(R(0.5) * msq, rho));
      if (fp.fix_small) {
        if (pth < R(fp.small_pressure)) pth = R(fp.small_pressure);
      } else if (fp.check_small && pth < R(fp.small_pressure)) {
        crash = 1;
      }
      const R cs = fsqrt(fdiv(g * pth, rho));
      if constexpr (WANT_CMIN) {
        cmax = mx2(tmp1 + cs, R(0));
        cmin = mn2(tmp1 - cs, R(0));
      } else {
        cmax = fabs(tmp1) + cs;
      }
    } else {
      const R csL = fdiv(g * wLp[P::E], wLp[P::RHO]);
      const R csR = fdiv(g * wRp[P::E], wRp[P::RHO]);
      const R cs = mx2(fsqrt(csL), fsqrt(csR));
      if constexpr (WANT_CMIN) cmin = mn2(wLp[MN], wRp[MN]) - cs;
      cmax = mx2(wLp[MN], wRp[MN]) + cs;
    }
  } else {
    if (fp.boundspeed == 1) {
      const R csL = fast_speed<P, R, ID>(wLp, g);
      const R csR = fast_speed<P, R, ID>(wRp, g);
      const R tmp1 = fsqrt(wLp[P::RHO]);
      const R tmp2 = fsqrt(wRp[P::RHO]);
      const R tmp3 = frcp(tmp1 + tmp2);
      const R umean = (PIN ? fma(wLp[MN], tmp1, wRp[MN] * tmp2) : wLp[MN] * tmp1 + wRp[MN] * tmp2) * tmp3;
      const R dv = wRp[MN] - wLp[MN];
      const R csq = PIN ? fma(tmp1, csL * csL, tmp2 * (csR * csR)) : tmp1 * (csL * csL) + tmp2 * (csR * csR);
      const R dmean = fsqrt(csq * tmp3 +
                           R(0.5) * tmp1 * tmp2 * (tmp3 * tmp3) * (dv * dv));
      if constexpr (WANT_CMIN) {
        cmin = umean - dmean;
        cmax = umean + dmean;
      } else {
        cmax = fabs(umean) + dmean;
      }
    } else if (fp.boundspeed == 2) {
      R wm[P::NW];
#pragma unroll
      for (int iw = 0; iw < P::NW; ++iw) wm[iw] = R(0.5) * (wLp[iw] + wRp[iw]);
      const R cs = fast_speed<P, R, ID>(wm, g);
      if constexpr (WANT_CMIN) {
        cmax = mx2(wm[MN] + cs, R(0));
        cmin = mn2(wm[MN] - cs, R(0));
      } else {
        cmax = fabs(wm[MN]) + cs;
      }
    } else {
      const R csL = fast_speed<P, R, ID>(wLp, g);
      const R csR = fast_speed<P, R, ID>(wRp, g);
      const R cs = mx2(csL, csR);
      if constexpr (WANT_CMIN) cmin = mn2(wLp[MN], wRp[MN]) - cs;
      cmax = mx2(wLp[MN], wRp[MN]) + cs;
    }
  }
}

// ---------------------------------------------------------------------------
// slope limiters, dwlimiter2 src/limiter/mod_limiter.t:128-334 for one cell:
// a = dwC(i-1), b = dwC(i); gives ldw(i) and rdw(i)
// ---------------------------------------------------------------------------
// the limited third-order slope factor of cada (src/limiter/mod_limiter.t:
// 231-252) for theta = th
template <class R>
__device__ __forceinline__ R cada_limited(R th) {
  const R cadalfa = R(0.5), cadbeta = R(2), cadgamma = R(1.6);
  const R A = (R(2) + th) * R(1.0 / 3.0);
  return mx2(R(0), mn2(A, mx2(-cadalfa * th, mn2(mn2(cadbeta * th, A), cadgamma))));
}

template <class R>
__device__ __forceinline__ void cada3_side(R th, R eta, R& out) {
  const R A = (R(2) + th) * R(1.0 / 3.0);
  const R lim = cada_limited(th);
  if (eta <= R(1) - R(1.0e-14)) {
    out = A;
  } else if (eta >= R(1) + R(1.0e-14)) {
    out = lim;
  } else {
    const R t2 = (eta - R(1)) * R(1.0e14);
    out = R(0.5) * ((R(1) - t2) * A + (R(1) + t2) * lim);
  }
}

template <class R, int LIM>
__device__ __forceinline__ void dwlimiter(int lim_rt, R a, R b, R rdelinv, R& ldw, R& rdw) {
  const int lim = LIM > 0 ? LIM : lim_rt;
  if (lim == LIM_MINMOD) {
    R t = copysign(R(1), b);
    t = t * mx2(R(0), mn2(fabs(b), t * a));
    ldw = t; rdw = t;
  } else if (lim == LIM_VANLEER) {
    const R t = fdiv(R(2) * mx2(a * b, R(0)), b + a + R(1.0e-12));
    ldw = t; rdw = t;
  } else if (lim == LIM_CADA3) {
    const R eps = R(1.4901161193847656e-08);  // sqrt(epsilon(1d0))
    const R eta = (b * b + a * a) * rdelinv;
    R l, r;
    cada3_side(fdiv(a, b + copysign(eps, b)), eta, l);
    cada3_side(fdiv(b, a + copysign(eps, a)), eta, r);
    ldw = l * b;
    rdw = r * a;
  } else if (lim == LIM_CADA) {
    const R eps = R(1.4901161193847656e-08);  // sqrt(epsilon(1d0))
    ldw = cada_limited(fdiv(a, b + copysign(eps, b))) * b;
    rdw = cada_limited(fdiv(b, a + copysign(eps, a))) * a;
  } else if (lim == LIM_KOREN) {
    const R t = copysign(R(1), b);
    const R t2 = mn2(R(2) * fabs(b), R(2) * t * a);
    ldw = t * mx2(R(0), mn2(t2, (a * t + R(2) * fabs(b)) * R(1.0 / 3.0)));
    rdw = t * mx2(R(0), mn2(t2, (R(2) * a * t + fabs(b)) * R(1.0 / 3.0)));
  } else if (lim == LIM_WOODWARD) {
    R t = copysign(R(1), b);
    t = R(2) * t * mx2(R(0), mn2(mn2(fabs(b), t * a), t * R(0.25) * (a + b)));
    ldw = t; rdw = t;
  } else if (lim == LIM_MCBETA) {
    R t = copysign(R(1), b);
    t = t * mx2(R(0), mn2(mn2(R(1.4) * fabs(b), R(1.4) * t * a), t * R(0.5) * (a + b)));
    ldw = t; rdw = t;
  } else if (lim == LIM_SUPERBEE) {
    R t = copysign(R(1), b);
    t = t * mx2(mx2(R(0), mn2(R(2) * fabs(b), t * a)), mn2(fabs(b), R(2) * t * a));
    ldw = t; rdw = t;
  } else {  // albada
    const R t = fdiv(a * (b * b + R(1.0e-12)) + b * (a * a + R(1.0e-12)), b * b + a * a + R(2.0e-12));
    ldw = t; rdw = t;
  }
}

// Limited slopes of one face: ldw(i) from (dwC(i-1), dwC(i)) and rdw(i+1)
// from (dwC(i), dwC(i+1)).  For cada3 both quotients share the denominator
// dwC(i) + sign(eps, dwC(i)); outside the bit-reproducible build it is
// inverted once.
template <class R, int LIM>
__device__ __forceinline__ void face_limit(int lim_rt, R dm, R d0, R dp, R rdelinv, R& ldw, R& rdw) {
  const int lim = LIM > 0 ? LIM : lim_rt;
  if (!kExact && lim == LIM_CADA3) {
    const R eps = R(1.4901161193847656e-08);
    const R inv = frcp(d0 + copysign(eps, d0));
    R l, r;
    cada3_side(dm * inv, (d0 * d0 + dm * dm) * rdelinv, l);
    cada3_side(dp * inv, (dp * dp + d0 * d0) * rdelinv, r);
    ldw = l * d0;
    rdw = r * d0;
    return;
  }
  R r2, l2;
  dwlimiter<R, LIM>(lim_rt, dm, d0, rdelinv, ldw, r2);
  dwlimiter<R, LIM>(lim_rt, d0, dp, rdelinv, l2, rdw);
}

// Both face states of one variable with cada3, FP64 production form.  With
// b = |d0| + eps, X = sign(d0) x and g the limiter times b,
//   phi(x/(d0 + sign(eps, d0))) d0 = (d0/b) g,
//   g = (2b + X)/3  or  max(0, min((2b + X)/3, max(-X/2, min(2X, 1.6b)))),
// so no quotient enters the minima and the face needs 1/b alone.  Every lane
// evaluates both forms: in the flows the limiter is made for most waves hold
// lanes of both kinds, and the minima cost less than the branches around
// them.  The weight f of the limited form, 0 below and 1 above the reference's
// 2e-14-wide blend, is one clamped multiply-add; the blend is f lim + (1 - f)
// third, which at f = 1 is lim itself: lim - third rounds at the size of the
// neighbouring jump, and a small cell beside a shock would take that error.
// The FP64 stage is bound by
// its instruction count (at two waves per SIMD): with the HLL and Einfeldt
// forms below a face takes about 560 instead of 780 VALU instructions and a
// 256^3 MHD-GLM stage 1.69 instead of 2.17 ms.
__device__ __forceinline__ void cada3_face64(const FVParams& fp, int id, double wm, double w0, double w1, double wp,
                                             double& wL, double& wR) {
  const double eps = 1.4901161193847656e-08;  // sqrt(epsilon(1d0))
  const double dm = w0 - wm, d0 = w1 - w0, dp = wp - w1;
  const double b4 = fma(4.0, fabs(d0), 4.0 * eps);  // 4 b
  const double q = d0 * frcp(b4);
  const double t43 = (1.0 / 3.0) * b4, t32 = 0.8 * b4, d2 = d0 * d0;
  const uint64_t sgn = __builtin_bit_cast(uint64_t, d0) & 0x8000000000000000ull;
  // 2 g of one side
  auto side = [&](double x) {
    const double X = __builtin_bit_cast(double, __builtin_bit_cast(uint64_t, x) ^ sgn);
    const double third = fma(2.0 / 3.0, X, t43);
    const double lim = fmax(0.0, fmin(third, fmax(-X, fmin(4.0 * X, t32))));
    const double f = fmin(fmax(fma(fma(x, x, d2), fp.cada3k[id], 0.5 - 0.5e14), 0.0), 1.0);
    return fma(f, lim, fma(-f, third, third));
  };
  wL = fma(side(dm), q, w0);
  wR = fma(-side(dp), q, w1);
}

// The same for FP32 faces, value for value what face_limit gives, without its
// branches: 1 -+ 1e-14 are 1 in FP32, so the blend holds for no number (a NaN
// difference makes A NaN as well), and eta <= 1 exactly where the squares are
// at most fp.cada3t; A <= max(x, A), so the limiter's inner minimum with A
// changes nothing under the outer one; max(0, min(A, y)) with y >= 0 is the
// median; and A, y and the limited value are held twice as large, an exact
// scaling.  12 VALU instructions per side; with branches a limited side took
// 26, 7 of them the blend's with no lane enabled (256^3 MHD-GLM stage, mixed:
// 1148 -> 1101 us).
template <class R>
__device__ __forceinline__ void cada3_face32(const FVParams& fp, int id, R wm, R w0, R w1, R wp, R& wL, R& wR) {
  const R eps = R(1.4901161193847656e-08);  // sqrt(epsilon(1d0))
  const R dm = w0 - wm, d0 = w1 - w0, dp = wp - w1;
  const R inv = frcp(d0 + copysign(eps, d0));
  const R d2 = d0 * d0, t = R(fp.cada3t[id]);
  auto side = [&](R x) {
    const R th = x * inv;
    const R A = (R(2) + th) * R(2.0 / 3.0);
    const R y = fmax(-th, fmin(R(4) * th, R(3.2)));
    const R lim = __builtin_amdgcn_fmed3f(R(0), A, y);
    return fma(x, x, d2) > t ? lim : A;
  };
  wL = fma(R(0.25), side(dm) * d0, w0);
  wR = fma(R(-0.25), side(dp) * d0, w1);
}

// WENO5limiter var=1 src/limiter/mod_weno.t:254-377, one variable, face
// between cells 0 and 1 of the stencil s[-2..3] (passed as s0..s5 =
// w(i-2)..w(i+3))
// PIN: 1 and 2 write out which of two products a multiply-add takes in (Fused)
template <class R, int PIN = 0>
__device__ __forceinline__ void weno5(R wmm, R wm, R w0, R wp, R wpp, R wppp, R& wl, R& wr) {
  const R bc1 = R(1.0833333333333333), bc2 = R(0.25);
  const R d1 = R(1.0 / 10.0), d2 = R(3.0 / 5.0), d3 = R(3.0 / 10.0);
  const R u11 = R(1.0 / 3.0), u12 = R(-7.0 / 6.0), u13 = R(11.0 / 6.0);
  const R u21 = R(-1.0 / 6.0), u22 = R(5.0 / 6.0), u23 = R(1.0 / 3.0);
  const R u31 = R(1.0 / 3.0), u32 = R(5.0 / 6.0), u33 = R(-1.0 / 6.0);
  const R weps = R(1.0e-18);
  {
    const R f1 = u11 * wmm + u12 * wm + u13 * w0;
    const R f2 = PIN == 0   ? u21 * wm + u22 * w0 + u23 * wp
                 : PIN == 1 ? fma(u23, wp, fma(u22, w0, u21 * wm))
                            : fma(u23, wp, fma(u21, wm, u22 * w0));
    const R f3 = PIN == 0 ? u31 * w0 + u32 * wp + u33 * wpp : fma(u33, wpp, fma(u31, w0, u32 * wp));
    R t = wmm + w0 - R(2) * wm, q = wmm - R(4) * wm + R(3) * w0;
    const R b1 = bc1 * (t * t) + bc2 * (q * q);
    t = wm + wp - R(2) * w0; q = wm - wp;
    const R b2 = bc1 * (t * t) + bc2 * (q * q);
    t = w0 + wpp - R(2) * wp; q = R(3) * w0 - R(4) * wp + wpp;
    const R b3 = bc1 * (t * t) + bc2 * (q * q);
    t = b1 + weps; const R t1 = t * t, a1 = fdiv(d1, t1);
    t = b2 + weps; const R t2 = t * t, a2 = fdiv(d2, t2);
    t = b3 + weps; const R t3 = t * t, a3 = fdiv(d3, t3);
    const R as = PIN == 0   ? a1 + a2 + a3
                 : PIN == 1 ? fma(d3, frcp(t3), fma(d2, frcp(t2), a1))
                            : fma(d3, frcp(t3), fma(d1, frcp(t1), a2));
    wl = fdiv(f1 * a1, as) + fdiv(f2 * a2, as) + fdiv(f3 * a3, as);
  }
  {
    const R f1 = u11 * wppp + u12 * wpp + u13 * wp;
    const R f2 = PIN == 0 ? u21 * wpp + u22 * wp + u23 * w0 : fma(u23, w0, fma(u21, wpp, u22 * wp));
    const R f3 = PIN == 0   ? u31 * wp + u32 * w0 + u33 * wm
                 : PIN == 1 ? fma(u33, wm, fma(u32, w0, u31 * wp))
                            : fma(u33, wm, fma(u31, wp, u32 * w0));
    R t = wppp + wp - R(2) * wpp, q = wppp - R(4) * wpp + R(3) * wp;
    const R b1 = bc1 * (t * t) + bc2 * (q * q);
    t = wpp + w0 - R(2) * wp; q = wpp - w0;
    const R b2 = bc1 * (t * t) + bc2 * (q * q);
    t = wp + wm - R(2) * w0; q = R(3) * wp - R(4) * w0 + wm;
    const R b3 = bc1 * (t * t) + bc2 * (q * q);
    t = b1 + weps; const R t1 = t * t, a1 = fdiv(d1, t1);
    t = b2 + weps; const R t2 = t * t, a2 = fdiv(d2, t2);
    t = b3 + weps; const R t3 = t * t, a3 = fdiv(d3, t3);
    const R as = PIN == 0 ? a1 + a2 + a3 : fma(d3, frcp(t3), fma(d2, frcp(t2), a1));
    wr = fdiv(f1 * a1, as) + fdiv(f2 * a2, as) + fdiv(f3 * a3, as);
  }
}

// The same for the FP64 production kernels, in the differences d1..d5 of the
// six cells: the left and right candidates share their second differences,
// and the weights d_k/t_k^2 (t_k = beta_k + eps) are cleared of their
// denominators by the products of the other two, so that one reciprocal per
// side takes the place of six: 85 operations for both sides against 168
// (1040 x 624 MHD-GLM stage: 80 instead of 108 us).
// The products overflow for differences beyond about 1e38 (the quotients hold
// to 1e77): a side that is not finite is evaluated again in quotients.
__device__ __forceinline__ void weno5_face64(double wmm, double wm, double w0, double wp, double wpp, double wppp,
                                             double& wl, double& wr) {
  const double d1 = wm - wmm, d2 = w0 - wm, d3 = wp - w0, d4 = wpp - wp, d5 = wppp - wpp;
  // 4 (beta + 1e-18) = 13/3 s^2 + q^2 + 4e-18
  const double e = 4.0e-18, c = 13.0 / 3.0;
  const double s1 = d2 - d1, s2 = d3 - d2, s3 = d4 - d3, s4 = d5 - d4;
  const double S1 = fma(c * s1, s1, e), S2 = fma(c * s2, s2, e), S3 = fma(c * s3, s3, e), S4 = fma(c * s4, s4, e);
  // 6 (candidate - centre value): the numerators of the ideal weights 1 : 6 : 3
  auto side = [](double t1, double t2, double t3, double g1, double g2, double g3) {
    double a1 = t2 * t3, a2 = t1 * t3, a3 = t1 * t2;
    a1 = a1 * a1;
    a2 = 6.0 * (a2 * a2);
    a3 = 3.0 * (a3 * a3);
    return (a1 * g1 + a2 * g2 + a3 * g3) * frcp(a1 + a2 + a3);
  };
  const double q1 = fma(3.0, d2, -d1), q2 = d2 + d3, q3 = fma(-3.0, d3, d4);
  const double p1 = fma(3.0, d4, -d5), p2 = d3 + d4, p3 = fma(-3.0, d3, d2);
  const double cl = side(fma(q1, q1, S1), fma(q2, q2, S2), fma(q3, q3, S3), fma(5.0, d2, -2.0 * d1), fma(2.0, d3, d2),
                         fma(4.0, d3, -d4));
  const double cr = side(fma(p1, p1, S4), fma(p2, p2, S3), fma(p3, p3, S2), fma(5.0, d4, -2.0 * d5), fma(2.0, d3, d4),
                         fma(4.0, d3, -d2));
  wl = fma(1.0 / 6.0, cl, w0);
  wr = fma(-1.0 / 6.0, cr, wp);
  if (__builtin_expect(!(fabs(cl) + fabs(cr) < 1.0e300), 0)) weno5(wmm, wm, w0, wp, wpp, wppp, wl, wr);
}

// get_Riemann_flux_hlld src/mod_finite_volume.t:505-718 (Miyoshi & Kusano
// 2005 with Guo 2016's star pressure; no B0, no stagger grid, ndir = 3):
// the single-star states w1 across the fast waves, the double-star states w2
// across the Alfven waves, then the region of the fan at the face.  wLp/wRp
// are the primitive states after modify_wLR, wLC/wRC the conserved ones.
template <class P, class R, int ID, bool CT = false>
__device__ __forceinline__ void hlld_flux(const R* wLC, const R* wRC, const R* wLp, const R* wRp, const R* fL,
                                          const R* fR, R sR, R sL, R* fC, R bx_ct = R(0)) {
  static_assert(P::MHD && P::NDIR == 3, "HLLD is provided for MHD with three vector components");
  constexpr int NW = P::NW, RHO = P::RHO, E = P::E, MG = P::MAG, MO = P::MOM;
  constexpr int I2 = (ID + 1) % 3, I3 = (ID + 2) % 3;
  constexpr int M1 = MO + ID, M2 = MO + I2, M3 = MO + I3;
  constexpr int B1 = MG + ID, B2 = MG + I2, B3 = MG + I3;
  // HLL estimate of the normal field (Li 2005 eq. 33); with constrained
  // transport the face field (src/mod_finite_volume.t:536-537)
  R Bx;
  if constexpr (CT) Bx = bx_ct;
  else Bx = fdiv(sR * wRC[B1] - sL * wLC[B1], sR - sL);
  const R ptR = wRp[E] + R(0.5) * (wRC[MG] * wRC[MG] + wRC[MG + 1] * wRC[MG + 1] + wRC[MG + 2] * wRC[MG + 2]);
  const R ptL = wLp[E] + R(0.5) * (wLC[MG] * wLC[MG] + wLC[MG + 1] * wLC[MG + 1] + wLC[MG + 2] * wLC[MG + 2]);
  const R vR = wRp[M1], vL = wLp[M1];
  const R suR = (sR - vR) * wRC[RHO];
  const R suL = (sL - vL) * wLC[RHO];
  const R sm = fdiv(suR * vR - suL * vL - ptR + ptL, suR - suL);
  // single-star states (velocities in the momentum slots until the end)
  R w1R[NW], w1L[NW], w2R[NW], w2L[NW];
  w1R[M1] = sm; w1L[M1] = sm; w2R[M1] = sm; w2L[M1] = sm;
  w1R[B1] = Bx; w1L[B1] = Bx;
  w1R[RHO] = fdiv(suR, sR - sm);
  w1L[RHO] = fdiv(suL, sL - sm);
  R r1R = suR * (sR - sm) - Bx * Bx;
  if (r1R != R(0)) r1R = frcp(r1R);
  R r1L = suL * (sL - sm) - Bx * Bx;
  if (r1L != R(0)) r1L = frcp(r1L);
  w1R[M2] = wRp[M2] - Bx * wRC[B2] * (sm - vR) * r1R;
  w1L[M2] = wLp[M2] - Bx * wLC[B2] * (sm - vL) * r1L;
  const R qR = (suR * (sR - vR) - Bx * Bx) * r1R;
  const R qL = (suL * (sL - vL) - Bx * Bx) * r1L;
  w1R[M3] = wRp[M3] - Bx * wRC[B3] * (sm - vR) * r1R;
  w1L[M3] = wLp[M3] - Bx * wLC[B3] * (sm - vL) * r1L;
  w1R[B3] = wRC[B3] * qR;
  w1L[B3] = wLC[B3] * qL;
  w1R[B2] = wRC[B2] * qR;
  w1L[B2] = wLC[B2] * qL;
  // total pressure of the star region (Guo eq. 25), then the energies
  const R pts = suR * (sm - vR) + ptR;
  {
    const R vbR = wRp[MO] * wRC[MG] + wRp[MO + 1] * wRC[MG + 1] + wRp[MO + 2] * wRC[MG + 2];
    const R vb1R = w1R[MO] * w1R[MG] + w1R[MO + 1] * w1R[MG + 1] + w1R[MO + 2] * w1R[MG + 2];
    w1R[E] = fdiv((sR - vR) * wRC[E] - ptR * vR + pts * sm + Bx * (vbR - vb1R), sR - sm);
    const R vbL = wLp[MO] * wLC[MG] + wLp[MO + 1] * wLC[MG + 1] + wLp[MO + 2] * wLC[MG + 2];
    const R vb1L = w1L[MO] * w1L[MG] + w1L[MO + 1] * w1L[MG + 1] + w1L[MO + 2] * w1L[MG + 2];
    w1L[E] = fdiv((sL - vL) * wLC[E] - ptL * vL + pts * sm + Bx * (vbL - vb1L), sL - sm);
  }
  // double-star states
  w2R[RHO] = w1R[RHO]; w2L[RHO] = w1L[RHO];
  w2R[B1] = Bx; w2L[B1] = Bx;
  const R sR1 = fsqrt(w1R[RHO]);
  const R sL1 = fsqrt(w1L[RHO]);
  const R tmp = frcp(sR1 + sL1);
  const R sgn = copysign(R(1), Bx);
  const R s1R = sm + fdiv(fabs(Bx), sR1);
  const R s1L = sm - fdiv(fabs(Bx), sL1);
  w2R[M2] = (sL1 * w1L[M2] + sR1 * w1R[M2] + (w1R[B2] - w1L[B2]) * sgn) * tmp;
  w2L[M2] = w2R[M2];
  w2R[B2] = (sL1 * w1R[B2] + sR1 * w1L[B2] + sL1 * sR1 * (w1R[M2] - w1L[M2]) * sgn) * tmp;
  w2L[B2] = w2R[B2];
  w2R[M3] = (sL1 * w1L[M3] + sR1 * w1R[M3] + (w1R[B3] - w1L[B3]) * sgn) * tmp;
  w2L[M3] = w2R[M3];
  w2R[B3] = (sL1 * w1R[B3] + sR1 * w1L[B3] + sL1 * sR1 * (w1R[M3] - w1L[M3]) * sgn) * tmp;
  w2L[B3] = w2R[B3];
  {
    const R d1R = w1R[MO] * w1R[MG] + w1R[MO + 1] * w1R[MG + 1] + w1R[MO + 2] * w1R[MG + 2];
    const R d2R = w2R[MO] * w2R[MG] + w2R[MO + 1] * w2R[MG + 1] + w2R[MO + 2] * w2R[MG + 2];
    w2R[E] = w1R[E] + sR1 * (d1R - d2R) * sgn;
    const R d1L = w1L[MO] * w1L[MG] + w1L[MO + 1] * w1L[MG + 1] + w1L[MO + 2] * w1L[MG + 2];
    const R d2L = w2L[MO] * w2L[MG] + w2L[MO + 1] * w2L[MG + 1] + w2L[MO + 2] * w2L[MG + 2];
    w2L[E] = w1L[E] - sL1 * (d1L - d2L) * sgn;
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    w1R[MO + c] = w1R[MO + c] * w1R[RHO];
    w1L[MO + c] = w1L[MO + c] * w1L[RHO];
    w2R[MO + c] = w2R[MO + c] * w2R[RHO];
    w2L[MO + c] = w2L[MO + c] * w2L[RHO];
  }
  // flux_type: GLM's psi and normal B take the known flux
  // (src/mhd/mod_mhd_phys.t:580-586)
#pragma unroll
  for (int iw = 0; iw < NW; ++iw) {
    if (P::GLM && (iw == P::PSI || iw == B1)) {
      fC[iw] = fL[iw];
    } else if (sL > R(0)) {
      fC[iw] = fL[iw];
    } else if (s1L >= R(0)) {
      fC[iw] = fL[iw] + sL * (w1L[iw] - wLC[iw]);
    } else if (sm >= R(0)) {
      fC[iw] = fL[iw] + sL * (w1L[iw] - wLC[iw]) + s1L * (w2L[iw] - w1L[iw]);
    } else if (s1R >= R(0)) {
      fC[iw] = fR[iw] + sR * (w1R[iw] - wRC[iw]) + s1R * (w2R[iw] - w1R[iw]);
    } else if (sR >= R(0)) {
      fC[iw] = fR[iw] + sR * (w1R[iw] - wRC[iw]);
    } else {
      fC[iw] = fR[iw];
    }
  }
}

// Both primitive face states with a TVD limiter; C0: index of cell i in st
template <class P, class R, int ID, int LIM, int C0>
__device__ __forceinline__ void tvd_states(const R (*st)[P::NW], const FVParams& fp, R* wL, R* wR) {
  if constexpr (LIM == LIM_CADA3 && kFast64<R>) {
    // cada3_face64 takes finite outer cells: an infinite one is as good as a
    // very large one, whose side is limited.  One test per face: any infinite
    // variable but psi makes its cell's pressure infinite or NaN, and after a
    // NaN nothing is finite in the general form either.  (256^3 MHD-GLM: this
    // costs 0.8%, a select on f per variable and side 2.6% to 4.6%; 2-D
    // constrained transport 2.4%.)
    R m[P::NW], p[P::NW];
#pragma unroll
    for (int iw = 0; iw < P::NW; ++iw) { m[iw] = st[C0 - 1][iw]; p[iw] = st[C0 + 2][iw]; }
    R far = m[P::E] * p[P::E];
    if constexpr (P::GLM) far = fma(m[P::PSI], p[P::PSI], far);
    if (__builtin_expect(!(fabs(far) < HUGE_VAL), 0)) {
#pragma unroll
      for (int iw = 0; iw < P::NW; ++iw) {
        if (fabs(m[iw]) == HUGE_VAL) m[iw] = copysign(0x1p1020, m[iw]);
        if (fabs(p[iw]) == HUGE_VAL) p[iw] = copysign(0x1p1020, p[iw]);
      }
    }
#pragma unroll
    for (int iw = 0; iw < P::NW; ++iw)
      cada3_face64(fp, ID, m[iw], st[C0][iw], st[C0 + 1][iw], p[iw], wL[iw], wR[iw]);
  } else {
#pragma unroll
    for (int iw = 0; iw < P::NW; ++iw) {
      if constexpr (LIM == LIM_CADA3 && !kExact) {
        cada3_face32(fp, ID, st[C0 - 1][iw], st[C0][iw], st[C0 + 1][iw], st[C0 + 2][iw], wL[iw], wR[iw]);
      } else {
        const R dm = st[C0][iw] - st[C0 - 1][iw];
        const R d0 = st[C0 + 1][iw] - st[C0][iw];
        const R dp = st[C0 + 2][iw] - st[C0 + 1][iw];
        R ldw, rdw;
        face_limit<R, LIM>(LIM, dm, d0, dp, R(fp.rdelinv[ID]), ldw, rdw);
        wL[iw] = st[C0][iw] + R(0.5) * ldw;
        wR[iw] = st[C0 + 1][iw] - R(0.5) * rdw;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// one face: reconstruct_LR (src/mod_finite_volume.t:1110-1228), modify_wLR
// (GLM, src/mhd/mod_mhd_phys.t:6326-6377), fluxes, bounds and the Riemann
// solver (src/mod_finite_volume.t:348-504, src/hd/mod_hd_hllc.t:56-257).
// st[k][iw] are primitive values of cells i-NG+1+k (face between i and i+1,
// NG = 2: st = w(i-1), w(i), w(i+1), w(i+2); NG = 3 adds w(i-2), w(i+3)).
// ---------------------------------------------------------------------------
// Constrained transport: the face's normal field in (the stage input's face
// field, and that of ps for the HLLD star states), the reconstructed
// velocities and signal speeds out for the edge electric fields.
struct CtIO {
  double bn, bx;
  double vL[3], vR[3];
  double cmax, cmin;
};

// Which product of a sum the multiply-adds of the mixed form's FP32 faces take
// in.  The compiler may fuse either, chooses anew for each place a face is
// inlined at, and changes its mind with the code around it.  The rule is that a
// face keeps the value it had before its kernel was rearranged: where the choice
// depends on the surroundings it is written out, and all such places are listed
// here.  An FP32 value that moves by its last bit moves a run by up to 1e-8.
//
// FIRST: the z face below a workgroup's first plane, which the block below
// forms in its march.  For ideal MHD with TVDLF, and with GLM and WENO5, the two
// were never rounded alike (mass_flux, einfeldt, weno): there the fluxes at
// block boundaries in z cancel to FP32 rounding only, and a result depends on
// the blocks' depth to that extent (64 x 64 x 128, 50 steps: the mass moves by
// 3e-13 and 1.4e-12, with the others and in FP64 by 4e-15).  All other faces two
// blocks share are formed alike in both.
template <class P, class R, int ID, int LIM, bool CT, bool FIRST>
struct Fused {
  static constexpr bool F32 = std::is_same<R, float>::value, WENO = LIM == LIM_WENO5;
  // to_cons: the pressure's product
  static constexpr bool pressure = F32 && (CT || LIM == LIM_CADA3);
  // weno5 (all variables but the density): 0 as compiled, 1 and 2 its two forms
  static constexpr int weno = !F32 || P::NDIM != 3 ? 0 : (P::GLM && ID == 2 && !FIRST ? 2 : 1);
  // phys_flux: b.v without the normal field's product
  static constexpr bool normal_field = F32 && CT && P::NDIM == 3 && (LIM == LIM_MINMOD || LIM == LIM_VANLEER);
  // cbounds with TVDLF: the left side's products of Einfeldt's means
  static constexpr bool einfeldt = F32 && FIRST && WENO && !P::GLM;
  // TVDLF: the left side's mass flux
  static constexpr bool mass_flux = F32 && P::MHD && (FIRST || CT) && !(P::GLM && WENO);
};

template <class P, class R, int RIEM, int ID, int LIM, int NG, bool CT = false, bool FIRST = false>
__device__ __forceinline__ void face_flux(const R (*st)[P::NW], const FVParams& fp, R ch, R* fC,
                                          int& crash, CtIO* ctio = nullptr) {
  constexpr int NW = P::NW;
  constexpr int C0 = NG - 1;  // index of cell i in st
  using Fu = Fused<P, R, ID, LIM, CT, FIRST>;
  R wLp[NW], wRp[NW];
  if constexpr (LIM == LIM_WENO5) {
    R tl[NW], tr[NW];
#pragma unroll
    for (int iw = 0; iw < NW; ++iw) {
      wLp[iw] = st[C0][iw];
      wRp[iw] = st[C0 + 1][iw];
      if constexpr (kFast64<R>)
        weno5_face64(st[C0 - 2][iw], st[C0 - 1][iw], st[C0][iw], st[C0 + 1][iw], st[C0 + 2][iw], st[C0 + 3][iw],
                     tl[iw], tr[iw]);
      else if (iw > 0)
        weno5<R, Fu::weno>(st[C0 - 2][iw], st[C0 - 1][iw], st[C0][iw], st[C0 + 1][iw], st[C0 + 2][iw],
                           st[C0 + 3][iw], tl[iw], tr[iw]);
      else
        weno5(st[C0 - 2][iw], st[C0 - 1][iw], st[C0][iw], st[C0 + 1][iw], st[C0 + 2][iw], st[C0 + 3][iw],
              tl[iw], tr[iw]);
    }
    // fix_limiter src/limiter/mod_weno.t:100-133 with hd/mhd check_w
    const bool bad = tl[P::RHO] < R(fp.small_density) || tl[P::E] < R(fp.small_pressure) ||
                     tr[P::RHO] < R(fp.small_density) || tr[P::E] < R(fp.small_pressure);
    if (!bad) {
#pragma unroll
      for (int iw = 0; iw < NW; ++iw) { wLp[iw] = tl[iw]; wRp[iw] = tr[iw]; }
    }
  } else if constexpr (LIM == 0 && std::is_same<R, float>::value) {
#pragma unroll
    for (int iw = 0; iw < NW; ++iw) {
      const R dm = st[C0][iw] - st[C0 - 1][iw];
      const R d0 = st[C0 + 1][iw] - st[C0][iw];
      const R dp = st[C0 + 2][iw] - st[C0 + 1][iw];
      R ldw, rdw;
      face_limit<R, 0>(fp.limiter, dm, d0, dp, R(fp.rdelinv[ID]), ldw, rdw);
      wLp[iw] = st[C0][iw] + R(0.5) * ldw;
      wRp[iw] = st[C0 + 1][iw] - R(0.5) * rdw;
    }
  } else if constexpr (LIM == 0) {
    // the limiter chosen once per face, not per variable and side (3-D MHD, cada3,
    // 3186 blocks of 8^3: 411 -> 290 us)
    switch (fp.limiter) {
      case LIM_MINMOD: tvd_states<P, R, ID, LIM_MINMOD, C0>(st, fp, wLp, wRp); break;
      case LIM_WOODWARD: tvd_states<P, R, ID, LIM_WOODWARD, C0>(st, fp, wLp, wRp); break;
      case LIM_MCBETA: tvd_states<P, R, ID, LIM_MCBETA, C0>(st, fp, wLp, wRp); break;
      case LIM_SUPERBEE: tvd_states<P, R, ID, LIM_SUPERBEE, C0>(st, fp, wLp, wRp); break;
      case LIM_VANLEER: tvd_states<P, R, ID, LIM_VANLEER, C0>(st, fp, wLp, wRp); break;
      case LIM_ALBADA: tvd_states<P, R, ID, LIM_ALBADA, C0>(st, fp, wLp, wRp); break;
      case LIM_KOREN: tvd_states<P, R, ID, LIM_KOREN, C0>(st, fp, wLp, wRp); break;
      case LIM_CADA: tvd_states<P, R, ID, LIM_CADA, C0>(st, fp, wLp, wRp); break;
      default: tvd_states<P, R, ID, LIM_CADA3, C0>(st, fp, wLp, wRp); break;
    }
  } else {
    tvd_states<P, R, ID, LIM, C0>(st, fp, wLp, wRp);
  }
  R wLC[NW], wRC[NW];
  const R inv_g1 = R(fp.inv_gamma_1);
  // modify_wLR replaces the normal field before the FP64 production kernels
  // form the energy; elsewhere its energy is exchanged in the conserved state
  constexpr bool GLM_FIRST = P::GLM && kFast64<R>;
  if constexpr (GLM_FIRST) {
    constexpr int B = P::MAG + ID, S = P::PSI;
    const R dB = wRp[B] - wLp[B];
    const R dPsi = wRp[S] - wLp[S];
    wLp[B] = R(0.5) * (wRp[B] + wLp[B] - fdiv(dPsi, ch));
    wLp[S] = R(0.5) * (wRp[S] + wLp[S] - dB * ch);
    wRp[B] = wLp[B];
    wRp[S] = wLp[S];
  }
#pragma unroll
  for (int iw = 0; iw < NW; ++iw) { wLC[iw] = wLp[iw]; wRC[iw] = wRp[iw]; }
  to_cons<P, R, Fu::pressure>(wLC, inv_g1);
  to_cons<P, R, Fu::pressure>(wRC, inv_g1);
  if constexpr (P::GLM && !GLM_FIRST) {
    constexpr int B = P::MAG + ID, S = P::PSI, E = P::E;
    const R dB = wRp[B] - wLp[B];
    const R dPsi = wRp[S] - wLp[S];
    wLp[B] = R(0.5) * (wRp[B] + wLp[B] - fdiv(dPsi, ch));
    wLp[S] = R(0.5) * (wRp[S] + wLp[S] - dB * ch);
    wRp[B] = wLp[B];
    wRp[S] = wLp[S];
    wRC[E] = wRC[E] - R(0.5) * (wRC[B] * wRC[B]);
    wLC[E] = wLC[E] - R(0.5) * (wLC[B] * wLC[B]);
    wRC[B] = wLp[B]; wRC[S] = wLp[S];
    wLC[B] = wLp[B]; wLC[S] = wLp[S];
    wRC[E] = wRC[E] + R(0.5) * (wRC[B] * wRC[B]);
    wLC[E] = wLC[E] + R(0.5) * (wLC[B] * wLC[B]);
  }
  if constexpr (CT) {
    // mhd_modify_wLR with stagger_grid (src/mhd/mod_mhd_phys.t:6338-6345)
    constexpr int B = P::MAG + ID;
    wLC[B] = R(ctio->bn);
    wRC[B] = wLC[B];
    wLp[B] = wLC[B];
    wRp[B] = wLC[B];
#pragma unroll
    for (int d = 0; d < P::NDIR; ++d) {
      ctio->vL[d] = wLp[P::MOM + d];
      ctio->vR[d] = wRp[P::MOM + d];
    }
  }
  R fL[NW], fR[NW];
  phys_flux<P, R, ID, Fu::normal_field>(wLC, wLp, ch, fL);
  phys_flux<P, R, ID, Fu::normal_field>(wRC, wRp, ch, fR);
  R cmax, cmin = R(0);
  if constexpr (RIEM == RIEM_TVDLF) {
    cbounds<P, R, ID, false, Fu::einfeldt>(wLC, wRC, wLp, wRp, fp, cmax, cmin, crash);
    if constexpr (CT) { ctio->cmax = cmax; ctio->cmin = cmin; }
    const R fac = R(-0.5) * R(fp.tvdlfeps) * cmax;
#pragma unroll
    for (int iw = 0; iw < NW; ++iw) {
      fC[iw] = R(0.5) * (fL[iw] + fR[iw]);
      if constexpr (Fu::mass_flux)
        if (iw == P::RHO) fC[iw] = R(0.5) * fma(wLp[P::MOM + ID], wLp[P::RHO], fR[P::RHO]);
      fC[iw] = fC[iw] + fac * (wRC[iw] - wLC[iw]);
    }
  } else {
    cbounds<P, R, ID, true>(wLC, wRC, wLp, wRp, fp, cmax, cmin, crash);
    if constexpr (CT) { ctio->cmax = cmax; ctio->cmin = cmin; }
    // flux_type: normal B gets Lax-Friedrichs dissipation only without GLM
    // (src/mhd/mod_mhd_phys.t:580-588)
    constexpr int BTV = (P::MHD && !P::GLM && P::NDIM > 1) ? (P::MAG + ID) : -1;
    if constexpr (RIEM == RIEM_HLLD) {
      if constexpr (CT) hlld_flux<P, R, ID, true>(wLC, wRC, wLp, wRp, fL, fR, cmax, cmin, fC, R(ctio->bx));
      else hlld_flux<P, R, ID>(wLC, wRC, wLp, wRp, fL, fR, cmax, cmin, fC);
    } else if constexpr (RIEM == RIEM_HLL && kFast64<R>) {
      // the three cases as weights of fL, fR and the jump, formed once
      const R inv = frcp(cmax - cmin);
      R aL = cmax * inv, aR = -cmin * inv, aD = cmin * aL;
      if (cmin >= R(0)) { aL = R(1); aR = R(0); aD = R(0); }
      else if (cmax <= R(0)) { aL = R(0); aR = R(1); aD = R(0); }
      // a side of weight 0 that is infinite (its energy flux is then infinite or
      // NaN) is not read
      if (__builtin_expect(!(fabs(fL[P::E] + fR[P::E]) < HUGE_VAL), 0)) {
#pragma unroll
        for (int iw = 0; iw < NW; ++iw) {
          if (iw == BTV) continue;
          if (cmin >= R(0)) { fR[iw] = fL[iw]; wRC[iw] = wLC[iw]; }
          else if (cmax <= R(0)) { fL[iw] = fR[iw]; wLC[iw] = wRC[iw]; }
        }
      }
#pragma unroll
      for (int iw = 0; iw < NW; ++iw) {
        if (iw == BTV) fC[iw] = -R(fp.tvdlfeps) * R(0.5) * mx2(cmax, R(fabs(cmin))) * (wRC[iw] - wLC[iw]);
        // both states carry the same normal field and psi, hence one flux
        else if (P::GLM && (iw == P::PSI || iw == P::MAG + ID)) fC[iw] = fL[iw];
        else fC[iw] = aL * fL[iw] + aR * fR[iw] + aD * (wRC[iw] - wLC[iw]);
      }
    } else if constexpr (RIEM == RIEM_HLL) {
      const R inv = frcp(cmax - cmin);
#pragma unroll
      for (int iw = 0; iw < NW; ++iw) {
        if (iw == BTV) {
          fC[iw] = -R(fp.tvdlfeps) * R(0.5) * mx2(cmax, R(fabs(cmin))) * (wRC[iw] - wLC[iw]);
        } else if (cmin >= R(0)) {
          fC[iw] = fL[iw];
        } else if (cmax <= R(0)) {
          fC[iw] = fR[iw];
        } else {
          const R num = cmax * fL[iw] - cmin * fR[iw] + cmin * cmax * (wRC[iw] - wLC[iw]);
          if constexpr (kExact) fC[iw] = num / (cmax - cmin);
          else fC[iw] = num * inv;
        }
      }
    } else {  // HLLC: hd_get_lCD / hd_get_wCD or mhd_get_lCD / mhd_get_wCD
      constexpr int RHO = P::RHO, MN = P::MOM + ID, E = P::E;
      int patchf = 1;
      if (cmin >= R(0)) patchf = -2;
      else if (cmax <= R(0)) patchf = 2;
      R lambdaCD = R(0);
      R Fhll[NW];
      // the HLL state of the magnetic field and momentum (MHD contact state)
      R whll[P::MHD ? NW : 1];
      if (patchf == 1) {
        R whll_m = R(0), whll_r = R(0);
        const R inv = frcp(cmax - cmin);
#pragma unroll
        for (int iw = 0; iw < NW; ++iw) {
          const R nf = cmax * fL[iw] - cmin * fR[iw] + cmin * cmax * (wRC[iw] - wLC[iw]);
          const R nw = cmax * wRC[iw] - cmin * wLC[iw] + fL[iw] - fR[iw];
          R wh;
          if constexpr (kExact) {
            Fhll[iw] = nf / (cmax - cmin);
            wh = nw / (cmax - cmin);
          } else {
            Fhll[iw] = nf * inv;
            wh = nw * inv;
          }
          if (iw == MN) whll_m = wh;
          if (iw == RHO) whll_r = wh;
          if constexpr (P::MHD) whll[iw] = wh;
        }
        lambdaCD = fdiv(whll_m, whll_r);
        bool cond = true;
        if (cmin < R(0) && lambdaCD > R(0) && lambdaCD < cmax) {
          patchf = -1;
        } else if (cmax > R(0) && lambdaCD < R(0) && lambdaCD > cmin) {
          patchf = 1;
        } else if (lambdaCD >= cmax || lambdaCD <= cmin) {
          lambdaCD = R(0);
          patchf = 3;
          cond = false;
        }
        if (cond && lambdaCD == R(0)) patchf = (-cmin >= cmax) ? 1 : -1;
      } else {
#pragma unroll
        for (int iw = 0; iw < NW; ++iw) Fhll[iw] = R(0);
      }
      if (patchf == 1 || patchf == -1) {
        const bool right = patchf == 1;
        const R cspeed = right ? cmax : cmin;
        R wSub[NW], fSub[NW], wCD[NW];
#pragma unroll
        for (int iw = 0; iw < NW; ++iw) {
          wSub[iw] = right ? wRC[iw] : wLC[iw];
          fSub[iw] = right ? fR[iw] : fL[iw];
        }
        const R vSub = fdiv(wSub[MN], wSub[RHO]);
        if constexpr (P::MHD) {
          // mhd_get_wCD src/mhd/mod_mhd_hllc.t:147-240 (Li 2005)
          constexpr int BN = P::MAG + ID;
          const R den = cspeed - lambdaCD;
          wCD[RHO] = fdiv(wSub[RHO] * (cspeed - vSub), den);
#pragma unroll
          for (int d = 0; d < P::NDIR; ++d) wCD[P::MAG + d] = whll[P::MAG + d];
#pragma unroll
          for (int d = 0; d < P::NDIR; ++d) {
            if (d != ID)
              wCD[P::MOM + d] = fdiv(cspeed * wSub[P::MOM + d] - fSub[P::MOM + d] - wCD[BN] * wCD[P::MAG + d], den);
            else
              wCD[P::MOM + d] = wCD[RHO] * lambdaCD;
          }
          R vb = whll[P::MOM] * whll[P::MAG];
#pragma unroll
          for (int d = 1; d < P::NDIR; ++d) vb = vb + whll[P::MOM + d] * whll[P::MAG + d];
          const R vdotb = fdiv(vb, whll[RHO]);
          const R pCD = wSub[RHO] * (cspeed - vSub) * (lambdaCD - vSub) + fSub[MN] - wSub[MN] * vSub + wCD[BN] * wCD[BN];
          wCD[E] = fdiv(cspeed * wSub[E] - fSub[E] + lambdaCD * pCD - vdotb * wCD[BN], den);
#pragma unroll
          for (int iw = 0; iw < NW; ++iw) {
            if (iw == BN || (P::GLM && iw == P::PSI)) fC[iw] = R(0);
            else fC[iw] = fSub[iw] + cspeed * (wCD[iw] - wSub[iw]);
          }
        } else {
          const R csmls = frcp(cspeed - lambdaCD);
          wCD[RHO] = wSub[RHO] * (cspeed - vSub) * csmls;
#pragma unroll
          for (int d = 0; d < P::NDIR; ++d) {
            if (d != ID) wCD[P::MOM + d] = (cspeed * wSub[P::MOM + d] - fSub[P::MOM + d]) * csmls;
            else wCD[P::MOM + d] = wCD[RHO] * lambdaCD;
          }
          const R pCD = wSub[RHO] * (cspeed - vSub) * (lambdaCD - vSub) + fSub[MN] - wSub[MN] * vSub;
          wCD[E] = (cspeed * wSub[E] - fSub[E] + lambdaCD * pCD) * csmls;
#pragma unroll
          for (int iw = 0; iw < NW; ++iw) fC[iw] = fSub[iw] + cspeed * (wCD[iw] - wSub[iw]);
        }
      } else if (patchf == -2) {
#pragma unroll
        for (int iw = 0; iw < NW; ++iw) fC[iw] = fL[iw];
      } else if (patchf == 2) {
#pragma unroll
        for (int iw = 0; iw < NW; ++iw) fC[iw] = fR[iw];
      } else {
#pragma unroll
        for (int iw = 0; iw < NW; ++iw) fC[iw] = Fhll[iw];
      }
      // flux_type: the normal field takes Lax-Friedrichs dissipation only
      // without GLM (src/mod_finite_volume.t:477-479)
      if constexpr (BTV >= 0)
        fC[BTV] = -R(fp.tvdlfeps) * R(0.5) * mx2(cmax, R(fabs(cmin))) * (wRC[BTV] - wLC[BTV]);
    }
  }
}

// cell-centred cmax for dt: hd_get_cmax src/hd/mod_hd_phys.t:787-811,
// mhd_get_cmax_origin src/mhd/mod_mhd_phys.t:2482-2550 (FP64, primitive
// w), written out without contraction (see cfl_cell)
template <class P, int ID>
__device__ __forceinline__ double cfl_cmax(const double* w, const FVParams& fp) {
#pragma clang fp contract(off)
  if constexpr (!P::MHD) {
    return fabs(w[P::MOM + ID]) + sqrt(fp.gamma * w[P::E] / w[P::RHO]);
  } else {
    // mhd_get_csound_prim, as fast_speed
    const double inv_rho = frcp(w[P::RHO]);
    const double cs = fp.gamma * w[P::E] * inv_rho;
    double b2 = w[P::MAG] * w[P::MAG];
#pragma unroll
    for (int d = 1; d < P::NDIR; ++d) b2 = b2 + w[P::MAG + d] * w[P::MAG + d];
    const double cfast2 = b2 * inv_rho + cs;
    const double bn = w[P::MAG + ID];
    double av = cfast2 * cfast2 - 4.0 * cs * (bn * bn) * inv_rho;
    if (av < 0.0) av = 0.0;
    return fabs(w[P::MOM + ID]) + fsqrt(0.5 * (cfast2 + fsqrt(av)));
  }
}

// getdt_courant (maxsum, slab_uniform; src/mod_dt.t:160-287) of one
// conserved cell folded into the running maxima maxtot (of sum_d
// cmax_d/dx_d) and cmaxb (of cmax).  Every operation is written here
// without contraction whatever the translation unit's setting, so that the
// dt kernel and the stage kernel's fused CFL partials round alike.
template <class P>
__device__ __forceinline__ void cfl_cell(const double* cons, const FVParams& fp, double& maxtot, double& cmaxb) {
#pragma clang fp contract(off)
  double w[P::NW];
#pragma unroll
  for (int iw = 0; iw < P::NW; ++iw) w[iw] = cons[iw];
  // to_prim (hd_to_primitive / mhd_to_primitive_origin)
  const double inv_rho = 1.0 / w[P::RHO];
#pragma unroll
  for (int d = 0; d < P::NDIR; ++d) w[P::MOM + d] = w[P::MOM + d] * inv_rho;
  double vsq = w[P::MOM] * w[P::MOM];
#pragma unroll
  for (int d = 1; d < P::NDIR; ++d) vsq = vsq + w[P::MOM + d] * w[P::MOM + d];
  if constexpr (!P::MHD) {
    w[P::E] = (fp.gamma - 1.0) * (w[P::E] - 0.5 * w[P::RHO] * vsq);
  } else {
    double bsq = w[P::MAG] * w[P::MAG];
#pragma unroll
    for (int d = 1; d < P::NDIR; ++d) bsq = bsq + w[P::MAG + d] * w[P::MAG + d];
    w[P::E] = fp.gamma_1 * (w[P::E] - 0.5 * (w[P::RHO] * vsq + bsq));
  }
  double cm = cfl_cmax<P, 0>(w, fp);
  cmaxb = fmax(cmaxb, cm);
  double tot = cm * fp.dxinv[0];
  if constexpr (P::NDIM > 1) {
    cm = cfl_cmax<P, 1>(w, fp);
    cmaxb = fmax(cmaxb, cm);
    tot = tot + cm * fp.dxinv[1];
  }
  if constexpr (P::NDIM > 2) {
    cm = cfl_cmax<P, 2>(w, fp);
    cmaxb = fmax(cmaxb, cm);
    tot = tot + cm * fp.dxinv[2];
  }
  maxtot = fmax(maxtot, tot);
}

}  // namespace FV_NS
