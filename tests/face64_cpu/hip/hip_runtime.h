// Host-compiler stand-in for the HIP qualifiers and the gfx950 math builtins.
// The FP64 reciprocal and reciprocal square root carry a relative error of
// 2^-24, as the instructions may, so that the refinement steps are checked.
#pragma once
#include <cmath>
#define __device__
#define __host__
#define __global__
#define __forceinline__ inline
#define __launch_bounds__(...)
using std::copysign;
using std::fabs;
using std::fma;
using std::fmax;
using std::fmin;
using std::sqrt;
inline float __builtin_amdgcn_rcpf(float x) { return 1.0f / x; }
inline float __builtin_amdgcn_sqrtf(float x) { return std::sqrt(x); }
inline double __builtin_amdgcn_rcp(double x) { return 1.0 / x * (1.0 + 0x1p-24); }
inline double __builtin_amdgcn_rsq(double x) { return 1.0 / std::sqrt(x) * (1.0 - 0x1p-24); }
