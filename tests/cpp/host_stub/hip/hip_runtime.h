// Stand-in for the HIP runtime header: lets the host compiler build the device header's scalar
// functions (tests/cpp/fault_solve.cpp).  The hardware estimates are rounded as coarsely as the
// hardware's may be (reciprocal 2^-23, exp2 and log2 in FP32).
#pragma once
#include <cmath>
#include <cstring>
#include <algorithm>
#define __device__
#define __host__
#define __global__
#define __forceinline__ inline
using std::max;
using std::min;
using std::isnan;
static inline double __builtin_amdgcn_rcp(double x) { return (double)(1.0f / (float)1.0f) / x * (1.0 + 1e-7); }
static inline float __builtin_amdgcn_rcpf(float x) { return (1.0f / x) * (1.0f + 1e-7f); }
static inline float __builtin_amdgcn_exp2f(float x) { return exp2f(x); }
static inline float __builtin_amdgcn_logf(float x) { return log2f(x); }
static inline float __builtin_amdgcn_fmed3f(float a, float b, float c) { return std::max(std::min(a, b), std::min(std::max(a, b), c)); }
