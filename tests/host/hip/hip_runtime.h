// Stand-in for the HIP runtime header that lets the host compiler build the
// device code of the FP64 march (tests/host/trace64_host.cpp): one lane a
// call, the hardware estimates replaced by exact values of the same kind.
#pragma once
#include <math.h>
#include <stddef.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>

#define __device__
#define __host__
#define __forceinline__ inline
#define __any(x) (x)
#define __builtin_amdgcn_rsq(x) (1.0 / std::sqrt((double)(x)))
#define __builtin_amdgcn_rsqf(x) (1.0f / std::sqrt((float)(x)))
#define __builtin_amdgcn_rcpf(x) (1.0f / (float)(x))
#define __builtin_amdgcn_sqrtf(x) std::sqrt((float)(x))
#define __builtin_amdgcn_sinf(x) std::sin(6.28318531f * (x))
#define __builtin_amdgcn_cosf(x) std::cos(6.28318531f * (x))

typedef int hipError_t;
typedef void* hipStream_t;
struct uint2 {
  unsigned x, y;
};
using std::isnan;
using std::max;
using std::min;
