// What the device headers without kernels need from the HIP runtime header, for tests that
// compile them with the host compiler.
#pragma once
#include <cmath>
#define __device__
#define __host__
#define __forceinline__ inline
#define __restrict__ __restrict
#define __builtin_amdgcn_fence(...) ((void)0)
#define __builtin_amdgcn_wave_barrier() ((void)0)
#define __syncthreads() ((void)0)
struct float2 { float x, y; };
static inline float2 make_float2(float x, float y) { return {x, y}; }
