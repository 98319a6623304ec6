// Stand-in for the HIP header: device arithmetic compiled for the host (the
// tests of rounding errors).  A wavefront's ordering point is the caller's.
#pragma once
#include <cmath>
#include <cstring>

#define __device__
#define __host__
#define __forceinline__ inline
#define __restrict__ __restrict

struct alignas(8) float2 {
  float x, y;
};
inline float2 make_float2(float x, float y) { return float2{x, y}; }

// the hardware's reciprocal, at its worst: one unit in the last place off
inline float __builtin_amdgcn_rcpf(float x) { return std::nextafter(1.0f / x, 4.0f * x); }

struct HostIndex {
  unsigned x;
};
extern HostIndex threadIdx;
void host_wave_sync();
#define __builtin_amdgcn_fence(order, scope) ((void)0)
#define __builtin_amdgcn_wave_barrier() host_wave_sync()
#define __builtin_amdgcn_sched_barrier(mask) ((void)0)
