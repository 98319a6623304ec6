// What the Fourier divisions need of a frequency, from the twiddle table.
#pragma once
#include "fft_core.h"

namespace vmbd {

constexpr float SQRT1_2 = 0.70710678118654752440f;

// sin and cos of an angle of frequency q of T, 0 <= q < T: one table entry,
// correctly rounded.  (The entries of 16 frequencies from two by the sum of
// angles take no loads, but twice the error of 4 sin^2 and of the difference
// filter.)
struct Freq {
  float s, c;
};
// half: pi q / T;  full: 2 pi q / T
__device__ __forceinline__ Freq half_freq(int q, int T, const float2* __restrict__ tw) {
  const float2 w = tw[q * (TW_LEN / 2 / T)];
  return Freq{-w.y, w.x};
}
__device__ __forceinline__ Freq full_freq(int q, int T, const float2* __restrict__ tw) {
  const float2 w = tw[q * (TW_LEN / T)];
  return Freq{-w.y, w.x};
}

// 4 sin^2(pi q / T) = 2 - 2 cos(2 pi q / T), without its cancellation near 0
__device__ __forceinline__ float four_sin2(Freq h) { return 4.f * h.s * h.s; }
// (1 + 2 cos(2 pi q / T))^2, from the smaller of the two squares
__device__ __forceinline__ float one_2cos_sq(Freq h) {
  const float s2 = h.s * h.s, c2 = h.c * h.c;
  const float v = s2 < c2 ? fmaf(-4.f * h.s, h.s, 3.f) : fmaf(4.f * h.c, h.c, -1.f);
  return v * v;
}
// r (e^{-2 pi i q / T} - 1), r = sqrt(2)/2: the transform of the difference
// filter r [-1 1] placed at the tile origin (f: full angle)
__device__ __forceinline__ float2 diff_filter(Freq f) {
  return make_float2(SQRT1_2 * (f.c - 1.f), -SQRT1_2 * f.s);
}

}  // namespace vmbd
