// The frequency terms of the Fourier divisions on the host: T, q, 4 sin^2,
// (1 + 2 cos)^2 and the difference filter, one line per frequency.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <vector>

#include "div_terms.h"

HostIndex threadIdx;
void host_wave_sync() {}

int main() {
  using namespace vmbd;
  std::vector<float2> tw(TW_PLAN);
  twiddle_table(tw.data());
  for (int T = 16; T <= 512; T *= 2)
    for (int q = 0; q < T; ++q) {
      const Freq h = half_freq(q, T, tw.data());
      const float2 d = diff_filter(full_freq(q, T, tw.data()));
      std::printf("%d %d %.9g %.9g %.9g %.9g\n", T, q, four_sin2(h), one_2cos_sq(h), d.x, d.y);
    }
}
