// The FFT core's FP32 arithmetic on the host against a transform in double:
// relative rms over a batch, one line per length, input and direction.  Each
// thread of a transform is a coroutine; the core's wavefront ordering points
// hand over to the next one.
#include <hip/hip_runtime.h>
#include <ucontext.h>

#include <complex>
#include <cstdio>
#include <functional>
#include <random>
#include <vector>

#include "fft_core.h"

HostIndex threadIdx;

namespace {

using cd = std::complex<double>;
constexpr size_t STACK = 1 << 18;
std::vector<ucontext_t> fibers;
std::vector<std::vector<char>> stacks;
std::vector<char> done;
ucontext_t caller;
std::function<void(int)> body;
int now;

void entry(int i) {
  body(i);
  done[i] = 1;
  for (size_t k = 1; k < fibers.size(); ++k) {
    const int j = (int)((i + k) % fibers.size());
    if (!done[j]) {
      now = j;
      setcontext(&fibers[j]);
    }
  }
  setcontext(&caller);
}

void run(int n, std::function<void(int)> f) {
  body = std::move(f);
  fibers.assign(n, ucontext_t{});
  done.assign(n, 0);
  stacks.resize(n);
  for (int i = 0; i < n; ++i) {
    stacks[i].resize(STACK);
    getcontext(&fibers[i]);
    fibers[i].uc_stack.ss_sp = stacks[i].data();
    fibers[i].uc_stack.ss_size = STACK;
    fibers[i].uc_link = nullptr;
    makecontext(&fibers[i], (void (*)())entry, 1, i);
  }
  now = 0;
  swapcontext(&caller, &fibers[0]);
}

void dft(std::vector<cd>& a, int s) {
  const size_t n = a.size();
  if (n == 1) return;
  std::vector<cd> e(n / 2), o(n / 2);
  for (size_t i = 0; i < n / 2; ++i) {
    e[i] = a[2 * i];
    o[i] = a[2 * i + 1];
  }
  dft(e, s);
  dft(o, s);
  for (size_t k = 0; k < n / 2; ++k) {
    const cd w = std::polar(1.0, s * 2 * M_PI * (double)k / (double)n) * o[k];
    a[k] = e[k] + w;
    a[k + n / 2] = e[k] - w;
  }
}

// smooth: a windowed image row; normal: noise
template <int N, int S, bool PLAN>
double rms(bool smooth, int reps, const float2* tw) {
  constexpr int TPT = N / 16;
  std::mt19937 g(N + smooth);
  std::normal_distribution<double> nd;
  std::uniform_real_distribution<double> ud;
  std::vector<float2> sl(vmbd::FftLds<N>::floats2), out(N);
  double num = 0, den = 0;
  for (int rep = 0; rep < reps; ++rep) {
    std::vector<cd> a(N);
    for (int i = 0; i < N; ++i) {
      const double w = 0.5 - 0.5 * std::cos(2 * M_PI * (i + 0.5) / N);
      const cd v = smooth ? w * cd(0.5 + 0.1 * ud(g) + 0.3 * std::sin(6.0 * i / N + rep),
                                   0.4 + 0.1 * ud(g) + 0.3 * std::cos(5.0 * i / N + rep))
                          : cd(nd(g), nd(g));
      a[i] = cd((float)v.real(), (float)v.imag());
    }
    run(TPT, [&](int t) {
      float2 v[16];
      for (int r = 0; r < 16; ++r) v[r] = make_float2((float)a[t + TPT * r].real(), (float)a[t + TPT * r].imag());
      vmbd::Twiddles<N> T;
      vmbd::twiddles_init<N, PLAN>(T, t, tw);
      vmbd::fft<N, S>(v, sl.data(), t, T);
      for (int m = 0; m < 16; ++m) out[t + TPT * m] = v[m];
    });
    dft(a, S);
    for (int i = 0; i < N; ++i) {
      num += std::norm(cd(out[i].x, out[i].y) - a[i]);
      den += std::norm(a[i]);
    }
  }
  return std::sqrt(num / den);
}

template <int N>
void line(const float2* tw) {
  constexpr bool P = N <= 512;  // a plan's tiles
  const int reps = 51200 / N;
  for (int smooth = 0; smooth < 2; ++smooth)
    std::printf("%d %d %.4e %.4e %.4e %.4e\n", N, smooth, rms<N, -1, P>(smooth, reps, tw),
                rms<N, +1, P>(smooth, reps, tw), rms<N, -1, false>(smooth, reps, tw),
                rms<N, +1, false>(smooth, reps, tw));
}

}  // namespace

void host_wave_sync() {
  const int me = now;
  now = (now + 1) % (int)fibers.size();
  swapcontext(&fibers[me], &fibers[now]);
}

int main() {
  std::vector<float2> tw(vmbd::TW_PLAN);
  vmbd::twiddle_table(tw.data());
  line<16>(tw.data());
  line<32>(tw.data());
  line<64>(tw.data());
  line<128>(tw.data());
  line<256>(tw.data());
  line<512>(tw.data());
  line<1024>(tw.data());
}
