// Radix-16/8/4/2 Stockham FFT core for gfx950 (wave64).
//
// One complex transform of length N (16 <= N <= 1024, power of two) is
// carried by TPT = N/16 threads that each hold 16 points in registers.  All
// TPT threads of a transform sit inside one wavefront (TPT <= 64 and TPT
// divides 64), so the exchanges between passes go through the transform's own
// LDS slice with wavefront-level ordering only, no workgroup barrier.
//
// Register mappings (both validated against numpy.fft on the host):
//   input : thread t, slot r  holds  x[t + TPT*r]
//   output: thread t, slot m  holds  X[t + TPT*m]
// The identical mapping on both sides lets a forward transform, a pointwise
// product and an inverse transform run back to back in registers.
//
// Algorithm: self-sorting Stockham passes with radix 16 first, then the
// remaining factor (Govindaraju et al., "High performance discrete Fourier
// transforms on graphics processors", SC'08): pass with span Ns and radix R
// reads x[j + r*N/R], multiplies by w^(r*(j mod Ns)) with w = e^{S 2 pi i/(Ns R)},
// applies an R-point DFT and writes (j/Ns)*Ns*R + (j mod Ns) + r*Ns.
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>

namespace vmbd {

// Twiddle table length.  tw[m] = exp(-2 pi i m / TW_LEN), rounded from FP64.
constexpr int TW_LEN = 1024;
// A plan's table goes on with the twiddles of the passes after the first as the
// butterflies take them (Twiddles), the entries of one butterfly together: the
// second passes of radix 2, 4, 8 and 16, then the third pass of 512 points.
constexpr int TW_P2 = TW_LEN;
constexpr int TW_P3 = TW_P2 + 240;
constexpr int TW_PLAN = TW_P3 + 128;

__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
  return make_float2(fmaf(a.x, b.x, -a.y * b.y), fmaf(a.x, b.y, a.y * b.x));
}
// a * conj(b)
__device__ __forceinline__ float2 cmulc(float2 a, float2 b) {
  return make_float2(fmaf(a.x, b.x, a.y * b.y), fmaf(a.y, b.x, -a.x * b.y));
}
__device__ __forceinline__ float2 cscale(float2 a, float s) { return make_float2(a.x * s, a.y * s); }
__device__ __forceinline__ float2 cconj(float2 a) { return make_float2(a.x, -a.y); }
// S * i * a
template <int S>
__device__ __forceinline__ float2 mul_si(float2 a) { return make_float2(-(float)S * a.y, (float)S * a.x); }

// Wavefront-scope ordering point for LDS exchanges inside one wavefront.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---------------------------------------------------------------- small DFTs
// All produce outputs in natural order in place; S = -1 forward, +1 inverse.
//
// Every transform of the operator is bound by VALU issue or waits behind it,
// and an FMA takes the issue slot of an addition, so both passes are written
// to put their multiplications into FMAs.  Per 256-point transform and thread
// (16 points): first pass 144 (from 160: constant twiddles factored out of
// the sums), second pass 208 (from 160 + 60 for the separate products), 352
// instead of 380 slots, with 8 twiddle register pairs instead of 15.
#define VMBD_R2H 0.70710678118654752440f
#define VMBD_C8 0.92387953251128675613f  // cos(pi/8)
#define VMBD_S8 0.38268343236508977173f  // sin(pi/8)
#define VMBD_T8 0.41421356237309504880f  // tan(pi/8)

// a + s * b, a + S * s * i * b (s real)
__device__ __forceinline__ float2 cfma(float s, float2 b, float2 a) {
  return make_float2(fmaf(s, b.x, a.x), fmaf(s, b.y, a.y));
}
template <int S>
__device__ __forceinline__ float2 cfma_si(float s, float2 b, float2 a) {
  return make_float2(fmaf(-(float)S * s, b.y, a.x), fmaf((float)S * s, b.x, a.y));
}
// (1 + S i f) * a and (f + S i) * a
template <int S>
__device__ __forceinline__ float2 mul_1f(float2 a, float f) {
  return make_float2(fmaf(-(float)S * f, a.y, a.x), fmaf((float)S * f, a.x, a.y));
}
template <int S>
__device__ __forceinline__ float2 mul_f1(float2 a, float f) {
  return make_float2(fmaf(f, a.x, -(float)S * a.y), fmaf(f, a.y, (float)S * a.x));
}

// 4-point DFT of which the first K inputs are nonzero
template <int S, int K = 4>
__device__ __forceinline__ void dft4(float2& a0, float2& a1, float2& a2, float2& a3) {
  if constexpr (K == 0) {
    a0 = a1 = a2 = a3 = make_float2(0.f, 0.f);
  } else if constexpr (K == 1) {
    a1 = a2 = a3 = a0;
  } else {
    const float2 t0 = K > 2 ? cadd(a0, a2) : a0, t1 = K > 2 ? csub(a0, a2) : a0;
    const float2 t2 = K > 3 ? cadd(a1, a3) : a1, t3 = mul_si<S>(K > 3 ? csub(a1, a3) : a1);
    a0 = cadd(t0, t2);
    a2 = csub(t0, t2);
    a1 = cadd(t1, t3);
    a3 = csub(t1, t3);
  }
}

// 16-point DFT whose inputs r >= NZ are zero (not read)
template <int S, int NZ = 16>
__device__ __forceinline__ void dft16(float2 (&v)[16]) {
  static_assert(NZ >= 3 && NZ <= 16, "NZ in [3,16]");
  constexpr bool A3 = NZ > 3;  // the n2 = 3 branch has inputs
  // n = 4 n1 + n2, k = k1 + 4 k2.  Step 1: DFT4 over n1 for each n2:
  // v[n2 + 4 k1] = Y[n2][k1]
  dft4<S, (NZ + 3) / 4>(v[0], v[4], v[8], v[12]);
  dft4<S, (NZ + 2) / 4>(v[1], v[5], v[9], v[13]);
  dft4<S, (NZ + 1) / 4>(v[2], v[6], v[10], v[14]);
  dft4<S, NZ / 4>(v[3], v[7], v[11], v[15]);
  // Step 2 and 3: a_n2 = Y[n2][k1] w16^(n2 k1), DFT4 over n2 -> X[k1 + 4 k2]
  float2 o[16];
  float2 t0, t1, u, d;
  {  // k1 = 0
    t0 = cadd(v[0], v[2]);
    t1 = csub(v[0], v[2]);
    u = A3 ? cadd(v[1], v[3]) : v[1];
    d = A3 ? csub(v[1], v[3]) : v[1];
    o[0] = cadd(t0, u);
    o[8] = csub(t0, u);
    o[4] = cadd(t1, mul_si<S>(d));
    o[12] = csub(t1, mul_si<S>(d));
  }
  {  // k1 = 1: w1 = C8 (1 + S i T8), w2 = R2H (1 + S i), w3 = C8 (T8 + S i)
    const float2 p = mul_1f<S>(v[6], 1.f);
    t0 = cfma(VMBD_R2H, p, v[4]);
    t1 = cfma(-VMBD_R2H, p, v[4]);
    const float2 q1 = mul_1f<S>(v[5], VMBD_T8);
    u = d = q1;
    if constexpr (A3) {
      const float2 q3 = mul_f1<S>(v[7], VMBD_T8);
      u = cadd(q1, q3);
      d = csub(q1, q3);
    }
    o[1] = cfma(VMBD_C8, u, t0);
    o[9] = cfma(-VMBD_C8, u, t0);
    o[5] = cfma_si<S>(VMBD_C8, d, t1);
    o[13] = cfma_si<S>(-VMBD_C8, d, t1);
  }
  {  // k1 = 2: w2, w4 = S i, w6 = R2H (-1 + S i) = S i w2
    t0 = cadd(v[8], mul_si<S>(v[10]));
    t1 = csub(v[8], mul_si<S>(v[10]));
    const float2 p1 = mul_1f<S>(v[9], 1.f);
    u = d = p1;
    if constexpr (A3) {
      const float2 p3 = mul_si<S>(mul_1f<S>(v[11], 1.f));
      u = cadd(p1, p3);
      d = csub(p1, p3);
    }
    o[2] = cfma(VMBD_R2H, u, t0);
    o[10] = cfma(-VMBD_R2H, u, t0);
    o[6] = cfma_si<S>(VMBD_R2H, d, t1);
    o[14] = cfma_si<S>(-VMBD_R2H, d, t1);
  }
  {  // k1 = 3: w3 = C8 (T8 + S i), w6 = R2H S i (1 + S i), w9 = -C8 (1 + S i T8)
    const float2 p = mul_si<S>(mul_1f<S>(v[14], 1.f));
    t0 = cfma(VMBD_R2H, p, v[12]);
    t1 = cfma(-VMBD_R2H, p, v[12]);
    const float2 q1 = mul_f1<S>(v[13], VMBD_T8);
    u = d = q1;
    if constexpr (A3) {
      const float2 q3 = mul_1f<S>(v[15], VMBD_T8);
      u = csub(q1, q3);
      d = cadd(q1, q3);
    }
    o[3] = cfma(VMBD_C8, u, t0);
    o[11] = cfma(-VMBD_C8, u, t0);
    o[7] = cfma_si<S>(VMBD_C8, d, t1);
    o[15] = cfma_si<S>(-VMBD_C8, d, t1);
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) v[i] = o[i];
}

// Radix-2 butterflies hi = a + W b, lo = a - W b.  w: forward twiddle
// (conjugated for S = +1); ROT: W = S i w.
// bfly_tan: w as (cos, tan) of its angle, |angle| < pi/2; W b = cos (b + i tan b)
// and both outputs are FMAs of a and that, six in all (Linzer and Feig,
// "Implementation of efficient FFT algorithms on fused multiply-add
// architectures", 1993).  bfly_exp: w as (cos, sin), any angle, eight FMAs (as a
// product and two sums it has the same eight slots, but the scheduler then keeps
// 30 registers more: the two-adjoint pass spilled 33 instead of 5).
// Each output is rounded from its own sum: lo taken as 2a - hi needs no product
// of its own either, but carries hi's rounding into a difference that may be
// small (256 points of smooth input 1.04e-7 rms against 64 bits, 512 points
// 1.11e-7, where these give 0.90e-7 and 0.95e-7).
template <int S, bool ROT>
__device__ __forceinline__ void bfly_tan(float2 a, float2 b, float2 w, float2& hi, float2& lo) {
  if constexpr (ROT) b = mul_si<S>(b);
  const float t = -(float)S * w.y;
  const float2 u = make_float2(fmaf(-t, b.y, b.x), fmaf(t, b.x, b.y));
  hi = cfma(w.x, u, a);
  lo = cfma(-w.x, u, a);
}
template <int S>
__device__ __forceinline__ void bfly_exp(float2 a, float2 b, float2 w, float2& hi, float2& lo) {
  const float y = -(float)S * w.y;
  hi = make_float2(fmaf(-y, b.y, fmaf(w.x, b.x, a.x)), fmaf(y, b.x, fmaf(w.x, b.y, a.y)));
  lo = make_float2(fmaf(y, b.y, fmaf(-w.x, b.x, a.x)), fmaf(-y, b.x, fmaf(-w.x, b.y, a.y)));
}

// Twiddles of an R-point DFT of w^r x_r: level R (spans R/2) uses w e_R^k,
// k < R/2, of which the second half is S i times the first; then level R/2
// with w^2, and so on.  Kept per level: R/4 (one at R = 2), R/2 in all.  Above
// level 2 the kept angles stay below a quarter turn and are held as (cos, tan);
// the last spans a half turn and is held as (cos, sin).
template <int R>
struct TwCount {
  static constexpr int top = R > 2 ? R / 4 : 1;
  static constexpr int n = R > 2 ? top + TwCount<(R > 2 ? R / 2 : 2)>::n : 1;
};
template <>
struct TwCount<2> {
  static constexpr int top = 1, n = 1;
};

// X[k] = sum_r x_r w^r e^{S 2 pi i r k / R}, decimation in time, natural order
template <int R, int S>
__device__ __forceinline__ void dft_tw(float2* x, const float2* w) {
  if constexpr (R == 2) {
    const float2 a = x[0], b = x[1];
    bfly_exp<S>(a, b, w[0], x[0], x[1]);
  } else {
    constexpr int H = R / 2;
    float2 e[H], o[H];
#pragma unroll
    for (int j = 0; j < H; ++j) {
      e[j] = x[2 * j];
      o[j] = x[2 * j + 1];
    }
    dft_tw<H, S>(e, w + TwCount<R>::top);
    // halves one after the other: interleaved, the 512-point two-adjoint pass
    // spills 24 registers instead of 10
    if constexpr (R == 16) __builtin_amdgcn_sched_barrier(0);
    dft_tw<H, S>(o, w + TwCount<R>::top);
    if constexpr (R == 16) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < H / 2; ++k) {
      bfly_tan<S, false>(e[k], o[k], w[k], x[k], x[k + H]);
      bfly_tan<S, true>(e[k + H / 2], o[k + H / 2], w[k], x[k + H / 2], x[k + H / 2 + H]);
    }
  }
}

// LDS slot of element i inside a transform's slice (one pad slot per 16).
__device__ __forceinline__ int lds_pad(int i) { return i + (i >> 4); }
template <int N>
struct FftLds {
  static constexpr int floats2 = N + N / 16;  // float2 slots per transform
};

// Radix plan of a length-N transform after the first radix-16 pass.
template <int N>
struct Plan {
  static constexpr int R1 = (N >= 256) ? 16 : N / 16;  // second pass radix
  static constexpr int R2 = (N > 256) ? N / 256 : 1;   // third pass radix
};

// Per-thread forward twiddles of the passes after the first, in the order of
// TwCount.  Second pass (span 16): the thread's 16/R1 butterflies j = t + b*TPT
// use w = e^{-2 pi i (j mod 16) / (16 R1)}.  Third pass (span 256): butterflies
// j = t + b*TPT use w = e^{-2 pi i j / (256 R2)}, of which b and b + 4 (R2 = 2)
// differ by a quarter turn, so four are kept.  They depend only on t: a kernel
// sets them up once for every transform it performs.
template <int N>
struct Twiddles {
  static constexpr int R1 = Plan<N>::R1;
  static constexpr int R2 = Plan<N>::R2;
  static constexpr int NB1 = (R1 > 1) ? 16 / R1 : 1;
  static constexpr int C1 = (R1 > 1) ? TwCount<(R1 > 1 ? R1 : 2)>::n : 1;
  static constexpr int C2 = (R2 > 1) ? TwCount<(R2 > 1 ? R2 : 2)>::n : 1;
  static constexpr int N2 = NB1 * C1, N3 = (R2 > 1) ? 4 * C2 : 1;
  float2 w[N2];
  float2 w3[N3];
  __device__ __forceinline__ void second(float2 (&o)[N2], int) const {
#pragma unroll
    for (int i = 0; i < N2; ++i) o[i] = w[i];
  }
  __device__ __forceinline__ void third(float2 (&o)[N3], int) const {
#pragma unroll
    for (int i = 0; i < N3; ++i) o[i] = w3[i];
  }
};

// (cos, tan) of w: one Newton step on the hardware reciprocal, which leaves the
// quotient's own rounding (100 transforms of 256^2: 39.6 us, 40.1 with the
// compiler's division; 37.5 with products of two entries, whose error is a
// fifth larger)
__device__ __forceinline__ float2 tw_tan(float2 w) {
  const float r = __builtin_amdgcn_rcpf(w.x), t = w.y * r;
  return make_float2(w.x, fmaf(fmaf(-t, w.x, w.y), r, t));
}

// twiddle array of an R-point DFT whose w has table index i
template <int R>
__device__ __forceinline__ void tw_load(float2* w, int i, const float2* __restrict__ tw) {
  if constexpr (R == 2) {
    w[0] = tw[i];
  } else {
    constexpr int top = TwCount<R>::top;
#pragma unroll
    for (int k = 0; k < top; ++k) w[k] = tw_tan(tw[i + k * (TW_LEN / R)]);
    tw_load<R / 2>(w + top, 2 * i, tw);
  }
}

// PLAN: every twiddle from a plan's table, as many instructions as forming
// them from w and w^4 takes and without the products' rounding (256 points 15 %
// rms); otherwise from the exponentials alone.
template <int N, bool PLAN = true>
__device__ __forceinline__ void twiddles_init(Twiddles<N>& T, int t, const float2* __restrict__ tw) {
  constexpr int R1 = Plan<N>::R1, R2 = Plan<N>::R2;
  static_assert(!PLAN || R2 <= 2, "a plan's tiles are at most 512 points");
  if constexpr (R1 > 1) {
#pragma unroll
    for (int b = 0; b < Twiddles<N>::NB1; ++b) {
      const int k = (t + b * (N / 16)) & 15;
      float2* w = T.w + b * Twiddles<N>::C1;
      if constexpr (PLAN) {
#pragma unroll
        for (int i = 0; i < Twiddles<N>::C1; ++i) w[i] = (tw + TW_P2 + 16 * (R1 / 2 - 1))[k * Twiddles<N>::C1 + i];
      } else {
        tw_load<R1>(w, k * (TW_LEN / (16 * R1)), tw);
      }
    }
  }
  if constexpr (R2 > 1) {
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int j = t + b * (N / 16);
      if constexpr (PLAN)
        T.w3[b] = (tw + TW_P3)[j];
      else if constexpr (R2 == 2)
        T.w3[b] = tw_tan(tw[2 * j]);
      else
        tw_load<R2>(T.w3 + b * Twiddles<N>::C2, j, tw);
    }
  }
}

// A plan's table on the host (TW_PLAN entries).  Exponentials are rounded from
// FP64; a tangent is the FP64 sine over the rounded cosine, so that their
// product is the sine to one rounding.
inline void twiddle_table(float2* tw) {
  auto sine = [](int i) { return std::sin(-2.0 * M_PI * (double)i / (double)TW_LEN); };
  for (int m = 0; m < TW_LEN; ++m)
    tw[m] = make_float2((float)std::cos(-2.0 * M_PI * (double)m / (double)TW_LEN), (float)sine(m));
  auto tan_entry = [&](int i) { return make_float2(tw[i].x, (float)(sine(i) / (double)tw[i].x)); };
  for (int R1 = 2; R1 <= 16; R1 *= 2)
    for (int k = 0; k < 16; ++k) {
      float2* o = tw + TW_P2 + 16 * (R1 / 2 - 1) + k * (R1 / 2);
      int i = k * (TW_LEN / (16 * R1));
      for (int R = R1; R > 2; R /= 2, i *= 2)  // the levels in the order of TwCount
        for (int q = 0; q < R / 4; ++q) *o++ = tan_entry(i + q * (TW_LEN / R));
      *o = tw[i];
    }
  for (int j = 0; j < 128; ++j) tw[TW_P3 + j] = tan_entry(2 * j);
}

// The same twiddles in LDS, shared by the transforms of a workgroup and read
// by the pass that uses them: a kernel that keeps the registers for its
// operands (slot i of thread t at i*TPT + t: consecutive lanes, no conflicts).
template <int N>
struct TwiddlesLds {
  using T = Twiddles<N>;
  static constexpr int TPT = N / 16;
  static constexpr int floats2 = TPT * (T::N2 + (T::R2 > 1 ? T::N3 : 0));
  const float2* p;
  // fills the table (the caller's barrier follows)
  static __device__ __forceinline__ void fill(float2* p, const float2* __restrict__ tw) {
    if ((int)threadIdx.x < TPT) {
      T r;
      twiddles_init<N>(r, threadIdx.x, tw);
#pragma unroll
      for (int i = 0; i < T::N2; ++i) p[i * TPT + threadIdx.x] = r.w[i];
      if constexpr (T::R2 > 1) {
#pragma unroll
        for (int i = 0; i < T::N3; ++i) p[(T::N2 + i) * TPT + threadIdx.x] = r.w3[i];
      }
    }
  }
  __device__ __forceinline__ void second(float2 (&o)[T::N2], int t) const {
#pragma unroll
    for (int i = 0; i < T::N2; ++i) o[i] = p[i * TPT + t];
  }
  __device__ __forceinline__ void third(float2 (&o)[T::N3], int t) const {
#pragma unroll
    for (int i = 0; i < T::N3; ++i) o[i] = p[(T::N2 + i) * TPT + t];
  }
};

// One Stockham pass after the first (NS > 1).  Reads 16 values of the slice,
// applies 16/R butterflies with their twiddles (from T: NB or, on a quarter
// turn from the first four, 4 arrays of TwCount<R>::n), writes 16 values (or keeps
// them in registers when LAST: slot m = b + r*(16/R) holds X[t + TPT*m]).
template <int N, int R, int NS, int S, bool LAST, class TWD>
__device__ __forceinline__ void stockham_pass(float2 (&v)[16], float2* sl, int t, const TWD& T) {
  constexpr int TPT = N / 16;
  constexpr int NB = 16 / R;
  float2 in[16];
  float2 w[NS > 16 ? Twiddles<N>::N3 : Twiddles<N>::N2];
  if constexpr (NS > 16)
    T.third(w, t);
  else
    T.second(w, t);
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int j = t + b * TPT;
#pragma unroll
    for (int r = 0; r < R; ++r) in[b * R + r] = sl[lds_pad(j + r * (N / R))];
  }
  wave_sync();
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int j = t + b * TPT;
    const int k = j & (NS - 1);
    float2* q = in + b * R;
    if constexpr (NS > 16 && R == 2) {
      // third pass of 512 points: butterfly b + 4 on a quarter turn from b
      const float2 x = q[0], y = q[1];
      if (b < 4)
        bfly_tan<S, false>(x, y, w[b & 3], q[0], q[1]);
      else
        bfly_tan<S, true>(x, y, w[b & 3], q[0], q[1]);
    } else {
      dft_tw<R, S>(q, w + b * TwCount<R>::n);
    }
    if constexpr (LAST) {
#pragma unroll
      for (int r = 0; r < R; ++r) v[b + r * NB] = q[r];
    } else {
      const int base = (j / NS) * NS * R + k;
#pragma unroll
      for (int r = 0; r < R; ++r) sl[lds_pad(base + r * NS)] = q[r];
    }
  }
  if constexpr (!LAST) wave_sync();
}

// Full complex FFT of length N on the slice `sl` (FftLds<N>::floats2 float2).
// v: input mapping on entry, output mapping on exit.  S=-1 forward, +1 inverse
// (unscaled).  Must be called by all TPT threads of the transform.
// NZ < 16: the caller guarantees x[t + TPT*r] = 0 for r >= NZ; those slots are
// not read, and the first pass shrinks to the arithmetic the nonzero inputs
// need (outputs a caller never reads are removed by the compiler once the
// call is inlined).
template <int N, int S, int NZ = 16, class TWD>
__device__ __forceinline__ void fft(float2 (&v)[16], float2* sl, int t, const TWD& T) {
  static_assert(N >= 16 && N <= 1024 && (N & (N - 1)) == 0, "N must be a power of two in [16,1024]");
  // pass 0: radix 16, Ns = 1, j = t, no twiddles; output index t*16 + r
  dft16<S, NZ>(v);
  if constexpr (N > 16) {
#pragma unroll
    for (int r = 0; r < 16; ++r) sl[lds_pad(t * 16 + r)] = v[r];
    wave_sync();
    constexpr int R1 = Plan<N>::R1;
    constexpr int R2 = Plan<N>::R2;
    if constexpr (R2 == 1) {
      stockham_pass<N, R1, 16, S, true>(v, sl, t, T);
    } else {
      stockham_pass<N, R1, 16, S, false>(v, sl, t, T);
      stockham_pass<N, R2, 256, S, true>(v, sl, t, T);
    }
  }
}

}  // namespace vmbd
