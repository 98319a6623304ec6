// Column pass of the closed-form deconvolutions (olaGPU.py:416-733; the
// per-patch Fourier divisions of gputools.cu:316-406) for gfx950.
//
// Same decomposition as the operator's column pass (ola_kernels.hip): one
// workgroup per (patch, strip of 16 row bins), one 64-lane wavefront holding
// four 256-point column transforms, the row bins of real rows in half-spectrum
// form with bins 0 and Tw/2 packed into column 0.  Per column the kernel
// transforms its row-pass operands, reads its cached spectra, forms the
// division of DivOp (ola_kernels.h) bin by bin with the filter energies in
// closed form, and either inverse-transforms the quotient and stores the rows
// the caller needs or (SPROD) stores the product as a spectrum.
//
// The packed column carries two Hermitian spectra D (row bin 0) and N (row
// bin Tw/2) as P = D + iN.  A division is not bilinear, so its operands are
// taken apart first: each transform of that column is staged in LDS and
// D(k) = (P(k) + conj P(-k))/2, N(k) = (P(k) - conj P(-k))/(2i) are formed from
// it; the quotients of both parts (Hermitian again) are put back as D' + iN'.
#include "col_device.h"
#include "div_terms.h"
#include "fft_core.h"
#include "ola_kernels.h"
#include "prof.h"

namespace vmbd {

namespace {

// the angle a division works with: full for the difference filters of DIV_S
template <int OP>
__device__ __forceinline__ Freq div_freq(int q, int T, const float2* __restrict__ tw) {
  return OP == DIV_S ? full_freq(q, T, tw) : half_freq(q, T, tw);
}

__device__ __forceinline__ float cabs2(float2 a) { return fmaf(a.x, a.x, a.y * a.y); }
__device__ __forceinline__ float2 cdivr(float2 a, float d) { return make_float2(a.x / d, a.y / d); }

// Hermitian parts (D, N) of a packed transform P at frequency k, given P(-k)
__device__ __forceinline__ void split(float2 p, float2 q, float2& d, float2& n) {
  d = make_float2(0.5f * (p.x + q.x), 0.5f * (p.y - q.y));
  n = make_float2(0.5f * (p.y + q.y), 0.5f * (q.x - p.x));
}
__device__ __forceinline__ float2 join(float2 d, float2 n) { return make_float2(d.x - n.y, d.y + n.x); }

// the division of one (row bin, column frequency) from its operand values
// (order as in DivOp); hx: row bin, hy: column frequency
template <int OP>
__device__ __forceinline__ float2 div_value(const float2 (&o)[4], Freq hx, Freq hy, DivParams p) {
  if constexpr (OP == DIV_X) {
    const float L = four_sin2(hx) + four_sin2(hy);
    return cdivr(cmulc(o[0], o[1]), cabs2(o[1]) + p.alpha * L + p.beta);
  } else if constexpr (OP == DIV_G) {
    const float L = one_2cos_sq(hy) * four_sin2(hx) + four_sin2(hy) * one_2cos_sq(hx);
    const float2 num = cadd(cmulc(o[1], o[0]), cmulc(o[3], o[2]));
    return cdivr(num, cabs2(o[0]) + cabs2(o[2]) + p.alpha * L + p.beta);
  } else if constexpr (OP == DIV_SPROD) {
    return cmulc(o[0], o[1]);
  } else {
    const float2 gx = diff_filter(hx), gy = diff_filter(hy);
    const float ab = p.alpha * p.beta;
    const float2 num = cadd(cadd(cmulc(o[0], gx), cmulc(o[1], gy)), cdivr(o[2], ab));
    return cdivr(num, cabs2(o[3]) / ab + cabs2(gx) + cabs2(gy) + p.gamma);
  }
}

template <int OP>
struct DivArity {
  static constexpr int n = (OP == DIV_X || OP == DIV_SPROD) ? 2 : 4;
  // operand j is a cached spectrum
  static constexpr bool spec(int j) { return (OP == DIV_X || OP == DIV_SPROD) ? j == 1 : OP == DIV_S && j >= 2; }
};

template <int TH, int OP>
__global__ __launch_bounds__(WG, 2) void k_cols_div(Geo g, ColIn a0, ColIn a1, ColIn a2, ColIn a3, DivParams prm,
                                                   ColOut o, float2* __restrict__ spec_out,
                                                   const float2* __restrict__ tw) {
  constexpr int TPT = TH / 16;
  constexpr int CS = WG / TPT;  // columns per workgroup
  constexpr int SL = FftLds<TH>::floats2;
  constexpr int NA = DivArity<OP>::n;
  // FFT slices (aliased by the row staging of the store), then NA slices in
  // which the packed column's operand transforms are staged
  __shared__ float2 sm[cmax<CS * SL, TH * (CS + 1)>::v + NA * SL];
  float2* pk = sm + cmax<CS * SL, TH * (CS + 1)>::v;

  const int NB = g.NB;
  const int strip = blockIdx.x;
  const int pfr = blockIdx.z, pk_ = blockIdx.y;
  const int p = pfr * g.Pf + pk_;
  const int cc = threadIdx.x / TPT;
  const int t = threadIdx.x - cc * TPT;
  const int c = strip * CS + cc;
  const bool active = c < NB - 1;  // bins [0, NB-1); NB-1 travels packed in bin 0
  const bool packed = c == 0;
  const bool wact = strip * CS + (int)(threadIdx.x >> 6) * (64 / TPT) < NB - 1;
  const int pm = div_by(pk_, g.dcsf1);
  const int grp = pfr * g.csf1 + (pk_ - pm * g.csf1);
  const int row0 = pm * g.hop0;
  const ColCtx cx{pm, pk_ - pm * g.csf1, pfr, g.hop0, g.Tw, tw};
  float2* sl = sm + cc * SL;

  Twiddles<TH> T;
  twiddles_init<TH>(T, t, tw);

  // the column's row bin; the column frequencies, one table entry each, set up
  // in LDS for all columns of the workgroup beside the first operand's loads
  // (16 loads per thread are 256 per CU and round, 16 cycles each).  DIV_X keeps
  // the sines only, which leaves four workgroups per CU; DIV_G has registers for
  // its thread's entries up to 256 points.  us per call, 1024^2 / 700 x 900 (512
  // points): 'direct' 82.0 / 67.6, in registers 83.3 / 75; 'gdirect' in registers
  // 80.2, in LDS 82.0 / 54.9; 'sparse' 607 / 434, loaded where used 625 / 476.
  const Freq hx = div_freq<OP>(min(c, NB - 2), g.Tw, tw);
  constexpr bool SINE = OP == DIV_X, REG = OP == DIV_G && TH <= 256, LDS = !REG && OP != DIV_SPROD;
  __shared__ std::conditional_t<SINE, float, Freq> fq[LDS ? TH : 1];
  Freq own[REG ? 16 : 1];
  auto hy = [&](int m) {
    if constexpr (SINE)
      return Freq{fq[t + TPT * m], 0.f};
    else if constexpr (REG)
      return own[m];
    else
      return fq[t + TPT * m];
  };
  const ColIn ins[4] = {a0, a1, a2, a3};
  // Operands are consumed one at a time: transformed (row-pass outputs) or
  // loaded (spectra), staged when the column is the packed one, and folded
  // into the running numerator / denominator of the plain columns.
  float2 num[16], acc[16];
#pragma unroll
  for (int m = 0; m < 16; ++m) num[m] = acc[m] = make_float2(0.f, 0.f);
  float2 prev[16];
#pragma unroll
  for (int j = 0; j < NA; ++j) {
    float2 v[16];
    if (DivArity<OP>::spec(j)) {
      col_load_spec<TH>(v, ins[j], p, c, NB, t);
    } else {
      col_load<TH>(v, ins[j], p, c, NB, t, grp, row0, cx);
      if (REG && j == 0) {
#pragma unroll
        for (int m = 0; m < 16; ++m) own[REG ? m : 0] = div_freq<OP>(t + TPT * m, TH, tw);
      }
      if (LDS && j == 0) {
        for (int k = threadIdx.x; k < TH; k += WG) {
          const Freq h = div_freq<OP>(k, TH, tw);
          if constexpr (SINE)
            fq[k] = h.s;
          else
            fq[k] = h;
        }
        __syncthreads();
      }
      if (wact) fft<TH, -1>(v, sl, t, T);
    }
    if (packed) {
#pragma unroll
      for (int m = 0; m < 16; ++m) pk[j * SL + lds_pad(t + TPT * m)] = v[m];
    }
    // plain columns: keep what the formula needs (pairs for DIV_X / SPROD /
    // DIV_G, running sums for DIV_S)
    if constexpr (OP == DIV_S) {
      const float ab = prm.alpha * prm.beta;
#pragma unroll
      for (int m = 0; m < 16; ++m) {
        if (j == 0) num[m] = cmulc(v[m], diff_filter(hx));
        if (j == 1) num[m] = cadd(num[m], cmulc(v[m], diff_filter(hy(m))));
        if (j == 2) num[m] = cadd(num[m], cdivr(v[m], ab));
        if (j == 3) acc[m] = make_float2(cabs2(v[m]) / ab, 0.f);
      }
    } else if constexpr (OP == DIV_G) {
      if (j == 0 || j == 2) {
#pragma unroll
        for (int m = 0; m < 16; ++m) prev[m] = v[m];
      } else {
#pragma unroll
        for (int m = 0; m < 16; ++m) {
          num[m] = cadd(num[m], cmulc(v[m], prev[m]));
          acc[m].x += cabs2(prev[m]);
        }
      }
    } else {
      if (j == 0) {
#pragma unroll
        for (int m = 0; m < 16; ++m) prev[m] = v[m];
      } else {
#pragma unroll
        for (int m = 0; m < 16; ++m) {
          float2 ov[4] = {prev[m], v[m], make_float2(0.f, 0.f), make_float2(0.f, 0.f)};
          num[m] = div_value<OP>(ov, hx, hy(m), prm);
        }
      }
    }
  }
  float2 Z[16];
#pragma unroll
  for (int m = 0; m < 16; ++m) {
    if constexpr (OP == DIV_S) {
      const float2 gx = diff_filter(hx), gy = diff_filter(hy(m));
      Z[m] = cdivr(num[m], acc[m].x + cabs2(gx) + cabs2(gy) + prm.gamma);
    } else if constexpr (OP == DIV_G) {
      const Freq hk = hy(m);
      const float L = one_2cos_sq(hk) * four_sin2(hx) + four_sin2(hk) * one_2cos_sq(hx);
      Z[m] = cdivr(num[m], acc[m].x + prm.alpha * L + prm.beta);
    } else {
      Z[m] = num[m];
    }
  }
  if (packed) {
    // both Hermitian parts of every staged operand, the division of each
    // part (row bins 0 and Tw/2), the quotient packed again
    wave_sync();
#pragma unroll
    for (int m = 0; m < 16; ++m) {
      const int k = t + TPT * m;
      const int kr = (TH - k) & (TH - 1);
      float2 od[4], on[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        od[j] = on[j] = make_float2(0.f, 0.f);
        if (j < NA) split(pk[j * SL + lds_pad(k)], pk[j * SL + lds_pad(kr)], od[j], on[j]);
      }
      // row bins 0 and Tw/2: half angles 0 and pi/2, full 0 and pi
      constexpr Freq h0{0.f, 1.f}, h1 = OP == DIV_S ? Freq{0.f, -1.f} : Freq{1.f, 0.f};
      Z[m] = join(div_value<OP>(od, h0, hy(m), prm), div_value<OP>(on, h1, hy(m), prm));
    }
  }
  if constexpr (OP == DIV_SPROD) {
    if (active) {
      float2* col = spec_out + ((size_t)p * NB + c) * TH;
#pragma unroll
      for (int m = 0; m < 16; ++m) col[t + TPT * m] = Z[m];
      if (packed) {  // bin NB-1 travels in bin 0: its column is written as zeros
        float2* coln = spec_out + ((size_t)p * NB + NB - 1) * TH;
#pragma unroll
        for (int m = 0; m < 16; ++m) coln[t + TPT * m] = make_float2(0.f, 0.f);
      }
    }
  } else {
    if (wact) fft<TH, +1>(Z, sl, t, T);
    col_store_rows<TH, CS, true>(Z, sm, o, p, strip, NB, g.NBP, cc, t);
  }
}

template <int TH>
hipError_t cols_div_t(const Geo& g, int op, const ColIn* a, DivParams prm, const ColOut& o, float2* spec_out,
                      const float2* tw, hipStream_t st) {
  constexpr int CS = WG / (TH / 16);
  const int strips = (g.NB - 1 + CS - 1) / CS;
  const dim3 grid((unsigned)strips, (unsigned)g.Pf, (unsigned)(g.P / g.Pf));
  static const char* names[4] = {"cols_div_x", "cols_div_g", "cols_sprod", "cols_div_s"};
  ProfScope ps(names[op & 3], st);
  const ColOut po = col_out_policy(g, o);
  switch (op) {
    case DIV_X:
      hipLaunchKernelGGL((k_cols_div<TH, DIV_X>), grid, dim3(WG), 0, st, g, a[0], a[1], a[2], a[3], prm, po,
                         spec_out, tw);
      break;
    case DIV_G:
      hipLaunchKernelGGL((k_cols_div<TH, DIV_G>), grid, dim3(WG), 0, st, g, a[0], a[1], a[2], a[3], prm, po,
                         spec_out, tw);
      break;
    case DIV_SPROD:
      hipLaunchKernelGGL((k_cols_div<TH, DIV_SPROD>), grid, dim3(WG), 0, st, g, a[0], a[1], a[2], a[3], prm, po,
                         spec_out, tw);
      break;
    case DIV_S:
      hipLaunchKernelGGL((k_cols_div<TH, DIV_S>), grid, dim3(WG), 0, st, g, a[0], a[1], a[2], a[3], prm, po,
                         spec_out, tw);
      break;
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace

hipError_t launch_cols_div(const Geo& g, int op, const ColIn* a, int na, DivParams prm, const ColOut& o,
                           float2* spec_out, const float2* tw, hipStream_t st) {
  const int need = (op == DIV_X || op == DIV_SPROD) ? 2 : 4;
  if (na != need || g.P <= 0) return hipErrorInvalidValue;
  for (int j = 0; j < na; ++j) {  // spectra where the kernel reads spectra
    const bool spec = op == DIV_X || op == DIV_SPROD ? j == 1 : op == DIV_S && j >= 2;
    if ((a[j].spec != 0) != spec) return hipErrorInvalidValue;
  }
  ColIn in[4] = {a[0], a[1], ColIn{}, ColIn{}};
  if (na == 4) {
    in[2] = a[2];
    in[3] = a[3];
  }
  switch (g.Th) {
    case 16: return cols_div_t<16>(g, op, in, prm, o, spec_out, tw, st);
    case 32: return cols_div_t<32>(g, op, in, prm, o, spec_out, tw, st);
    case 64: return cols_div_t<64>(g, op, in, prm, o, spec_out, tw, st);
    case 128: return cols_div_t<128>(g, op, in, prm, o, spec_out, tw, st);
    case 256: return cols_div_t<256>(g, op, in, prm, o, spec_out, tw, st);
    case 512: return cols_div_t<512>(g, op, in, prm, o, spec_out, tw, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace vmbd
