// Image stencils and pointwise filters of the deconvolution path for gfx950
// (kernel.cu, edgetaper.cu, resize.cu of the reference).
//
// Every stencil reads its input and writes a separate output (Jacobi
// semantics): the reference's shock and bilateral kernels update the image
// in place while neighbouring blocks still read their halos (kernel.cu:86,
// 134).  Border handling follows the reference kernels exactly:
//   shock      top/left rows and columns replicate, bottom/right read 0 (kernel.cu:22-30)
//   bilateral  out-of-image neighbours are skipped (kernel.cu:124)
//   laplace    'valid' or zero border ('same')
// 16x16 workgroups tile the image; the bilateral filter stages its tile and
// halo in LDS (121 taps per pixel).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "../../include/vmbd_filters.h"
#include "capi_util.h"
#include "prof.h"

namespace vmbd {
namespace {

constexpr int BX = 16, BY = 16;

inline dim3 grid2(int rows, int cols) { return dim3((cols + BX - 1) / BX, (rows + BY - 1) / BY); }

__device__ __forceinline__ float at_shock(const float* a, int H, int W, int i, int j) {
  // kernel.cu:20-30: negative indices clamp to 0, indices past the end read 0
  if (i < 0) i = 0;
  if (j < 0) j = 0;
  if (i >= H || j >= W) return 0.f;
  return a[(long long)i * W + j];
}

// one Osher-Rudin shock step (kernel.cu:36-86)
__global__ __launch_bounds__(BX* BY) void k_shock(float* out, const float* a, int H, int W, float dt, float h) {
  const int i = blockIdx.y * BY + threadIdx.y, j = blockIdx.x * BX + threadIdx.x;
  if (i >= H || j >= W) return;
  const float c = at_shock(a, H, W, i, j);
  const float l = at_shock(a, H, W, i, j - 1), r = at_shock(a, H, W, i, j + 1);
  const float u = at_shock(a, H, W, i - 1, j), d = at_shock(a, H, W, i + 1, j);
  float t1 = -c + r, t2 = c - l;
  const float Ix = (t1 + t2) / 2.f;
  float mx = (t1 * t2 < 0.f) ? 0.f : fminf(fabsf(t1), fabsf(t2));
  t1 = -c + d;
  t2 = c - u;
  const float Iy = (t1 + t2) / 2.f;
  float my = (t1 * t2 < 0.f) ? 0.f : fminf(fabsf(t1), fabsf(t2));
  const float flow = sqrtf(mx * mx + my * my);
  const float Ixx = r + l - 2.f * c;
  const float Iyy = d + u - 2.f * c;
  const float Ixy = (at_shock(a, H, W, i + 1, j + 1) - at_shock(a, H, W, i + 1, j - 1) -
                     at_shock(a, H, W, i - 1, j + 1) + at_shock(a, H, W, i - 1, j - 1)) /
                    4.f;
  float Inn = (Iyy * Iy * Iy + 2.f * Ixy * Iy * Ix + Ixx * Ix * Ix) / (Ix * Ix + Iy * Iy + 0.00000001f);
  if (Ix == 0.f && Iy == 0.f) Inn = Ixx;
  out[(long long)i * W + j] = c - dt * copysignf(flow, Inn) / h;
}

// bilateral filter (kernel.cu:90-136), tile + halo in LDS (dynamic size)
__global__ __launch_bounds__(BX* BY) void k_bfilter(float* out, const float* a, int H, int W, int w, float sd,
                                                    float sr) {
  extern __shared__ float tile[];
  const int TW = BX + 2 * w, TH = BY + 2 * w;
  const int i0 = blockIdx.y * BY - w, j0 = blockIdx.x * BX - w;
  for (int idx = threadIdx.y * BX + threadIdx.x; idx < TW * TH; idx += BX * BY) {
    const int ti = idx / TW, tj = idx - (idx / TW) * TW;
    const int ii = i0 + ti, jj = j0 + tj;
    tile[idx] = (ii >= 0 && ii < H && jj >= 0 && jj < W) ? a[(long long)ii * W + jj] : 0.f;
  }
  __syncthreads();
  const int i = blockIdx.y * BY + threadIdx.y, j = blockIdx.x * BX + threadIdx.x;
  if (i >= H || j >= W) return;
  const float c = tile[(threadIdx.y + w) * TW + threadIdx.x + w];
  const float inv_r = 1.f / (2.f * sr * sr), inv_d = 1.f / (2.f * sd * sd);
  float sw = 0.f, acc = 0.f;
  for (int x = -w; x <= w; ++x) {
    for (int y = -w; y <= w; ++y) {
      if (i + y >= 0 && i + y < H && j + x >= 0 && j + x < W) {
        const float v = tile[(threadIdx.y + w + y) * TW + threadIdx.x + w + x];
        const float dv = v - c;
        const float wt = expf(-(dv * dv * inv_r + (float)(x * x + y * y) * inv_d));
        sw += wt;
        acc += wt * v;
      }
    }
  }
  out[(long long)i * W + j] = acc / sw;
}

// The same filter for a half size WR known at compile time (the MFBD prior's
// w = 5), R pixels of one column per thread, 64 columns x 4R rows per
// workgroup: a column of 2 WR + R values is read from LDS once for its R
// pixels, the spatial factor is folded into one exponent, exp(-t) evaluated as
// the hardware 2^(-t log2 e).  Bound by VALU issue: five instructions and one
// quarter-rate exponential per tap.  The in-image test is made only in
// workgroups whose window crosses the image border, in code of its own: inside
// one unrolled loop it was a branch per tap, 121 blocks that overlapped nothing
// and 242 registers (two wavefronts per SIMD); 2048^2 took 229 us, this
// 104.  Same sums in the same order as k_bfilter.
constexpr int BFX = 64;
template <int WR, int R, bool EDGE>
__device__ __forceinline__ void bfilter_taps(const float* tc, int i0, int j, int H, int W, float kr, float kd,
                                             float (&sw)[R], float (&acc)[R]) {
  constexpr int TW = BFX + 2 * WR;
  float c[R];
#pragma unroll
  for (int q = 0; q < R; ++q) {
    c[q] = tc[q * TW];
    sw[q] = acc[q] = 0.f;
  }
#pragma unroll 1
  for (int x = -WR; x <= WR; ++x) {
    if (EDGE && (j + x < 0 || j + x >= W)) continue;
    float v[R + 2 * WR];
#pragma unroll
    for (int r = 0; r < R + 2 * WR; ++r) v[r] = tc[(r - WR) * TW + x];
#pragma unroll
    for (int y = -WR; y <= WR; ++y) {
      const float sp = (float)(x * x + y * y) * kd;
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const float dv = v[q + y + WR] - c[q];
        float wt = __builtin_amdgcn_exp2f(fmaf(dv * dv, kr, sp));
        if (EDGE) wt = (i0 + q + y >= 0 && i0 + q + y < H) ? wt : 0.f;
        sw[q] += wt;
        acc[q] += wt * v[q + y + WR];
      }
    }
  }
}

template <int WR, int R>
__global__ __launch_bounds__(256) void k_bfilter_w(float* out, const float* a, int H, int W, float sd, float sr) {
  constexpr int TW = BFX + 2 * WR, TH = 4 * R + 2 * WR;
  __shared__ float tile[TW * TH];
  const int ti0 = blockIdx.y * 4 * R - WR, tj0 = blockIdx.x * BFX - WR;
  for (int idx = threadIdx.x; idx < TW * TH; idx += 256) {
    const int ti = idx / TW, tj = idx - (idx / TW) * TW;
    const int ii = ti0 + ti, jj = tj0 + tj;
    tile[idx] = (ii >= 0 && ii < H && jj >= 0 && jj < W) ? a[(long long)ii * W + jj] : 0.f;
  }
  __syncthreads();
  const int lj = threadIdx.x & (BFX - 1), li = (int)(threadIdx.x / BFX) * R;
  const int i0 = blockIdx.y * 4 * R + li, j = blockIdx.x * BFX + lj;
  if (i0 >= H || j >= W) return;
  const float* tc = tile + (li + WR) * TW + lj + WR;
  constexpr float LOG2E = 1.44269504088896340736f;
  const float kr = -LOG2E / (2.f * sr * sr), kd = -LOG2E / (2.f * sd * sd);
  float sw[R], acc[R];
  if (ti0 >= 0 && tj0 >= 0 && ti0 + TH <= H && tj0 + TW <= W)  // uniform per workgroup
    bfilter_taps<WR, R, false>(tc, i0, j, H, W, kr, kd, sw, acc);
  else
    bfilter_taps<WR, R, true>(tc, i0, j, H, W, kr, kd, sw, acc);
#pragma unroll
  for (int q = 0; q < R; ++q)
    if (i0 + q < H) out[(long long)(i0 + q) * W + j] = acc[q] / sw[q];
}

#define SQRT2H 0.70710678118654752440f

// kernel.cu:180-242
__global__ __launch_bounds__(BX* BY) void k_gradient(float* gx, float* gy, const float* y, int H, int W, int same) {
  const int i = blockIdx.y * BY + threadIdx.y, j = blockIdx.x * BX + threadIdx.x;
  if (i >= H || j >= W) return;
  const float c = y[(long long)i * W + j];
  if (same) {
    gy[(long long)i * W + j] = (i < H - 1) ? SQRT2H * (c - y[(long long)(i + 1) * W + j]) : 0.f;
    gx[(long long)i * W + j] = (j < W - 1) ? SQRT2H * (c - y[(long long)i * W + j + 1]) : 0.f;
  } else {
    if (i < H - 1) gy[(long long)i * W + j] = SQRT2H * (c - y[(long long)(i + 1) * W + j]);
    if (j < W - 1) gx[(long long)i * (W - 1) + j] = SQRT2H * (c - y[(long long)i * W + j + 1]);
  }
}

// kernel.cu:244-266: replicate padding, (top, left) = floor(sf/2)
__global__ __launch_bounds__(BX* BY) void k_impad(float* out, int OH, int OW, const float* im, int H, int W, int top,
                                                  int left) {
  const int i = blockIdx.y * BY + threadIdx.y, j = blockIdx.x * BX + threadIdx.x;
  if (i >= OH || j >= OW) return;
  int si = i - top, sj = j - left;
  si = si < 0 ? 0 : (si >= H ? H - 1 : si);
  sj = sj < 0 ? 0 : (sj >= W ? W - 1 : sj);
  out[(long long)i * OW + j] = im[(long long)si * W + sj];
}

#define LAP_N 0.22360679774997896964f  // 1/sqrt(20)
#define LAP_C 0.89442719099991587856f  // 4/sqrt(20)

// kernel.cu:268-333 (per slice of a stack of K images); zero_k: the first and
// last slice are zero (laplace_stack_same, kernel.cu:364)
__global__ __launch_bounds__(BX* BY) void k_laplace(float* out, const float* im, int H, int W, int same, int K,
                                                    int zero_k) {
  const int i = blockIdx.y * BY + threadIdx.y, j = blockIdx.x * BX + threadIdx.x;
  const int k = blockIdx.z;
  const float* s = im + (long long)k * H * W;
  if (same) {
    if (i >= H || j >= W) return;
    float v = 0.f;
    const bool kin = !zero_k || (k > 0 && k < K - 1);
    if (kin && i > 0 && i < H - 1 && j > 0 && j < W - 1) {
      const long long c = (long long)i * W + j;
      v = -LAP_N * (s[c + W] + s[c - W] + s[c + 1] + s[c - 1]) + LAP_C * s[c];
    }
    out[(long long)k * H * W + (long long)i * W + j] = v;
  } else {
    if (i >= H - 2 || j >= W - 2) return;
    const long long c = (long long)(i + 1) * W + j + 1;
    out[(long long)k * (H - 2) * (W - 2) + (long long)i * (W - 2) + j] =
        -LAP_N * (s[c + W] + s[c - W] + s[c + 1] + s[c - 1]) + LAP_C * s[c];
  }
}

// kernel.cu:377-418: 7-point 3-D Laplacian, zero on every face
__global__ __launch_bounds__(BX* BY) void k_laplace3d(float* out, const float* im, int D, int H, int W) {
  const int i = blockIdx.y * BY + threadIdx.y, j = blockIdx.x * BX + threadIdx.x;
  const int k = blockIdx.z;
  if (i >= H || j >= W) return;
  const long long HW = (long long)H * W;
  const long long c = k * HW + (long long)i * W + j;
  float v = 0.f;
  if (i > 0 && i < H - 1 && j > 0 && j < W - 1 && k > 0 && k < D - 1)
    v = -(im[c + W] + im[c - W] + im[c + 1] + im[c - 1] + im[c + HW] + im[c - HW]) + 6.f * im[c];
  out[c] = v;
}

// hyper-Laplacian w-step, alpha = 2/3 (kernel.cu:555-578)
__global__ __launch_bounds__(256) void k_alpha23(float* y, long long n, float beta) {
  const long long e = (long long)blockIdx.x * 256 + threadIdx.x;
  if (e >= n) return;
  const float v = y[e];
  float x = v;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float t1 = (2.f / 3.f) / cbrtf(fabsf(x));
    x -= (copysignf(t1, x) + beta * (x - v)) / (t1 / (-3.f * fabsf(x)) + beta);
  }
  if (!isfinite(x)) x = 0.f;
  float t = cbrtf(fabsf(x));
  t *= t;
  if (t + beta * 0.5f * (x - v) * (x - v) > beta * 0.5f * v * v) x = 0.f;
  y[e] = x;
}

// general-alpha w-step (kernel.cu:529-553)
__global__ __launch_bounds__(256) void k_alpha(float* y, long long n, float beta, float alpha) {
  const long long e = (long long)blockIdx.x * 256 + threadIdx.x;
  if (e >= n) return;
  const float v = y[e];
  float x = v;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float fd = alpha * (x > 0.f ? 1.f : -1.f) * powf(fabsf(x), alpha - 1.f) + beta * (x - v);
    const float fdd = alpha * (alpha - 1.f) * powf(fabsf(x), alpha - 2.f) + beta;
    x -= fd / fdd;
  }
  if (!isfinite(x)) x = 0.f;
  if (powf(fabsf(x), alpha) + beta * 0.5f * (x - v) * (x - v) > beta * 0.5f * v * v) x = 0.f;
  y[e] = x;
}

// edgetaper.cu:6-31 (tables already divided by max(wx)*max(wy) on the host)
__global__ __launch_bounds__(BX* BY) void k_edgetaper(float* im, int H, int W, const float* wx, int hx,
                                                      const float* wy, int hy) {
  const int i = blockIdx.y * BY + threadIdx.y, j = blockIdx.x * BX + threadIdx.x;
  if (i >= H || j >= W) return;
  if (!(i < hy || i > H - 1 - hy || j < hx || j > W - 1 - hx)) return;
  float v = im[(long long)i * W + j];
  if (i < hy) v *= wy[i];
  else if (i > H - 1 - hy) v *= wy[H - 1 - i];
  if (j < hx) v *= wx[j];
  else if (j > W - 1 - hx) v *= wx[W - 1 - j];
  im[(long long)i * W + j] = v;
}

// The same taper with its tables as kernel arguments (tables computed per
// call on the host need no copy to the device, which would wait for the
// stream's earlier work).
constexpr int TAPER_MAX = 128;
struct TaperTab {
  int hx, hy;
  float wx[TAPER_MAX], wy[TAPER_MAX];
};
__device__ __forceinline__ float taper_at(const TaperTab& t, float v, int i, int j, int H, int W) {
  if (i < t.hy) v *= t.wy[i];
  else if (i > H - 1 - t.hy) v *= t.wy[H - 1 - i];
  if (j < t.hx) v *= t.wx[j];
  else if (j > W - 1 - t.hx) v *= t.wx[W - 1 - j];
  return v;
}
__global__ __launch_bounds__(BX* BY) void k_edgetaper_tab(float* im, int H, int W, TaperTab t) {
  const int i = blockIdx.y * BY + threadIdx.y, j = blockIdx.x * BX + threadIdx.x;
  if (i >= H || j >= W) return;
  if (!(i < t.hy || i > H - 1 - t.hy || j < t.hx || j > W - 1 - t.hx)) return;
  im[(long long)i * W + j] = taper_at(t, im[(long long)i * W + j], i, j, H, W);
}

// The end of 'direct' (olaGPU.py:531-546) in one pass: max(num, 0) over the
// tapered den clipped to [0.01, 10], its inner rows [o0, o0 + m) and columns
// [o1, o1 + n) replicated outwards to H x W (p0, p1: first inner row and
// column of the result).  As six passes it read and wrote the image eleven
// times.
__global__ __launch_bounds__(BX* BY) void k_direct_ratio(float* out, const float* num, const float* den, int H, int W,
                                                         int o0, int o1, int m, int n, int p0, int p1, TaperTab t) {
  const int i = blockIdx.y * BY + threadIdx.y, j = blockIdx.x * BX + threadIdx.x;
  if (i >= H || j >= W) return;
  const int si = o0 + min(max(i - p0, 0), m - 1), sj = o1 + min(max(j - p1, 0), n - 1);
  float a = num[(long long)si * W + sj];
  a = a < 0.f ? 0.f : a;
  float d = taper_at(t, den[(long long)si * W + sj], si, sj, H, W);
  d = d < 0.01f ? 0.01f : d;
  d = d > 10.f ? 10.f : d;
  out[(long long)i * W + j] = a / d;
}

// Taper tables of a PSF size (edgetaper_windows in gputools.py): the sizes
// made odd, the rising halves of two Bartlett-Hann windows over the product
// of their maxima.  False when they do not fit the kernel arguments.
bool taper_tab(TaperTab& t, int s0, int s1) {
  const int n1 = s1 + 1 - s1 % 2, n0 = s0 + 1 - s0 % 2;
  t.hx = n1 / 2;
  t.hy = n0 / 2;
  if (s0 <= 0 || s1 <= 0 || t.hx > TAPER_MAX || t.hy > TAPER_MAX) return false;
  auto win = [](int k, int n) {
    if (n <= 1) return 1.0;
    const double fac = std::fabs((double)k / (double)n - 0.5);
    return 0.62 - 0.48 * fac + 0.38 * std::cos(2.0 * M_PI * fac);
  };
  auto top = [&](int n) {
    double m = 0.0;
    for (int k = 0; k < n; ++k) m = std::max(m, win(k, n));
    return m;
  };
  const double mx = top(n1) * top(n0);
  for (int k = 0; k < t.hx; ++k) t.wx[k] = (float)(win(k, n1) / mx);
  for (int k = 0; k < t.hy; ++k) t.wy[k] = (float)(win(k, n0) / mx);
  return true;
}

// resize.cu:5-15: sample at normalised (j/OW, i/OH) with bilinear filtering
// and clamp addressing (texel centres at +0.5), per slice
__global__ __launch_bounds__(BX* BY) void k_resize(float* out, int OH, int OW, const float* in, int H, int W) {
  const int i = blockIdx.y * BY + threadIdx.y, j = blockIdx.x * BX + threadIdx.x;
  const int k = blockIdx.z;
  if (i >= OH || j >= OW) return;
  const float* s = in + (long long)k * H * W;
  const float xs = (float)j / (float)OW * (float)W - 0.5f;
  const float ys = (float)i / (float)OH * (float)H - 0.5f;
  const float fx = floorf(xs), fy = floorf(ys);
  const float ax = xs - fx, ay = ys - fy;
  auto cl = [](int v, int n) { return v < 0 ? 0 : (v >= n ? n - 1 : v); };
  const int x0 = cl((int)fx, W), x1 = cl((int)fx + 1, W);
  const int y0 = cl((int)fy, H), y1 = cl((int)fy + 1, H);
  const float t0 = s[(long long)y0 * W + x0] * (1.f - ax) + s[(long long)y0 * W + x1] * ax;
  const float t1 = s[(long long)y1 * W + x0] * (1.f - ax) + s[(long long)y1 * W + x1] * ax;
  out[(long long)k * OH * OW + (long long)i * OW + j] = t0 * (1.f - ay) + t1 * ay;
}

}  // namespace
}  // namespace vmbd

using namespace vmbd;

#define FILT_DONE(what)                                              \
  do {                                                               \
    hipError_t e__ = hipGetLastError();                              \
    if (e__ != hipSuccess) return vmbd_fail_hip(what, e__);          \
    return VMBD_OK;                                                  \
  } while (0)

extern "C" {

int vmbd_shock_step(float* out, const float* in, int32_t H, int32_t W, float dt, float h, vmbd_stream_t stream) {
  vmbd_clear_error();
  if (!out || !in || out == in || H <= 0 || W <= 0) return vmbd_fail(VMBD_E_ARG, "vmbd_shock_step: bad argument");
  hipStream_t st = (hipStream_t)stream;
  ProfScope ps("shock", st);
  hipLaunchKernelGGL(k_shock, grid2(H, W), dim3(BX, BY), 0, st, out, in, H, W, dt, h);
  FILT_DONE("vmbd_shock_step");
}

int vmbd_bilateral(float* out, const float* in, int32_t H, int32_t W, int32_t w, float sigma_d, float sigma_r,
                   vmbd_stream_t stream) {
  vmbd_clear_error();
  if (!out || !in || out == in || H <= 0 || W <= 0 || w < 0 || w > 24)
    return vmbd_fail(VMBD_E_ARG, "vmbd_bilateral: bad argument (half size in [0,24], out != in)");
  hipStream_t st = (hipStream_t)stream;
  const size_t shm = (size_t)(BX + 2 * w) * (BY + 2 * w) * sizeof(float);
  ProfScope ps("bilateral", st);
  // four pixels per thread from two workgroups per CU on (at 512 x 1024 and
  // above), one where that would leave CUs without work
  const dim3 g4((W + BFX - 1) / BFX, (H + 15) / 16), g1((W + BFX - 1) / BFX, (H + 3) / 4);
  if (w == 5 && (long long)g4.x * g4.y >= 512)
    hipLaunchKernelGGL((k_bfilter_w<5, 4>), g4, dim3(256), 0, st, out, in, H, W, sigma_d, sigma_r);
  else if (w == 5 && g1.y <= 65535)
    hipLaunchKernelGGL((k_bfilter_w<5, 1>), g1, dim3(256), 0, st, out, in, H, W, sigma_d, sigma_r);
  else
    hipLaunchKernelGGL(k_bfilter, grid2(H, W), dim3(BX, BY), shm, st, out, in, H, W, w, sigma_d, sigma_r);
  FILT_DONE("vmbd_bilateral");
}

int vmbd_gradient(float* gx, float* gy, const float* y, int32_t H, int32_t W, int32_t same, vmbd_stream_t stream) {
  vmbd_clear_error();
  if (!gx || !gy || !y || H <= 1 || W <= 1) return vmbd_fail(VMBD_E_ARG, "vmbd_gradient: bad argument");
  hipStream_t st = (hipStream_t)stream;
  ProfScope ps("gradient", st);
  hipLaunchKernelGGL(k_gradient, grid2(H, W), dim3(BX, BY), 0, st, gx, gy, y, H, W, same);
  FILT_DONE("vmbd_gradient");
}

int vmbd_impad(float* out, const float* in, int32_t H, int32_t W, int32_t padh, int32_t padw, vmbd_stream_t stream) {
  vmbd_clear_error();
  if (!out || !in || H <= 0 || W <= 0 || padh < 0 || padw < 0) return vmbd_fail(VMBD_E_ARG, "vmbd_impad: bad argument");
  hipStream_t st = (hipStream_t)stream;
  const int OH = H + padh, OW = W + padw;
  ProfScope ps("impad", st);
  hipLaunchKernelGGL(k_impad, grid2(OH, OW), dim3(BX, BY), 0, st, out, OH, OW, in, H, W, padh / 2, padw / 2);
  FILT_DONE("vmbd_impad");
}

int vmbd_laplace(float* out, const float* in, int32_t K, int32_t H, int32_t W, int32_t same, int32_t zero_end_slices,
                 vmbd_stream_t stream) {
  vmbd_clear_error();
  if (!out || !in || K <= 0 || H <= 2 || W <= 2) return vmbd_fail(VMBD_E_ARG, "vmbd_laplace: bad argument");
  hipStream_t st = (hipStream_t)stream;
  dim3 g = grid2(H, W);
  g.z = K;
  ProfScope ps("laplace", st);
  hipLaunchKernelGGL(k_laplace, g, dim3(BX, BY), 0, st, out, in, H, W, same, K, zero_end_slices);
  FILT_DONE("vmbd_laplace");
}

int vmbd_laplace3d(float* out, const float* in, int32_t D, int32_t H, int32_t W, vmbd_stream_t stream) {
  vmbd_clear_error();
  if (!out || !in || D <= 0 || H <= 0 || W <= 0) return vmbd_fail(VMBD_E_ARG, "vmbd_laplace3d: bad argument");
  hipStream_t st = (hipStream_t)stream;
  dim3 g = grid2(H, W);
  g.z = D;
  ProfScope ps("laplace3d", st);
  hipLaunchKernelGGL(k_laplace3d, g, dim3(BX, BY), 0, st, out, in, D, H, W);
  FILT_DONE("vmbd_laplace3d");
}

int vmbd_shrink_alpha23(float* y, int64_t n, float beta, vmbd_stream_t stream) {
  vmbd_clear_error();
  if (!y || n < 0) return vmbd_fail(VMBD_E_ARG, "vmbd_shrink_alpha23: bad argument");
  if (n == 0) return VMBD_OK;
  hipStream_t st = (hipStream_t)stream;
  ProfScope ps("shrink23", st);
  hipLaunchKernelGGL(k_alpha23, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, y, (long long)n, beta);
  FILT_DONE("vmbd_shrink_alpha23");
}

int vmbd_shrink_alpha(float* y, int64_t n, float beta, float alpha, vmbd_stream_t stream) {
  vmbd_clear_error();
  if (!y || n < 0) return vmbd_fail(VMBD_E_ARG, "vmbd_shrink_alpha: bad argument");
  if (n == 0) return VMBD_OK;
  hipStream_t st = (hipStream_t)stream;
  ProfScope ps("shrink", st);
  hipLaunchKernelGGL(k_alpha, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, y, (long long)n, beta, alpha);
  FILT_DONE("vmbd_shrink_alpha");
}

int vmbd_edgetaper(float* im, int32_t H, int32_t W, const float* wx, int32_t hx, const float* wy, int32_t hy,
                   vmbd_stream_t stream) {
  vmbd_clear_error();
  if (!im || H <= 0 || W <= 0 || hx < 0 || hy < 0 || (hx && !wx) || (hy && !wy))
    return vmbd_fail(VMBD_E_ARG, "vmbd_edgetaper: bad argument");
  hipStream_t st = (hipStream_t)stream;
  ProfScope ps("edgetaper", st);
  hipLaunchKernelGGL(k_edgetaper, grid2(H, W), dim3(BX, BY), 0, st, im, H, W, wx, hx, wy, hy);
  FILT_DONE("vmbd_edgetaper");
}

int vmbd_edgetaper_psf(float* im, int32_t H, int32_t W, int32_t s0, int32_t s1, vmbd_stream_t stream) {
  vmbd_clear_error();
  TaperTab t;
  if (!im || H <= 0 || W <= 0 || s0 <= 0 || s1 <= 0) return vmbd_fail(VMBD_E_ARG, "vmbd_edgetaper_psf: bad argument");
  if (!taper_tab(t, s0, s1))
    return vmbd_fail(VMBD_E_UNSUP, "vmbd_edgetaper_psf: %d x %d tapers more than %d rows or columns", s0, s1, TAPER_MAX);
  hipStream_t st = (hipStream_t)stream;
  ProfScope ps("edgetaper", st);
  hipLaunchKernelGGL(k_edgetaper_tab, grid2(H, W), dim3(BX, BY), 0, st, im, H, W, t);
  FILT_DONE("vmbd_edgetaper_psf");
}

int vmbd_direct_ratio(float* out, const float* num, const float* den, int32_t H, int32_t W, int32_t s0, int32_t s1,
                      int32_t o0, int32_t o1, int32_t m, int32_t n, vmbd_stream_t stream) {
  vmbd_clear_error();
  TaperTab t;
  if (!out || !num || !den || H <= 0 || W <= 0 || s0 <= 0 || s1 <= 0 || o0 < 0 || o1 < 0 || m <= 0 || n <= 0 ||
      o0 + m > H || o1 + n > W)
    return vmbd_fail(VMBD_E_ARG, "vmbd_direct_ratio: bad argument");
  if (!taper_tab(t, s0, s1))
    return vmbd_fail(VMBD_E_UNSUP, "vmbd_direct_ratio: %d x %d tapers more than %d rows or columns", s0, s1, TAPER_MAX);
  hipStream_t st = (hipStream_t)stream;
  ProfScope ps("direct_ratio", st);
  hipLaunchKernelGGL(k_direct_ratio, grid2(H, W), dim3(BX, BY), 0, st, out, num, den, H, W, o0, o1, m, n, (H - m) / 2,
                     (W - n) / 2, t);
  FILT_DONE("vmbd_direct_ratio");
}

int vmbd_resize(float* out, int32_t OH, int32_t OW, const float* in, int32_t K, int32_t H, int32_t W,
                vmbd_stream_t stream) {
  vmbd_clear_error();
  if (!out || !in || OH <= 0 || OW <= 0 || K <= 0 || H <= 0 || W <= 0)
    return vmbd_fail(VMBD_E_ARG, "vmbd_resize: bad argument");
  hipStream_t st = (hipStream_t)stream;
  dim3 g = grid2(OH, OW);
  g.z = K;
  ProfScope ps("resize", st);
  hipLaunchKernelGGL(k_resize, g, dim3(BX, BY), 0, st, out, OH, OW, in, H, W);
  FILT_DONE("vmbd_resize");
}

}  // extern "C"
