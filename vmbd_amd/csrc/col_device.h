// Device helpers shared by the column-pass kernels (ola_kernels.hip,
// deconv_kernels.hip): workgroup size, the column loads of row-pass output or
// cached spectra, and the staged row-major store of a strip's columns.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "fft_core.h"
#include "ola_kernels.h"

namespace vmbd {

constexpr int WG = 256;
constexpr int NXCD = 8;  // XCDs of an MI355X; workgroups are dealt to them round-robin

// NT: a store for data that passes through memory once between two launches;
// it leaves the L2 to the operands that are read again.
typedef float float2_nt __attribute__((ext_vector_type(2)));
template <bool NT>
__device__ __forceinline__ void store_f2(float2* p, float2 v) {
  if constexpr (NT)
    __builtin_nontemporal_store((float2_nt){v.x, v.y}, (float2_nt*)p);
  else
    *p = v;
}

template <int A, int B>
struct cmax {
  static constexpr int v = A > B ? A : B;
};

// 16-byte global load of 4 consecutive floats at a 4-byte-aligned address
// (gfx950 vector memory accepts unaligned addresses)
__device__ __forceinline__ void ld4(float (&d)[4], const float* p) { __builtin_memcpy(d, p, 16); }

// Slots of a column against the operand's stored rows [rlo, rlo + nr): bit r
// of `full` where all TPT rows of slot r are stored, of `part` where some
// are.  Both are uniform, so the loads below branch on the scalar unit.
struct ColSlots {
  unsigned full, part;
};
template <int TPT>
__device__ __forceinline__ ColSlots col_slots(int rlo, int nr) {
  const int hi = rlo + nr;
  const unsigned in = (1u << (hi / TPT)) - 1u, some = (1u << ((hi + TPT - 1) / TPT)) - 1u;
  ColSlots m;
  m.full = in & ~((1u << ((rlo + TPT - 1) / TPT)) - 1u);
  m.part = some & ~((1u << (rlo / TPT)) - 1u) & ~m.full;
  return m;
}

// Slot r of a column from base[vo + TPT*r] (T: float2 rows, or their float
// factors): a full slot is a plain load at an immediate offset, a partial one
// (at most two per column) takes a lane mask, the others are zero.
template <int TPT, class T>
__device__ __forceinline__ void col_slot(T& v, const T* base, unsigned vo, int t, int r, int rlo, int nr, ColSlots m) {
  v = T{};
  if (m.full >> r & 1) v = (base + vo)[TPT * r];
  if (m.part >> r & 1) {
    asm volatile("");  // keeps this block a scalar branch, not lane selects in every slot
    const int rr = t + TPT * r - rlo;
    if (rr >= 0 && rr < nr) v = (base + vo)[TPT * r];
  }
}

// Column c of a cached spectrum.  Here and below, addresses are a uniform
// base plus one 32-bit lane offset, and columns past the last bin read the
// last one (their results are never stored): 6-8 VALU instructions per slot
// less than with a masked 64-bit address of its own.
template <int TH>
__device__ __forceinline__ void col_load_spec(float2 (&v)[16], const ColIn& in, int p, int c, int NB, int t) {
  constexpr int TPT = TH / 16;
  const float2* base = in.p + (size_t)p * NB * TH;
  const unsigned vo = (unsigned)min(c, NB - 2) * TH + t;
#pragma unroll
  for (int r = 0; r < 16; ++r) v[r] = (base + vo)[TPT * r];
}

// Column c of row-pass output in the FFT input mapping.  NZ < 16: only slots
// r < NZ can hold stored rows (rlo + nr <= NZ*TPT); the others are left unset
// (the transform does not read them).  XS: shared image rows, each scaled by
// its patch row's factor in.rsc.
template <int TH, int NZ = 16, bool XS = false>
__device__ __forceinline__ void col_load(float2 (&v)[16], const ColIn& in, int p, int c, int NB, int t, int grp,
                                         int row0, const ColCtx& cx) {
  constexpr int TPT = TH / 16;
  const float2* base =
      (in.shared ? in.p + (size_t)grp * NB * in.pitch + row0 : in.p + (size_t)p * NB * in.pitch) - in.rlo;
  const unsigned vo = (unsigned)min(c, NB - 2) * (unsigned)in.pitch + t;
  const ColSlots m = col_slots<TPT>(in.rlo, in.nr);
  if constexpr (!XS) {
#pragma unroll
    for (int r = 0; r < NZ; ++r) col_slot<TPT>(v[r], base, vo, t, r, in.rlo, in.nr, m);
  } else {
    const float* rs = in.rsc + (size_t)cx.pm * in.nr - in.rlo;
    float sc[NZ];
#pragma unroll
    for (int r = 0; r < NZ; ++r) {
      col_slot<TPT>(sc[r], rs, (unsigned)t, t, r, in.rlo, in.nr, m);
      col_slot<TPT>(v[r], base, vo, t, r, in.rlo, in.nr, m);
    }
#pragma unroll
    for (int r = 0; r < NZ; ++r) {
      v[r].x *= sc[r];
      v[r].y *= sc[r];
    }
    // floor columns at the canvas edge: the pixel's own term, at its row's
    // weight (no patch-row factor), as bin c of a unit impulse at column ec:
    // e^{-2 pi i c ec / Tw}; the packed column holds bins 0 and Tw/2
    // (factors 1 and (-1)^ec)
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int ecol = e ? in.ecol[1] : in.ecol[0];
      const int en = e ? in.en[1] : in.en[0];
      const int ec = e ? in.ec[1] : in.ec[0];
      if (in.ex && ecol >= 0 && cx.pn == en) {
        // row q of the operand's term sits in lane q % 64 of table register
        // q / 64 (one gather per 64 rows) and reaches the lanes that hold it
        // in a transform by a cross-lane permute
        constexpr int K = (TPT * NZ + 63) / 64;
        const int lane = threadIdx.x & 63;
        float tab[K];
        const float* xf = in.ex + (size_t)cx.pfr * in.exf + ecol;
#pragma unroll
        for (int k = 0; k < K; ++k) {
          const int q = 64 * k + lane - in.rlo;
          const int u = cx.pm * cx.hop0 + q;
          tab[k] = (q >= 0 && q < in.nr && u < in.exH) ? xf[(size_t)u * in.exld] * in.einv[u] : 0.f;
        }
        const float2 E = c == 0 ? make_float2(1.f, (ec & 1) ? -1.f : 1.f)
                                : cx.tw[((long long)c * ec * (TW_LEN / cx.Tw)) & (TW_LEN - 1)];
#pragma unroll
        for (int r = 0; r < NZ; ++r) {
          const float dl = __shfl(tab[(TPT * r) / 64], (TPT * r) % 64 + t, 64);
          v[r].x += dl * E.x;
          v[r].y += dl * E.y;
        }
      }
    }
  }
}

// stage rows [0,nrows) of the strip in LDS and store row-major [P][nrows][NBP]
// (WGC threads per workgroup).
// The staging area aliases the FFT slices: barriers on both sides, except
// after the kernel's last store (LAST), where no slice is used again.
// MM < 16: the caller guarantees nrows <= MM*TPT, so slots m >= MM are never
// stored (and the transform's outputs there are dead code).
template <int TH, int CS, bool LAST = false, int MM = 16, int WGC = WG>
__device__ __forceinline__ void col_store_rows(const float2 (&v)[16], float2* st, const ColOut& o, int p, int strip,
                                               int NB, int NBP, int cc, int t) {
  constexpr int TPT = TH / 16;
  constexpr int RS = WGC / CS;  // rows stored per step (= TPT)
  const int nrows = o.nrows;
  __syncthreads();  // all transforms of the workgroup are done with the slices
  float2* sw = st + t * (CS + 1) + cc;
#pragma unroll
  for (int m = 0; m < MM; ++m) {
    if (TPT * (m + 1) <= nrows)  // uniform: no lane mask on whole slots
      sw[TPT * m * (CS + 1)] = v[m];
    else if (t + TPT * m < nrows)
      sw[TPT * m * (CS + 1)] = v[m];
  }
  __syncthreads();
  const int c0 = strip * CS;
  const int ci = threadIdx.x & (CS - 1);
  if (c0 + ci < NB - 1) {  // bin NB-1 travels packed in bin 0
    const int r0 = threadIdx.x / CS;
    float2* dst = o.p + (size_t)p * nrows * NBP + c0;
    const unsigned vo = (unsigned)(r0 * NBP + ci);
    const float2* sr = st + r0 * (CS + 1) + ci;
    const size_t step = (size_t)RS * NBP;
    auto rows = [&](auto nt) {
      int k = 0;
      // four steps of whole rows at a time, their LDS reads together
      for (; k + 4 * RS <= nrows; k += 4 * RS) {
        float2 x[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = sr[i * RS * (CS + 1)];
#pragma unroll
        for (int i = 0; i < 4; ++i) store_f2<decltype(nt)::value>(dst + i * step + vo, x[i]);
        dst += 4 * step;
        sr += 4 * RS * (CS + 1);
      }
      for (; k < nrows; k += RS) {
        if (k + r0 < nrows) store_f2<decltype(nt)::value>(dst + vo, sr[0]);
        dst += step;
        sr += RS * (CS + 1);
      }
    };
    if (o.nt)
      rows(std::true_type{});
    else
      rows(std::false_type{});
  }
  if (!LAST) __syncthreads();  // staging drained before the slices are reused
}

}  // namespace vmbd
