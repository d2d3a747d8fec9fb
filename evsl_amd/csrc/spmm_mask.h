// spmm_mask.h -- the fused Chebyshev step on matrices coded by row masks.
//
// A stencil or lattice operator repeats a few (column offset, value) pairs
// off the diagonal: 4 on a 2-D grid, 6 on a 3-D grid, 12 on a periodic 3-D
// lattice.  With at most kMaskPairs pairs, every row's columns ascending and
// every diagonal stored, a row is one mask (bit p: it holds pair p; pairs in
// order of their offsets) and its diagonal value.  The pairs sit in scalar
// registers, so a lane needs its mask, its diagonal and the gathers at its
// own address plus a scalar: nothing is staged, no block table is read, no
// barrier separates the loads, and a row takes 1 or 2 bytes instead of one to
// twelve per nonzero.  The products and their order are the CSR kernel's
// (ascending columns, the diagonal between the negative and the positive
// offsets), so the bits are the same; an absent pair adds the product of its
// value and zero.
//
// Bound: HBM (Infinity Cache while the working set fits); a one-column step is
// within 4 us, the launch, of its bytes at the copy rate.  Measured against the
// CSR kernel's best layout (us per step, y-flush cycle; 100^3 Laplacian / 80^3
// periodic lattice): FP64 1 column 16.9 -> 9.6 / 9.6 -> 7.2, 4 columns 28.9 ->
// 20.3 / 18.1 -> 14.8; FP32 1 column 11.6 -> 6.3 / 6.8 -> 4.9, 8 columns 29.2 ->
// 22.7 (6.3 TB/s) / 18.0 -> 16.1, 16 columns 66.8 -> 66.4 / 28.5 -> 25.7.  At 16
// and more columns of the larger grid both kernels re-read x from HBM (blocks
// are kept narrower there, filter_block_cap).
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "dev.h"
#include "spmm_kernel.h"

namespace evsl_dev {
namespace {

template <typename VT>
struct MaskTab {
  int np, nneg;  // pairs, those with a negative offset
  int off[kMaskPairs];
  VT val[kMaskPairs];  // 0 past np
};

// the fused multiply-adds that the compiler forms in the CSR kernel, spelled
// out: both kernels have to round alike
__device__ __forceinline__ double fma_(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// Rows of block `blk`: R passes of NG = 256 / (B / V) rows, lane layout as
// cheb_spmm_block's (V columns a lane); r = blk NG R + pass NG + lane group.
template <typename VT, int B, int V, int R, int MODE, typename MT, bool NT>
__global__ __launch_bounds__(kWG) void k_cheb_mask(
    int n, const MT* __restrict__ rmask, const VT* __restrict__ dg, const MaskTab<VT> tab, int nblk,
    const VT* __restrict__ xk, const VT* __restrict__ xkm1, VT* __restrict__ xkp1,
    double* __restrict__ y, const VT* __restrict__ v0, const double* __restrict__ scol,
    const double* __restrict__ mu0col, double t_, double cc_, int first, int yflush,
    double* __restrict__ part) {
  constexpr int L = B / V, NG = kWG / L;
  constexpr int U = 6;  // gathers in flight per lane: the pairs of a 3-D grid
  using Vec = VecT<VT, V>;
  using VecY = VecT<double, V>;
  const int blk = xcd_remap(blockIdx.x, nblk);
  const int tid = threadIdx.x;
  const int grp = tid / L, c0 = (tid % L) * V;
  const VT t = (VT)t_, cc = (VT)cc_;
  constexpr bool kY = MODE == kCheb || MODE == kRes;
  double dacc[V];
#pragma unroll
  for (int j = 0; j < V; ++j) dacc[j] = 0.0;
  auto ld = [](const VT* p) { return *reinterpret_cast<const Vec*>(p); };
  auto ld_last = [](const auto* p) {
    using ET = typename std::remove_cv<typename std::remove_reference<decltype(*p)>::type>::type;
    using RV = VecT<ET, V>;
    if constexpr (NT) {
      using EV = typename ExtVec<ET, V>::type;
      const EV e = __builtin_nontemporal_load(reinterpret_cast<const EV*>(p));
      RV r;
      __builtin_memcpy(&r, &e, sizeof(RV));
      return r;
    } else {
      return *reinterpret_cast<const RV*>(p);
    }
  };
  auto st_last = [](auto* p, const auto& v) {
    using ET = typename std::remove_reference<decltype(*p)>::type;
    using RV = VecT<ET, V>;
    static_assert(sizeof(v) == sizeof(RV), "store width");
    if constexpr (NT) {
      using EV = typename ExtVec<ET, V>::type;
      EV e;
      __builtin_memcpy(&e, &v, sizeof(RV));
      __builtin_nontemporal_store(e, reinterpret_cast<EV*>(p));
    } else {
      *reinterpret_cast<RV*>(p) = v;
    }
  };
#pragma unroll
  for (int pass = 0; pass < R; ++pass) {
    // uniform base of the pass's rows; a lane adds li
    const int rb = (blk * R + pass) * NG;
    const size_t base = (size_t)rb * B;
    const unsigned li = (unsigned)(grp * B + c0);
    if (!(grp < NG && rb + grp < n)) continue;
    const unsigned m = rmask[(size_t)rb + grp];
    const VT d = dg[(size_t)rb + grp];
    const VT* xb = xk + base;
    const Vec xr = ld(xb + li);
    Vec km1{}, rr{};
    VecY yo{};
    if (MODE != kPlain && xkm1) km1 = ld_last(xkm1 + base + li);
    if (kY && yflush > 0 && !first) yo = ld_last(y + base + li);
    if (MODE == kRes || MODE == kKpm) rr = ld(v0 + base + li);
    VT acc[V];
#pragma unroll
    for (int j = 0; j < V; ++j) acc[j] = 0;
    int p0 = 0;
    for (; p0 < tab.np; p0 += U) {
      Vec xx[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        xx[u] = Vec{};
        if ((m >> (p0 + u)) & 1u) xx[u] = ld(xb + (ptrdiff_t)tab.off[p0 + u] * B + li);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (p0 + u == tab.nneg) {
#pragma unroll
          for (int j = 0; j < V; ++j) acc[j] = fma_(d, xr.v[j], acc[j]);
        }
        const VT a = tab.val[p0 + u];
#pragma unroll
        for (int j = 0; j < V; ++j) acc[j] = fma_(a, xx[u].v[j], acc[j]);
      }
    }
    if (tab.nneg == p0) {
#pragma unroll
      for (int j = 0; j < V; ++j) acc[j] = fma_(d, xr.v[j], acc[j]);
    }
    Vec w;
#pragma unroll
    for (int j = 0; j < V; ++j) {
      if (MODE == kPlain) {
        w.v[j] = acc[j];
        continue;
      }
      VT wj = fma_(t, fma_(-cc, xr.v[j], acc[j]), -km1.v[j]);
      if (MODE == kRes) wj = fma_((VT)scol[c0 + j], rr.v[j], wj);
      w.v[j] = wj;
    }
    st_last(xkp1 + base + li, w);
    if (kY && yflush > 0) {
      // the terms of the last yflush degrees, as in cheb_spmm_block
      VecY yn;
#pragma unroll
      for (int j = 0; j < V; ++j) {
        double cs, cs1 = 0.0, cs2 = 0.0, cm = 0.0;
        if (MODE == kCheb) {
          cs = scol[c0 + j];
          if (yflush >= 2) cs1 = scol[c0 + j - B];
          if (yflush >= 3) cs2 = scol[c0 + j - 2 * B];
          if (first) cm = mu0col[c0 + j];
        } else {
          cs = mu0col[0];
          if (yflush >= 2) cs1 = mu0col[-2];
          if (yflush >= 3) cs2 = mu0col[-4];
          if (first) cm = mu0col[1];
        }
        double yv = first ? cm * (double)xr.v[j] : yo.v[j];
        if (yflush >= 3) yv = fma_(cs2, (double)km1.v[j], yv);
        if (yflush >= 2) yv = fma_(cs1, (double)xr.v[j], yv);
        yn.v[j] = fma_(cs, (double)w.v[j], yv);
      }
      st_last(y + base + li, yn);
    }
    if (MODE == kKpm) {
#pragma unroll
      for (int j = 0; j < V; ++j) dacc[j] = fma_((double)w.v[j], (double)rr.v[j], dacc[j]);
    }
  }
  if constexpr (MODE == kKpm) {
    // the block's dots in the tree of cheb_spmm_block (same rows per block
    // and lane, see mask_launch), so the moments have the CSR kernel's bits
    static_assert(kWG % L == 0, "KPM blocks need B/V | 256");
    __shared__ double s_red[kWG * V];
#pragma unroll
    for (int j = 0; j < V; ++j) s_red[tid * V + j] = dacc[j];
    __syncthreads();
    for (int st = NG / 2; st > 0; st >>= 1) {
      if (grp < st) {
#pragma unroll
        for (int j = 0; j < V; ++j) s_red[tid * V + j] += s_red[(tid + st * L) * V + j];
      }
      __syncthreads();
    }
    if (grp == 0) {
#pragma unroll
      for (int j = 0; j < V; ++j) part[(size_t)blk * B + c0 + j] = s_red[tid * V + j];
    }
  }
}

template <typename VT, int B, int V, int R, int MODE>
hipError_t launch_mask(const Csr& A, const void* xk, const void* xkm1, void* xkp1, void* y,
                       const void* v0, const double* s, const double* mu0, double t, double cc,
                       bool first, int yflush, double* part, hipStream_t st) {
  constexpr int NG = kWG / (B / V);
  MaskTab<VT> tab{};
  const VT* dg;
  tab.np = A.npair;
  tab.nneg = A.nneg;
  for (int p = 0; p < A.npair; ++p) {
    tab.off[p] = A.moff[p];
    if constexpr (sizeof(VT) == 4)
      tab.val[p] = A.mval32[p];
    else
      tab.val[p] = A.mval64[p];
  }
  if constexpr (sizeof(VT) == 4)
    dg = A.dg32;
  else
    dg = A.dg64;
  if (!dg || !A.rmask) return hipErrorInvalidValue;
  const int nblk = (A.n + NG * R - 1) / (NG * R);
  const int f = first ? 1 : 0;
#define EVSL_MASK_LAUNCH(MT_, NT_)                                                             \
  hipLaunchKernelGGL((k_cheb_mask<VT, B, V, R, MODE, MT_, NT_>), dim3(nblk), dim3(kWG), 0, st, \
                     A.n, (const MT_*)A.rmask, dg, tab, nblk, (const VT*)xk, (const VT*)xkm1, \
                     (VT*)xkp1, (double*)y, (const VT*)v0, s, mu0, t, cc, f, yflush, part)
  const bool byte = A.mbytes == 1;
  if constexpr (kStreamingCapable<MODE, B>) {
    if (streaming_launch(A, B, (int)sizeof(VT), MODE)) {
      if (byte)
        EVSL_MASK_LAUNCH(unsigned char, true);
      else
        EVSL_MASK_LAUNCH(unsigned short, true);
      return hipGetLastError();
    }
  }
  if (byte)
    EVSL_MASK_LAUNCH(unsigned char, false);
  else
    EVSL_MASK_LAUNCH(unsigned short, false);
#undef EVSL_MASK_LAUNCH
  return hipGetLastError();
}

}  // namespace
}  // namespace evsl_dev
