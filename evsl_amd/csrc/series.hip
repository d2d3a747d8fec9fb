// series.hip -- whole Chebyshev series of small row-mask matrices in one launch.
//
// A step of a matrix of 10^4 rows is a launch of about 4 us for a few hundred
// nanoseconds of work.  Here every column of a filter is a job of one XCD: the
// first `parts` workgroups of a launch that find themselves on the XCD split
// its rows between them and run all the degrees, exchanging T_k through the
// XCD's L2 and meeting once a degree.  A lane keeps its rows' masks, diagonals,
// T_{k-1}, T_k and the FP64 sum in registers, so a degree is the gathers of
// T_k, one store and the meeting; up to 8 columns (of one matrix or several)
// run side by side, further ones follow on the same XCDs.  The arithmetic is
// the row-mask step's (spmm_mask.h), and so are the bits.
//
// T_k is stored through to the XCD's L2, completely before its workgroup counts
// itself in, and read with agent-scope loads, which pass the reading CU's own
// L1 by; the counter is agent-scope too.  Bound: the meeting (about 1.2 us: the
// stores' acknowledgement, the count and a poll, each through L2).
// A step then takes (us, FP64 / FP32, one launch a degree in brackets; degree
// 400 with the call's own overhead): 64^2 grid 1.7 / 1.7 (3.6), 100 x 97 grid
// 2.0 / 1.9 (3.5), 22 x 23 x 24 grid 2.3 / 1.8 (3.5), 22^3 lattice 2.7 / 1.9
// (3.9), 30 x 32 x 34 grid 3.4 / 2.1 (3.5 / 3.3), 40^3 3.2 / 2.6 (3.5 / 3.3);
// eight columns 2.1, 2.4, 2.9 / 2.0, 3.4 / 2.2, 3.8 / 2.3 and 3.6 / 3.0 (3.6 -
// 5.6).  Gathers of a workgroup's own rows from LDS instead helped the largest
// FP64 grid (3.4 -> 2.8) and cost everywhere else (FP32 2.1 -> 2.6); plain loads
// with the L1 invalidated every eighth step cost 2 us a step.
//
// Waits are bounded.  A workgroup that does not see the others in `limit`
// polls -- they are not resident because other work holds their CUs -- reports
// the launch as failed and leaves, as do the others; the host then runs the
// series by launches (series_check).  A job whose XCD got no workgroup never
// reports its start, which counts as failed as well.
#include <hip/hip_runtime.h>

#include "dev.h"

namespace evsl_dev {
namespace {

constexpr int kSerWG = 512;

__device__ __forceinline__ double fma_(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

template <typename T>
__device__ __forceinline__ T ld_agent(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The workgroups of an XCD meet: everything they stored before is in its L2,
// and so seen by all of them, after.  `count` grows by one per workgroup and
// meeting, `want` is its value once all have come.  False once a wait has
// reached its limit.
__device__ __forceinline__ bool meet(unsigned* count, unsigned want, unsigned limit, int* s_ok) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned v =
        __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
    unsigned polls = 0;
    while (v < want && polls < limit) {
      v = ld_agent(count);
      ++polls;
    }
    *s_ok = v >= want;
  }
  __syncthreads();
  return *s_ok != 0;
}

// H: pairs on either side of the diagonal that the instance has room for;
// RPT: rows per lane
template <typename VT, int H, int RPT>
__global__ __launch_bounds__(kSerWG) void k_cheb_series(const SeriesArgs a) {
  constexpr int P = 2 * H;
  constexpr int IG = H <= 3 || RPT < 2 ? RPT : 2;  // rows in flight
  __shared__ int s_rank, s_ok;
  unsigned xcc;
  asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID, 0, 4)" : "=s"(xcc));
  if (xcc >= (unsigned)kSeriesXcds) return;
  const int tid = threadIdx.x;
  if (tid == 0)
    s_rank = (int)__hip_atomic_fetch_add(a.words + xcc * kSeriesStride, 1u, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  const int rank = s_rank;
  if (rank >= a.parts) return;
  unsigned* count = a.words + xcc * kSeriesStride + 32;
  unsigned want = 0;
  for (int j = (int)xcc; j < a.njobs; j += kSeriesXcds) {
    const SeriesJob& q = a.job[j];
    if (rank == 0 && tid == 0)
      __hip_atomic_store(a.status + 1 + j, a.id, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    const int n = q.n;
    const int chunk = ((n + a.parts - 1) / a.parts + 63) & ~63;
    const int r0 = rank * chunk, r1 = min(n, r0 + chunk);
    // pairs in the instance's places: the negative offsets end at H
    const SeriesPairs& tab = *q.pairs;
    const int nneg = tab.nneg, np = tab.np;
    int off[P];
    VT val[P];
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int s = p - (H - nneg);
      const bool in = s >= 0 && s < np;
      off[p] = in ? tab.off[in ? s : 0] : 0;
      val[p] = in ? (sizeof(VT) == 4 ? (VT)tab.val32[in ? s : 0] : (VT)tab.val64[in ? s : 0]) : (VT)0;
    }
    const VT t1 = (VT)q.t1, t2 = (VT)q.t2, cc = (VT)q.cc;
    const VT* dgp = static_cast<const VT*>(q.dg);
    VT* buf = static_cast<VT*>(q.ring);
    unsigned m[RPT];
    VT d[RPT], xk[RPT], km1[RPT];
    double y[RPT];
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
      const int r = r0 + i * kSerWG + tid;
      m[i] = 0;
      d[i] = xk[i] = km1[i] = (VT)0;
      y[i] = 0.0;
      if (r < r1) {
        m[i] = (q.mbytes == 1 ? (unsigned)static_cast<const unsigned char*>(q.rmask)[r]
                              : (unsigned)static_cast<const unsigned short*>(q.rmask)[r])
               << (H - nneg);
        d[i] = dgp[r];
        xk[i] = (VT)q.in[r];
        y[i] = q.mu[0] * (double)xk[i];
        buf[r] = xk[i];
      }
    }
    if (!meet(count, want += a.parts, a.limit, &s_ok)) {
      if (tid == 0)
        __hip_atomic_store(a.status, a.id, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      return;
    }
    for (int k = 1; k <= q.deg; ++k) {
      const VT* src = buf + (size_t)((k - 1) & 1) * n;
      VT* dst = buf + (size_t)(k & 1) * n;
      const VT t = k == 1 ? t1 : t2;
      const double mu = q.mu[(size_t)k * q.mu_step];
#pragma unroll
      for (int i0 = 0; i0 < RPT; i0 += IG) {
        VT xx[IG][P];
#pragma unroll
        for (int u = 0; u < IG; ++u) {
          const int r = r0 + (i0 + u) * kSerWG + tid;
#pragma unroll
          for (int p = 0; p < P; ++p) {
            xx[u][p] = (VT)0;
            if ((m[i0 + u] >> p) & 1u) xx[u][p] = ld_agent(src + (r + off[p]));
          }
        }
#pragma unroll
        for (int u = 0; u < IG; ++u) {
          const int i = i0 + u, r = r0 + i * kSerWG + tid;
          VT acc = (VT)0;
#pragma unroll
          for (int p = 0; p < P; ++p) {
            if (p == H) acc = fma_(d[i], xk[i], acc);
            acc = fma_(val[p], xx[u][p], acc);
          }
          const VT w = fma_(t, fma_(-cc, xk[i], acc), -km1[i]);
          y[i] = fma_(mu, (double)w, y[i]);
          km1[i] = xk[i];
          xk[i] = w;
          if (r < r1 && k < q.deg) dst[r] = w;
        }
      }
      if (k < q.deg && !meet(count, want += a.parts, a.limit, &s_ok)) {
        if (tid == 0)
          __hip_atomic_store(a.status, a.id, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        return;
      }
    }
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
      const int r = r0 + i * kSerWG + tid;
      if (r < r1) q.out[r] = y[i];
    }
  }
}

template <typename VT>
hipError_t launch_series(int H, int rpt, int grid, const SeriesArgs& a, hipStream_t st) {
#define EVSL_SERIES(H_, R_)                                                            \
  if (H <= H_ && rpt <= R_) {                                                          \
    hipLaunchKernelGGL((k_cheb_series<VT, H_, R_>), dim3(grid), dim3(kSerWG), 0, st, a); \
    return hipGetLastError();                                                          \
  }
#define EVSL_SERIES_H(H_) \
  EVSL_SERIES(H_, 1)      \
  EVSL_SERIES(H_, 2)      \
  EVSL_SERIES(H_, 4)
  EVSL_SERIES_H(2)
  EVSL_SERIES_H(3)
  EVSL_SERIES_H(6)
#undef EVSL_SERIES_H
#undef EVSL_SERIES
  return hipErrorInvalidValue;
}

}  // namespace

int series_rows_per_lane(int n) {
  const int chunk = ((n + kSeriesParts - 1) / kSeriesParts + 63) / 64 * 64;
  return (chunk + kSerWG - 1) / kSerWG;
}

hipError_t cheb_series(bool fp32, const SeriesArgs& a, int half, int rows_per_lane,
                       hipStream_t st) {
  if (a.njobs < 1 || a.njobs > kSeriesMaxJobs || a.parts < 1 || a.parts > 64 ||
      half < 0 || half > kSeriesMaxHalf || rows_per_lane < 1 || rows_per_lane > kSeriesMaxRows)
    return hipErrorInvalidValue;
  // a quarter more workgroups than are needed: those an XCD does not need
  // leave at once
  const int grid = kSeriesXcds * (a.parts + a.parts / 4);
  return fp32 ? launch_series<float>(half, rows_per_lane, grid, a, st)
              : launch_series<double>(half, rows_per_lane, grid, a, st);
}

}  // namespace evsl_dev
