// series.hip -- whole Chebyshev series of small row-mask matrices in one launch.
//
// A step of a matrix of 10^4 rows is a launch of about 4 us for a few hundred
// nanoseconds of work.  Here every column of a filter is a job of one XCD: the
// first `parts` workgroups of a launch that find themselves on the XCD (two a
// CU) split its rows between them and run all the degrees, exchanging T_k
// through the XCD's L2.  A lane keeps its rows' cell addresses, values,
// diagonals, T_{k-1}, T_k and the FP64 sum in registers, so a degree is the
// gathers of T_k and one store.  The arithmetic is the row-mask step's
// (spmm_mask.h), and so are the bits.
//
// Nothing meets: a value of T_k travels with its tag in every eight bytes, and
// a gather whose tags are not T_{k-1}'s is looked at again.  Two slots do: a row
// overwrites T_{k-2} once it has seen T_{k-1} of its neighbours, which had to
// read its T_{k-2} for that -- hence the paired rows.  Waiting waves look only
// at one cell of every other wave they read (one load), not at all they need:
// repeated whole gathers fill the L2's queues and stores take tens of
// microseconds.  Loads are agent-scope, which pass the CU's own L1 by.
//
// Bound: latency, a store and two loads through L2 (0.8 us), and for the larger
// ones the gathers at 64 bytes a clock and CU (16 a value in FP64, 8 in FP32).
// A step takes (us, FP64 / FP32, one column; in brackets with a counted meeting
// of the workgroups after every step, and one launch a degree): 100 x 97 grid
// 0.86 / 0.82 (2.0 / 1.9, 3.5), 22 x 23 x 24 grid 1.0 / 1.0 (2.3 / 1.8, 3.5),
// 22^3 lattice 1.1 / 1.0 (2.7 / 1.9, 3.9), 31 x 32 x 33 grid 1.3 / 1.1 (3.4 /
// 2.1, 3.4), 40^3 grid 2.2 / 1.9 (3.2 / 2.6, 3.4); eight columns within 5% of
// that (launches 3.6 - 5.6).
// Choices, measured on the same grids: 64 workgroups of a row a lane against 32
// of two, 1.3 against 2.0 at 32,736 rows; a row at a time against both rows'
// gathers in flight, 2.2 against 5.7 - 8.5 on the 40^3 lattice; a few
// workgroups more than needed leave some CUs with three, 1.4 against 1.0; for
// lattices the row's own six entries against its twelve possible pairs, 1.1
// against 1.8.
//
// Waits are bounded.  A wave that does not see its cells in `limit` looks --
// the others are not resident because other work holds their CUs -- reports
// the launch as failed and leaves, as do the others; the host then runs the
// series by launches.  Which XCD a workgroup comes to is the hardware's choice:
// the one that takes an XCD's last share reports the start of its jobs, and a
// job that is not reported counts as failed as well.  So every share of a job
// that counts as done had a workgroup, and every wave of those has either ended
// it or reported that it gave up.
#include <hip/hip_runtime.h>

#include "dev.h"

namespace evsl_dev {
namespace {

constexpr int kSerWG = 512;
constexpr unsigned kNoCell = 0x80000000u;  // past every ring: loads 0, stores nothing
constexpr int kAgent = 16;                 // cache policy sc1: agent scope

__device__ __forceinline__ double fma_(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

using U2 = unsigned __attribute__((ext_vector_type(2)));
using U4 = unsigned __attribute__((ext_vector_type(4)));

// A value of T_k and its tag, one in every eight bytes.
template <typename VT>
struct Cell;
template <>
struct Cell<float> {
  using W = U2;
  static __device__ __forceinline__ W load(__amdgpu_buffer_rsrc_t r, unsigned at, unsigned base) {
    return __builtin_amdgcn_raw_buffer_load_b64(r, at, base, kAgent);
  }
  static __device__ __forceinline__ void store(__amdgpu_buffer_rsrc_t r, unsigned at, unsigned base,
                                               float v, unsigned tag) {
    __builtin_amdgcn_raw_buffer_store_b64(W{__float_as_uint(v), tag}, r, at, base, 0);
  }
  static __device__ __forceinline__ unsigned differs(W w, unsigned tag) { return w.y ^ tag; }
  static __device__ __forceinline__ float value(W w) { return __uint_as_float(w.x); }
};
template <>
struct Cell<double> {
  using W = U4;
  static __device__ __forceinline__ W load(__amdgpu_buffer_rsrc_t r, unsigned at, unsigned base) {
    return __builtin_amdgcn_raw_buffer_load_b128(r, at, base, kAgent);
  }
  static __device__ __forceinline__ void store(__amdgpu_buffer_rsrc_t r, unsigned at, unsigned base,
                                               double v, unsigned tag) {
    __builtin_amdgcn_raw_buffer_store_b128(
        W{(unsigned)__double2loint(v), tag, (unsigned)__double2hiint(v), tag}, r, at, base, 0);
  }
  static __device__ __forceinline__ unsigned differs(W w, unsigned tag) {
    return (w.y ^ tag) | (w.w ^ tag);
  }
  static __device__ __forceinline__ double value(W w) {
    return __hiloint2double((int)w.z, (int)w.x);
  }
};

// H: pairs on either side of the diagonal that the instance has room for, or
// (SLOT) half the entries off the diagonal that its rows have at most; RPT: rows
// per lane
template <typename VT, int H, int RPT, bool SLOT>
__global__ __launch_bounds__(kSerWG, 4) void k_cheb_series(const SeriesArgs a) {
  constexpr int P = 2 * H;
  using C = Cell<VT>;
  using W = typename C::W;
  __shared__ int s_rank;
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
  for (int j = (int)xcc; j < a.njobs; j += kSeriesXcds) {
    const SeriesJob& q = a.job[j];
    if (rank == a.parts - 1 && tid == 0)
      __hip_atomic_store(a.status + 1 + j, a.id, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    const int n = q.n;
    const int chunk = ((n + a.parts - 1) / a.parts + 63) & ~63;
    const int r0 = rank * chunk, r1 = min(n, r0 + chunk);
    const SeriesPairs& tab = *q.pairs;
    const int nneg = tab.nneg, np = tab.np;
    // the pairs in the instance's places, the negative offsets ending at H; with
    // SLOT every row's own entries in their order
    constexpr int RV = SLOT ? RPT : 1;
    VT val[RV][P];
    unsigned cell[RPT][P];
    int dpos[RV];
    const VT t1 = (VT)q.t1, t2 = (VT)q.t2, cc = (VT)q.cc;
    const VT* dgp = static_cast<const VT*>(q.dg);
    const unsigned half = (unsigned)n * sizeof(W);
    const __amdgpu_buffer_rsrc_t ring =
        __builtin_amdgcn_make_buffer_rsrc(q.ring, 0, (int)(2 * half), 0x00027000);
    unsigned at[RPT];
    VT d[RPT], xk[RPT], km1[RPT];
    double y[RPT];
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
      const int r = r0 + i * kSerWG + tid;
      unsigned m = 0;
      at[i] = kNoCell;
      d[i] = xk[i] = km1[i] = (VT)0;
      y[i] = 0.0;
      if (r < r1) {
        m = q.mbytes == 1 ? (unsigned)static_cast<const unsigned char*>(q.rmask)[r]
                          : (unsigned)static_cast<const unsigned short*>(q.rmask)[r];
        at[i] = (unsigned)r * (unsigned)sizeof(W);
        d[i] = dgp[r];
        xk[i] = (VT)q.in[r];
        y[i] = q.mu[0] * (double)xk[i];
      }
      C::store(ring, at[i], 0, xk[i], a.tag);
      if constexpr (SLOT) dpos[i] = __popc(m & ((1u << nneg) - 1u));
#pragma unroll
      for (int p = 0; p < P; ++p) {
        int s = p - (H - nneg);
        bool in = s >= 0 && s < np;
        if constexpr (SLOT) {
          in = m != 0;
          s = in ? __ffs((int)m) - 1 : 0;
          m &= m - 1u;
        }
        s = in ? s : 0;
        if (SLOT || i == 0)
          val[SLOT ? i : 0][p] = in ? (sizeof(VT) == 4 ? (VT)tab.val32[s] : (VT)tab.val64[s]) : (VT)0;
        if constexpr (!SLOT) in = in && ((m >> s) & 1u);
        cell[i][p] = in ? at[i] + (unsigned)(tab.off[s] * (int)sizeof(W)) : kNoCell;
      }
    }
    // a lane each for the first and the last cell that the wave's rows read at a
    // place; one lane will do for another wave's 64 rows, none for its own
    const int lane = tid & 63;
    unsigned watch[RPT];
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
      watch[i] = kNoCell;
#pragma unroll
      for (int p = 0; p < P; ++p) {
        const unsigned long long has = __ballot(cell[i][p] != kNoCell);
        if (has) {
          const int c0 = __builtin_amdgcn_readlane((int)cell[i][p], __ffsll(has) - 1);
          const int c1 = __builtin_amdgcn_readlane((int)cell[i][p], 63 - __clzll(has));
          if (lane == 2 * p) watch[i] = (unsigned)c0 + 4u;
          if (lane == 2 * p + 1) watch[i] = (unsigned)c1 + 4u;
        }
      }
      const unsigned wave = watch[i] / (64u * (unsigned)sizeof(W));
#pragma unroll
      for (int u = 0; u < RPT; ++u)
        if (wave == (unsigned)(r0 + u * kSerWG + (tid & ~63)) / 64u) watch[i] = kNoCell;
      for (int l = 0; l < 2 * P; ++l)
        if (lane > l && wave == (unsigned)__builtin_amdgcn_readlane((int)wave, l))
          watch[i] = kNoCell;
    }
    // coefficients, 64 degrees at a time: a lane holds one, the next are on their way
    double mus = q.mu[(size_t)min(lane, q.deg) * q.mu_step];
    double mun = q.mu[(size_t)min(64 + lane, q.deg) * q.mu_step];
    for (int k = 1; k <= q.deg; ++k) {
      const unsigned src = ((k - 1) & 1) ? half : 0, dst = (k & 1) ? half : 0;
      const unsigned tag = a.tag + (unsigned)k;
      const VT t = k == 1 ? t1 : t2;
      if ((k & 63) == 0) {
        mus = mun;
        mun = q.mu[(size_t)min(k + 64 + lane, q.deg) * q.mu_step];
      }
      const double mu =
          __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(mus), k & 63),
                           __builtin_amdgcn_readlane(__double2loint(mus), k & 63));
#pragma unroll
      for (int i = 0; i < RPT; ++i) {
        W xx[P];
        unsigned at_ = watch[i], bad, looks = 0;
        do {
          for (;;) {
            asm volatile("" ::: "memory");
            const unsigned got = __builtin_amdgcn_raw_buffer_load_b32(ring, at_, src, kAgent);
            if (!__any(at_ != kNoCell && got != tag - 1u) || ++looks >= a.limit) break;
            __builtin_amdgcn_s_sleep(1);
          }
          asm volatile("" ::: "memory");
#pragma unroll
          for (int p = 0; p < P; ++p) xx[p] = C::load(ring, cell[i][p], src);
          bad = 0;
#pragma unroll
          for (int p = 0; p < P; ++p)
            bad |= cell[i][p] == kNoCell ? 0u : C::differs(xx[p], tag - 1u);
          if (__any(bad != 0)) {  // every lane watches a cell that it misses
            at_ = kNoCell;
#pragma unroll
            for (int p = 0; p < P; ++p)
              if (cell[i][p] != kNoCell && C::differs(xx[p], tag - 1u)) at_ = cell[i][p] + 4u;
          }
        } while (__any(bad != 0) && ++looks < a.limit);
        if (__any(bad != 0)) {
          if (lane == 0)
            __hip_atomic_store(a.status, a.id, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
          return;
        }
        VT acc = (VT)0;
#pragma unroll
        for (int p = 0; p < P; ++p) {
          if constexpr (SLOT) {
            const VT with = fma_(d[i], xk[i], acc);
            acc = dpos[i] == p ? with : acc;
          } else if (p == H) {
            acc = fma_(d[i], xk[i], acc);
          }
          acc = fma_(val[SLOT ? i : 0][p], C::value(xx[p]), acc);  // absent: 0 (kNoCell)
        }
        if constexpr (SLOT) {
          const VT with = fma_(d[i], xk[i], acc);
          acc = dpos[i] == P ? with : acc;
        }
        const VT w = fma_(t, fma_(-cc, xk[i], acc), -km1[i]);
        if (k < q.deg) C::store(ring, at[i], dst, w, tag);
        y[i] = fma_(mu, (double)w, y[i]);
        km1[i] = xk[i];
        xk[i] = w;
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
hipError_t launch_series(int H, bool slot, int rpt, int grid, const SeriesArgs& a,
                         hipStream_t st) {
#define EVSL_SERIES(H_, R_, S_)                                                              \
  if (H <= H_ && slot == S_ && rpt <= R_) {                                                  \
    hipLaunchKernelGGL((k_cheb_series<VT, H_, R_, S_>), dim3(grid), dim3(kSerWG), 0, st, a); \
    return hipGetLastError();                                                                \
  }
#define EVSL_SERIES_H(H_, S_) EVSL_SERIES(H_, 1, S_) EVSL_SERIES(H_, 2, S_)
  EVSL_SERIES_H(3, true)
  EVSL_SERIES_H(2, false)
  EVSL_SERIES_H(3, false)
  EVSL_SERIES_H(6, false)
#undef EVSL_SERIES_H
#undef EVSL_SERIES
  return hipErrorInvalidValue;
}

}  // namespace

int series_rows_per_lane(int n) {
  const int chunk = ((n + kSeriesParts - 1) / kSeriesParts + 63) / 64 * 64;
  return (chunk + kSerWG - 1) / kSerWG;
}

hipError_t cheb_series(bool fp32, const SeriesArgs& a, int half, int row, int rows_per_lane,
                       hipStream_t st) {
  if (a.njobs < 1 || a.njobs > kSeriesMaxJobs || a.parts < 1 || a.parts > 64 ||
      a.grid < 1 || a.grid > kSeriesXcds * kSeriesParts ||
      half < 0 || half > kSeriesMaxHalf || rows_per_lane < 1 || rows_per_lane > kSeriesMaxRows)
    return hipErrorInvalidValue;
  const int grid = a.grid;
  const bool slot = half > 3 && row <= 6;
  if (slot) half = 3;
  return fp32 ? launch_series<float>(half, slot, rows_per_lane, grid, a, st)
              : launch_series<double>(half, slot, rows_per_lane, grid, a, st);
}

}  // namespace evsl_dev
