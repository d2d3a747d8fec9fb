// lanstep.hip -- the vector work of a Lanczos step: the three-term recurrence,
// the Gram-Schmidt pass against the basis, and the modified Gram-Schmidt chain
// of the bounds and DOS runs.
//
// A step on 10^4 rows is a handful of microseconds of work in every kernel, so
// launches and waits are what it costs.  Each kernel here takes up to kLanCols
// columns (the slices of a batch advance together, blockIdx.y), finishes the
// sum that the next one needs itself (every block adds the previous kernel's
// partials, in the order of sum_scalar) instead of waiting for a launch that
// does, and keeps many loads in flight.  The order of every sum is the one of
// the separate kernels (kernels.hip), which larger matrices still run for the
// Gram-Schmidt pass, so the bits are the same.  Measured on 9,700 rows and 165
// basis vectors: V^T w 17.0 -> 5.2 us (16 rows a thread went one after the
// other; now two columns a workgroup and four rows in flight), w - V h 10.5 ->
// 9.3 us (four threads a row, one for each of its four sums).  The runs of an
// LanDos call go through the step's nine launches eight at a time: 20 runs of 40
// steps on a 20^3 grid with the bounds before them 44.0 -> 23.7 ms, the rest of
// it the host's draws of the vectors and the bounds' steps.
#include <hip/hip_runtime.h>

#include "dev.h"

namespace evsl_dev {
namespace {

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  return v;
}

// sum over the first 256 threads of a block; valid in thread 0.  Every thread
// of the block calls it.
__device__ __forceinline__ double sum256(double v, double* sh /*4*/) {
  v = wave_sum(v);
  if (threadIdx.x < 256 && (threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  const double r = sh[0] + sh[1] + sh[2] + sh[3];
  __syncthreads();
  return r;
}

// sum_scalar of part[0..cnt), in every thread of the block
__device__ __forceinline__ double sum_all(const double* __restrict__ part, int cnt, double* sh) {
  double a = 0.0;
  if (threadIdx.x < 256)
    for (int i = threadIdx.x; i < cnt; i += 256) a += part[i];
  return sum256(a, sh);
}

// vnew -= beta zold (vnew from the block wi where there is one); P1 = partials
// of vnew.v
__global__ __launch_bounds__(256) void k_lan_axpy(size_t n, const LanCols cols) {
  __shared__ double sh[4];
  const LanCol& q = cols.c[blockIdx.y];
  const double* __restrict__ zold = q.zold;
  const double* __restrict__ v = q.v;
  double* __restrict__ w = q.vnew;
  const double* __restrict__ wi = q.wi;
  const size_t ldi = q.ldi;
  const double a = zold ? -(q.beta_d ? *q.beta_d : q.beta) : 0.0;
  double d = 0.0;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
    double x = wi ? wi[i * ldi] : w[i];
    if (zold) x = __builtin_fma(a, zold[i], x);
    if (zold || wi) w[i] = x;
    d = __builtin_fma(x, v[i], d);
  }
  d = sum256(d, sh);
  if (threadIdx.x == 0) q.part[blockIdx.x] = d;
}

// alpha = sum P1 (out[0]); vnew -= alpha v; P2 = partials of ||vnew||^2
__global__ __launch_bounds__(256) void k_lan_alpha(size_t n, const LanCols cols) {
  __shared__ double sh[4];
  const LanCol& q = cols.c[blockIdx.y];
  const double* __restrict__ v = q.v;
  double* __restrict__ w = q.vnew;
  const double alpha = sum_all(q.part, gridDim.x, sh);
  const double a = -1.0 * alpha;
  double d = 0.0;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
    const double x = __builtin_fma(a, v[i], w[i]);
    w[i] = x;
    d = __builtin_fma(x, x, d);
  }
  d = sum256(d, sh);
  if (threadIdx.x == 0) {
    q.part[kRedBlocks + blockIdx.x] = d;
    if (blockIdx.x == 0) q.out[0] = alpha;
  }
}

constexpr int kGtRows = 4096;  // rows per chunk, as k_gemv_t_partial

// gt[c * nch + chunk] = sum over the chunk's rows of V(r, c) * vnew(r), NC
// columns a workgroup; TWO: the same with v for vnew behind it (gt2)
template <int NC, bool F32, bool TWO>
__global__ __launch_bounds__(256) void k_lan_gemv_t(size_t n, const LanCols cols, int nch) {
  __shared__ double sh[TWO ? 8 : 4][NC];
  const LanCol& q = cols.c[blockIdx.y];
  const int ch = blockIdx.x % nch, c0 = blockIdx.x / nch * NC;
  const int nc = min(NC, q.k - c0);
  if (nc <= 0) return;
  const double* __restrict__ w = q.vnew;
  const double* __restrict__ w2 = q.v;
  double acc[NC], acc2[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) acc[c] = acc2[c] = 0.0;
  const size_t rbeg = (size_t)ch * kGtRows, rend = min(n, rbeg + kGtRows);
  constexpr int U = 4;  // rows (F32: row pairs) in flight
  if constexpr (F32) {
    static_assert(!TWO || !F32, "two products only against the FP64 basis");
    const float* V = q.V32 + (size_t)c0 * q.ld32;
    for (size_t r0 = rbeg + 2 * threadIdx.x; r0 < rend; r0 += 512 * U) {
      float2 x[U][NC];
      double w0[U], w1[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const size_t r = r0 + 512 * u;
        w0[u] = r < rend ? w[r] : 0.0;
        w1[u] = r + 1 < rend ? w[r + 1] : 0.0;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          x[u][c] = make_float2(0.f, 0.f);
          if (c < nc && r + 1 < rend)
            x[u][c] = *reinterpret_cast<const float2*>(V + (size_t)c * q.ld32 + r);
          else if (c < nc && r < rend)
            x[u][c].x = V[(size_t)c * q.ld32 + r];
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          acc[c] = __builtin_fma((double)x[u][c].x, w0[u], acc[c]);
          acc[c] = __builtin_fma((double)x[u][c].y, w1[u], acc[c]);
        }
    }
  } else {
    const double* V = q.V + (size_t)c0 * n;
    for (size_t r0 = rbeg + threadIdx.x; r0 < rend; r0 += 256 * U) {
      double x[U][NC], w0[U], w1[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const size_t r = r0 + 256 * u;
        w0[u] = r < rend ? w[r] : 0.0;
        w1[u] = TWO && r < rend ? w2[r] : 0.0;
#pragma unroll
        for (int c = 0; c < NC; ++c) x[u][c] = c < nc && r < rend ? V[(size_t)c * n + r] : 0.0;
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          acc[c] = __builtin_fma(x[u][c], w0[u], acc[c]);
          if (TWO) acc2[c] = __builtin_fma(x[u][c], w1[u], acc2[c]);
        }
    }
  }
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const double s = wave_sum(acc[c]);
    if (lane == 0) sh[wid][c] = s;
    if (TWO) {
      const double s2 = wave_sum(acc2[c]);
      if (lane == 0) sh[4 + wid][c] = s2;
    }
  }
  __syncthreads();
  if (threadIdx.x < nc) {
    const int c = threadIdx.x;
    q.gt[(size_t)(c0 + c) * nch + ch] = sh[0][c] + sh[1][c] + sh[2][c] + sh[3][c];
    if (TWO) q.gt2[(size_t)(c0 + c) * nch + ch] = sh[4][c] + sh[5][c] + sh[6][c] + sh[7][c];
  }
}

// k_gemv_t_reduce's sum of cnt <= 16 partials: a wave's tree over 64 lanes, the
// lanes from 16 on zero
__device__ __forceinline__ double tree16(const double* __restrict__ p, int cnt) {
  double v[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) v[i] = i < cnt ? p[i] : 0.0;
#pragma unroll
  for (int off = 8; off > 0; off >>= 1)
#pragma unroll
    for (int i = 0; i < off; ++i) v[i] += v[i + off];
  return v[0];
}

constexpr int kHTile = 2048;

// vnew -= V h, h summed from the partials gt (HPART) or given (hvec); P3 =
// partials of ||vnew||^2, one per 256 threads' rows.  Four threads a row (F32: a
// row pair), thread t of them with the columns c = t mod 4 in k_gemv_n's sum
// a_t; the columns past a multiple of four go to a_0.
template <bool F32, bool HPART>
__global__ __launch_bounds__(1024) void k_lan_gemv_n(size_t n, const LanCols cols, int nch) {
  __shared__ double s_h[kHTile];
  __shared__ double s_a[3][F32 ? 512 : 256];
  __shared__ double sh[4];
  const LanCol& q = cols.c[blockIdx.y];
  const int lr = threadIdx.x & 255, t = threadIdx.x >> 8, k = q.k;
  const size_t i = (size_t)blockIdx.x * 256 + lr, r = F32 ? 2 * i : i;
  const bool in = r < n, pair = F32 && r + 1 < n;
  double a = 0.0, b = 0.0;
  for (int cb = 0; cb < k; cb += kHTile) {
    const int nc = min(kHTile, k - cb), main = nc & ~3;
    __syncthreads();
    for (int c = threadIdx.x; c < nc; c += 1024)
      s_h[c] = HPART ? tree16(q.gt + (size_t)(cb + c) * nch, nch) : q.hvec[cb + c];
    __syncthreads();
    if (in) {
      if constexpr (F32) {
        const float* V = q.V32 + (size_t)cb * q.ld32 + r;
        auto one = [&](int c) {
          if (pair) {
            const float2 x = *reinterpret_cast<const float2*>(V + (size_t)c * q.ld32);
            a = __builtin_fma((double)x.x, s_h[c], a);
            b = __builtin_fma((double)x.y, s_h[c], b);
          } else {
            a = __builtin_fma((double)V[(size_t)c * q.ld32], s_h[c], a);
          }
        };
#pragma unroll 8
        for (int c = t; c < main; c += 4) one(c);
        if (t == 0)
          for (int c = main; c < nc; ++c) one(c);
      } else {
        const double* V = q.V + (size_t)cb * n + r;
#pragma unroll 8  // 16: 14.9 us
        for (int c = t; c < main; c += 4) a = __builtin_fma(V[(size_t)c * n], s_h[c], a);
        if (t == 0)
          for (int c = main; c < nc; ++c) a = __builtin_fma(V[(size_t)c * n], s_h[c], a);
      }
    }
  }
  if (t > 0) {
    s_a[t - 1][lr] = a;
    if (F32) s_a[t - 1][256 + lr] = b;
  }
  __syncthreads();
  double d = 0.0;
  if (t == 0 && in) {
    double* w = q.vnew;
    const double x = w[r] - ((a + s_a[0][lr]) + (s_a[1][lr] + s_a[2][lr]));
    w[r] = x;
    d = x * x;
    if (pair) {
      const double y =
          w[r + 1] - ((b + s_a[0][256 + lr]) + (s_a[1][256 + lr] + s_a[2][256 + lr]));
      w[r + 1] = y;
      d = __builtin_fma(y, y, d);
    }
  }
  d = sum256(d, sh);
  if (threadIdx.x == 0) q.part[2 * kRedBlocks + blockIdx.x] = d;
}

// out[1] = sum of P2 (rb of them) by block x = 0, out[slot] = sum of P3 (np) by
// the other; first = 1 leaves the first out
__global__ __launch_bounds__(256) void k_lan_sums(const LanCols cols, int rb, int first, int slot) {
  __shared__ double sh[4];
  const LanCol& q = cols.c[blockIdx.y];
  const bool p3 = blockIdx.x + first > 0;
  const double s = p3 ? sum_all(q.part + 2 * kRedBlocks, q.np, sh)
                      : sum_all(q.part + kRedBlocks, rb, sh);
  if (threadIdx.x == 0) q.out[p3 ? slot : 1] = s;
}

// vnew *= a and its copies in FP32 and in the block xi; a = beta, or 1 / *beta_d
__global__ __launch_bounds__(256) void k_lan_scal(size_t n, const LanCols cols) {
  const LanCol& q = cols.c[blockIdx.y];
  const double a = q.beta_d ? 1.0 / *q.beta_d : q.beta;
  double* __restrict__ x = q.vnew;
  float* __restrict__ x32 = q.x32;
  double* __restrict__ xi = q.xi;
  const size_t ldi = q.ldi;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
    const double y = x[i] * a;
    x[i] = y;
    if (x32) x32[i] = (float)y;
    if (xi) xi[i * ldi] = y;
  }
}

// The projections of a modified Gram-Schmidt sweep from two products: with
// a_i = v_i.w and G(i, l) = v_i.v_l (l < i), the sweep's
// h_i = v_i.(w - sum_{l < i} h_l v_l) are the solution of (I + G) h = a.  Sums
// the partials of a (gt) and of the newest basis vector's row of G (gt2, kept
// in G), then solves in panels of 64 rows.  One workgroup a column.
__global__ __launch_bounds__(256) void k_mgs_solve(const LanCols cols, int nch, int ldg) {
  __shared__ double s_g[64][65];
  __shared__ double s_p[64];
  const LanCol& q = cols.c[blockIdx.y];
  double* G = q.G;
  const int k = q.k, lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  double* h = const_cast<double*>(q.hvec);
  for (int c = wid; c < k; c += 4) {
    double a = 0.0, g = 0.0;
    for (int i = lane; i < nch; i += 64) {
      a += q.gt[(size_t)c * nch + i];
      g += q.gt2[(size_t)c * nch + i];
    }
    a = wave_sum(a);
    g = wave_sum(g);
    if (lane == 0) {
      h[c] = a;
      if (c + 1 < k) G[(size_t)(k - 1) * ldg + c] = g;
    }
  }
  __syncthreads();
  for (int p0 = 0; p0 < k; p0 += 64) {
    const int np = min(64, k - p0);
    for (int e = threadIdx.x; e < 64 * 64; e += 256) {
      const int i = e >> 6, l = e & 63;
      s_g[i][l] = (i < np && l < i) ? G[(size_t)(p0 + i) * ldg + p0 + l] : 0.0;
    }
    __syncthreads();
    if (wid == 0) {
      double a = lane < np ? h[p0 + lane] : 0.0;
      for (int l = 0; l < np; ++l) {
        const double hl = __shfl(a, l, 64);
        a -= s_g[lane][l] * hl;  // 0 for lane <= l
      }
      s_p[lane] = a;
      if (lane < np) h[p0 + lane] = a;
    }
    __syncthreads();
    for (int i = p0 + np + threadIdx.x; i < k; i += 256) {
      double a = h[i];
      for (int l = 0; l < np; ++l) a -= G[(size_t)i * ldg + p0 + l] * s_p[l];
      h[i] = a;
    }
    __syncthreads();
  }
}

// *b2 = sum of P3, *b = its root
__global__ __launch_bounds__(256) void k_lan_norm(const LanCols cols) {
  __shared__ double sh[4];
  const LanCol& q = cols.c[blockIdx.y];
  const double s = sum_all(q.part + 2 * kRedBlocks, q.np, sh);
  if (threadIdx.x == 0) {
    *q.b2 = s;
    *q.b = sqrt(s);
  }
}

inline unsigned blocks(size_t n, size_t per, size_t cap) {
  const size_t g = (n + per - 1) / per;
  return (unsigned)(g < 1 ? 1 : g > cap ? cap : g);
}

}  // namespace

bool lan_small(size_t n) { return gemv_t_chunks(n) <= 16; }

size_t lan_part_elems(size_t n) { return 2 * (size_t)kRedBlocks + (n + 255) / 256; }

hipError_t lan_recurrence(size_t n, const LanCols& cols, int ncol, hipStream_t st) {
  const dim3 grid(blocks(n, 256, kRedBlocks), ncol);
  hipLaunchKernelGGL(k_lan_axpy, grid, dim3(256), 0, st, n, cols);
  hipLaunchKernelGGL(k_lan_alpha, grid, dim3(256), 0, st, n, cols);
  return hipGetLastError();
}

hipError_t lan_gram_schmidt(size_t n, LanCols& cols, int ncol, bool f32, hipStream_t st) {
  if (!lan_small(n)) return hipErrorInvalidValue;
  const int nch = gemv_t_chunks(n);
  int kmax = 0;
  for (int j = 0; j < ncol; ++j) kmax = cols.c[j].k > kmax ? cols.c[j].k : kmax;
  const unsigned gt = (unsigned)(nch * ((kmax + 1) / 2));
  const size_t rows = f32 ? 512 : 256;
  const unsigned gn = (unsigned)((n + rows - 1) / rows);
  for (int j = 0; j < ncol; ++j) cols.c[j].np = (int)gn;
  if (f32) {
    hipLaunchKernelGGL((k_lan_gemv_t<2, true, false>), dim3(gt, ncol), dim3(256), 0, st, n, cols, nch);
    hipLaunchKernelGGL((k_lan_gemv_n<true, true>), dim3(gn, ncol), dim3(1024), 0, st, n, cols, nch);
  } else {
    hipLaunchKernelGGL((k_lan_gemv_t<2, false, false>), dim3(gt, ncol), dim3(256), 0, st, n, cols, nch);
    hipLaunchKernelGGL((k_lan_gemv_n<false, true>), dim3(gn, ncol), dim3(1024), 0, st, n, cols, nch);
  }
  return hipGetLastError();
}

hipError_t lan_sums(size_t n, const LanCols& cols, int ncol, bool second, hipStream_t st) {
  hipLaunchKernelGGL(k_lan_sums, dim3(second ? 1 : 2, ncol), dim3(256), 0, st, cols,
                     (int)blocks(n, 256, kRedBlocks), second ? 1 : 0, second ? 3 : 2);
  return hipGetLastError();
}

hipError_t lan_scale(size_t n, const LanCols& cols, int ncol, hipStream_t st) {
  hipLaunchKernelGGL(k_lan_scal, dim3(blocks(n, 256, 4096), ncol), dim3(256), 0, st, n, cols);
  return hipGetLastError();
}

hipError_t lan_mgs(size_t n, LanCols& cols, int ncol, int ldg, hipStream_t st) {
  const int nch = gemv_t_chunks(n), k = cols.c[0].k;
  const unsigned gn = (unsigned)((n + 255) / 256);
  for (int j = 0; j < ncol; ++j) cols.c[j].np = (int)gn;
  if (lan_small(n))
    hipLaunchKernelGGL((k_lan_gemv_t<2, false, true>), dim3(nch * ((k + 1) / 2), ncol), dim3(256),
                       0, st, n, cols, nch);
  else
    hipLaunchKernelGGL((k_lan_gemv_t<8, false, true>), dim3(nch * ((k + 7) / 8), ncol), dim3(256),
                       0, st, n, cols, nch);
  hipLaunchKernelGGL(k_mgs_solve, dim3(1, ncol), dim3(256), 0, st, cols, nch, ldg);
  hipLaunchKernelGGL((k_lan_gemv_n<false, false>), dim3(gn, ncol), dim3(1024), 0, st, n, cols, nch);
  hipLaunchKernelGGL(k_lan_norm, dim3(1, ncol), dim3(256), 0, st, cols);
  return hipGetLastError();
}

hipError_t lan_normalise(size_t n, LanCols& cols, int ncol, hipStream_t st) {
  for (int j = 0; j < ncol; ++j) {
    LanCol& q = cols.c[j];
    if (hipError_t e = dot_partial(n, q.vnew, q.vnew, q.part + 2 * kRedBlocks, st)) return e;
    q.np = kRedBlocks;
    q.beta_d = q.b;
  }
  hipLaunchKernelGGL(k_lan_norm, dim3(1, ncol), dim3(256), 0, st, cols);
  return lan_scale(n, cols, ncol, st);
}

}  // namespace evsl_dev
