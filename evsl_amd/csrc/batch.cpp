// batch.cpp -- all slices of one matrix as one batched filtered Lanczos run,
// and the FP64 Rayleigh-Ritz refinement of the mixed-precision form.
//
// Each slice is the reference's ChebLanNr (SRC/cheblanNr.c:57-434) with its
// own filter, basis, recurrence and stopping test.  What changes is the
// schedule: every round takes the current Lanczos vector of each active
// slice, interleaves them into one row-major block and advances all of them
// through one fused SpMM launch per degree (per-column filter coefficients),
// so A is read once per degree for the whole batch.  Slices leave the batch
// when their restricted-trace test passes.
//
// Mixed precision (EVSL_PREC_MIXED): the filter runs on FP32 values and
// vectors with FP32 accumulation; the Lanczos recurrence, re-orthogonalization
// and the tridiagonal eigensolve stay FP64.  Accuracy is won back at the end:
// the Ritz vectors of T above a guard threshold are filtered once more with
// the FP64 filter, orthonormalized (Cholesky QR) and rotated by the
// eigenvectors of the FP64 Rayleigh quotient U^T A U; residuals are FP64.
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <string>
#include <vector>

#include "internal.h"

namespace evsl {
namespace {

constexpr double kOrthTol = 1e-14;
const double kEpsM = EVSL_DBL_EPS_MULT * DBL_EPSILON;
constexpr int kBmaxPow = 32;

int pow2_at_least(int b) {
  int p = 1;
  while (p < b) p <<= 1;
  return p;
}
// block widths the kCheb kernel is instantiated for
int kernel_width(int b) { return b <= 8 ? b : pow2_at_least(b); }

// Columns of one filter block on A: kBmaxPow, or fewer for the row-mask kernel,
// whose matrix is a small part of a step's bytes, where the block's vectors
// (three of the vector type, y in FP64, and the residual block of kRes) outgrow
// 200 MB: they then stay in the 256 MB Infinity Cache from step to step
// (100^3, us per column and step at 4 / 8 / 16 / 32 columns: FP32 3.4 / 2.8 /
// 4.2 / 4.1, FP64 5.1 / 6.8 / 6.7 / 6.9, FP32 residual step - / 3.1 / - / 4.4;
// 80^3 lattice FP32 2.2 / 2.0 / 1.6 / 2.3).  At least one 16-byte vector a lane
// and two lanes a row.  A column's bits do not depend on its block.
int filter_block_cap(const evsl_dev::Csr& A, bool f32, evsl_dev::Mode mode) {
  int B = kBmaxPow;
  if (!evsl_dev::mask_launch(A, B, f32, mode)) return B;
  const double vs = f32 ? 4 : 8;
  const double col = ((mode == evsl_dev::kRes ? 4.0 : 3.0) * vs + 8.0) * A.n;
  while (B > (f32 ? 8 : 4) && B * col > 200e6) B >>= 1;
  return B;
}

// Launches k = k0..k1 of the Chebyshev filter of per-column coefficient
// table mus (row d holds degree d, B entries per row) over the row-major
// block X0 of B columns, accumulating into Y.  The y flushes are scheduled
// within the segment, so its last launch leaves no pending term; ring slot
// (k-1)%3 of bufs receives T_k.
int block_filter_seg(int B, const FilterOp& op, const double* mus_d, int k0, int k1,
                     const void* X0, void* const bufs[3], void* Y) {
  Context& c = ctx();
  const size_t vs = op.f32 ? 4 : 8;
  for (int k = k0; k <= k1; ++k) {
    void* xkp1 = bufs[(k - 1) % 3];
    const void* xk = (k == 1) ? X0 : bufs[(k - 2) % 3];
    const void* xkm1 = (k == 1) ? nullptr : (k == 2 ? X0 : bufs[(k - 3) % 3]);
    const int yf = evsl_dev::y_flush(k - k0 + 1, k1 - k0 + 1);
    EVSL_HIP(evsl_dev::cheb_spmm(op.A, B, op.f32, evsl_dev::kCheb, xk, xkm1, xkp1, Y, nullptr,
                                 mus_d + (size_t)k * B, mus_d, k == 1 ? op.t1 : op.t2, op.cc,
                                 k == 1, yf, nullptr, c.stream));
    c.astats.filter_bytes += c.A.mat_bytes((int)vs, B) +
                             evsl_dev::cheb_vec_bytes(yf, k == 1, (int)vs) * B * c.n;
  }
  c.astats.n_filter_steps += k1 - k0 + 1;
  c.astats.n_filter_cols += (size_t)(k1 - k0 + 1) * B;
  return 0;
}

// The whole series k = 1..maxdeg at one width.
int block_filter(int B, const FilterOp& op, const double* mus_d, int maxdeg, const void* X0,
                 void* const bufs[3], void* Y) {
  return block_filter_seg(B, op, mus_d, 1, maxdeg, X0, bufs, Y);
}

// Shared work buffers of the blocked filter (sized for Bmax columns; the
// output blocks Y, Y2 are FP64 in both precisions).  The
// coefficient tables stay on the device while the same filters come back
// (the batched solver filters the same slices step after step), so a filter
// pass issues no host-device copy and no synchronisation.
struct BlockWork {
  DevBuf X0, bufs, Y, Y2, zero, junk;
  int Bcap = 0;
  bool f32 = false;
  struct CoefTab {
    DevBuf mus;
    std::vector<const polparams*> key;  // filters (in column order) of `mus`
    int kind = -1;                      // layout of `mus`: B, or 0 for phased
    std::vector<size_t> off;            // phased: offset of each phase's table
  };
  // the tables of a pass's blocks, at most kCoefTabs (a further block takes
  // over the oldest)
  static constexpr size_t kCoefTabs = 8;
  std::vector<std::unique_ptr<CoefTab>> tabs;
  size_t next_tab = 0;
  int ensure(int n, int B, bool fp32, int maxdeg) {
    const size_t vs = fp32 ? 4 : 8;
    const size_t nb = (size_t)n * B * vs;
    EVSL_HIP(X0.alloc(nb));
    EVSL_HIP(bufs.alloc(3 * nb));
    EVSL_HIP(Y.alloc((size_t)n * B * sizeof(double)));
    EVSL_HIP(Y2.alloc((size_t)n * B * sizeof(double)));
    EVSL_HIP(zero.alloc((size_t)n * sizeof(double)));
    EVSL_HIP(junk.alloc((size_t)n * sizeof(double)));
    if (B > Bcap) {
      EVSL_HIP(hipMemsetAsync(zero.p, 0, (size_t)n * sizeof(double), ctx().stream));
      Bcap = B;
    }
    f32 = fp32;
    return 0;
  }
  void* buf(int i, int n, int B) const {
    return bufs.as<char>() + (size_t)i * n * B * (f32 ? 4 : 8);
  }
  // uploads `tab` as the coefficient table of (key, kind) unless it is there
  template <typename Build>
  int coef_table(const std::vector<const polparams*>& key, int kind, Build build, CoefTab** out) {
    for (auto& t : tabs)
      if (t->kind == kind && t->key == key) {
        *out = t.get();
        return 0;
      }
    if (tabs.size() < kCoefTabs) {
      next_tab = tabs.size();
      tabs.push_back(std::make_unique<CoefTab>());
    }
    CoefTab& t = *tabs[next_tab];
    next_tab = (next_tab + 1) % kCoefTabs;
    std::vector<double> tab;
    t.off.clear();
    t.kind = -1;
    build(tab, t.off);
    // the copy below is ordered after the launches that read the old table
    EVSL_HIP(t.mus.alloc(tab.size() * sizeof(double)));
    EVSL_HIP(hipMemcpy(t.mus.p, tab.data(), tab.size() * sizeof(double), hipMemcpyHostToDevice));
    t.key = key;
    t.kind = kind;
    *out = &t;
    return 0;
  }
};

evsl_dev::ColPtrs col_ptrs(const double* const* p, int cnt) {
  evsl_dev::ColPtrs cp{};
  for (int i = 0; i < cnt; ++i) cp.p[i] = const_cast<double*>(p[i]);
  return cp;
}

// Columns of different degrees (b <= 8, every degree >= 3): ordered by
// decreasing degree, the series runs at width b up to the smallest degree,
// whose columns are then written out and dropped; the live recurrence
// vectors T_k, T_{k-1} and the partial sums Y are narrowed to the remaining
// columns, and so on.  An odd remainder of 3, 5 or 7 columns keeps one
// finished column as a passenger (zero coefficients, its output already
// written): odd widths have only the one-column-per-lane layout, and at
// 7 columns it ran 45.6 us a step against 30.5 us for 8 (5: 35.4 against
// 33.2 for 6; 3: 24.9 against 21.8 for 4; 1 stays 1, at 13.9 against 18.2
// for 2; FP32 on the 100^3 Laplacian).  Each column sees the same
// arithmetic as in one full-width run (per-column sums do not depend on the
// block width).
int filter_columns_phased(int b, const double* const* xin, double* const* yout,
                          const polparams* const* pols, bool f32, BlockWork& W) {
  Context& c = ctx();
  const int n = c.n;
  std::vector<int> ord(b);
  for (int i = 0; i < b; ++i) ord[i] = i;
  std::stable_sort(ord.begin(), ord.end(),
                   [&](int x, int y) { return pols[x]->deg > pols[y]->deg; });
  const int md = pols[ord[0]]->deg;
  if (int e = W.ensure(n, b, f32, md)) return e;
  std::vector<const double*> in(b);
  std::vector<double*> out(b);
  std::vector<const polparams*> key(b);
  for (int i = 0; i < b; ++i) {
    in[i] = xin[ord[i]];
    out[i] = yout[ord[i]];
    key[i] = pols[ord[i]];
  }
  // phase p runs degrees up to the smallest degree of its live columns, at
  // width `active` (the live columns and at most one passenger); its table
  // holds coefficient rows 0..kend for those columns, zero past a column's
  // degree.  The next phase keeps `keep` live columns at width `next`.
  auto phases = [&](auto&& visit) {
    int live = b, active = b, k0 = 1;
    while (live > 0) {
      const int kend = key[live - 1]->deg;
      int keep = live;
      while (keep > 0 && key[keep - 1]->deg == kend) --keep;
      const int next = (keep >= 3 && (keep & 1) && keep + 1 <= active) ? keep + 1 : keep;
      visit(active, live, k0, kend, keep, next);
      live = keep;
      active = next;
      k0 = kend + 1;
    }
  };
  BlockWork::CoefTab* ct = nullptr;
  if (int e = W.coef_table(key, 0, [&](std::vector<double>& tab, std::vector<size_t>& off) {
        phases([&](int active, int, int, int kend, int, int) {
          off.push_back(tab.size());
          tab.resize(tab.size() + (size_t)(kend + 1) * active, 0.0);
          double* t = tab.data() + off.back();
          for (int i = 0; i < active; ++i)
            for (int d = 0; d <= kend && d <= key[i]->deg; ++d)
              t[(size_t)d * active + i] = key[i]->mu[d];
        });
      }, &ct))
    return e;
  EVSL_HIP(evsl_dev::pack_cols(n, b, col_ptrs(in.data(), b), W.X0.p, f32, c.stream));
  FilterOp op;
  if (int e = make_filter_op(key[0]->cc, key[0]->dd, f32, &op)) return e;
  void* slot[3] = {W.buf(0, n, b), W.buf(1, n, b), W.buf(2, n, b)};
  void* Y = W.Y.p;
  void* Yspare = W.Y2.p;
  const size_t vs = f32 ? 4 : 8;
  int phase = 0, err = 0;
  phases([&](int active, int live, int k0, int kend, int keep, int next) {
    if (err) return;
    const double* mus_d = ct->mus.as<double>() + ct->off[phase++];
    if ((err = block_filter_seg(active, op, mus_d, k0, kend, W.X0.p, slot, Y))) return;
    hipError_t he = evsl_dev::unpack_range(n, active, keep, live, Y, false,
                                           col_ptrs(out.data() + keep, live - keep), c.stream);
    if (he == hipSuccess && next > 0 && next < active) {
      // T_kend sits in slot (kend-1)%3 and T_{kend-1} in slot (kend-2)%3
      // (kend >= 3); narrow them into the free slots and swap the pointers
      const int sa = (kend - 1) % 3, sb = (kend - 2) % 3, sf = kend % 3;
      void* pa = slot[sa];
      void* pb = slot[sb];
      void* pf = slot[sf];
      he = evsl_dev::narrow_cols(n, active, next, pa, pf, f32, c.stream);
      if (he == hipSuccess) he = evsl_dev::narrow_cols(n, active, next, pb, pa, f32, c.stream);
      slot[sa] = pf;
      slot[sb] = pa;
      slot[sf] = pb;
      if (he == hipSuccess) he = evsl_dev::narrow_cols(n, active, next, Y, Yspare, false, c.stream);
      std::swap(Y, Yspare);
      c.astats.filter_bytes += (2.0 * vs + 8.0) * (double)n * (active + next);
    }
    if (he != hipSuccess) {
      set_error("filter_columns_phased: unpack/narrow", he);
      err = EVSL_ERR_DEVICE;
    }
  });
  return err;
}

// y_c = p_c(A) x_c for columns given by device pointers (FP64 in/out), using
// the interleaved block filter, at most 32 columns per launch.  pols[c] may
// differ per column (same cc, dd).  Blocks wider than 8 are padded to 16 or
// 32 with zero columns whose output goes to a scratch vector.  Nothing here
// waits for the device.
// deferred: a series launch's outcome is left to the caller (series_failed at
// its next synchronisation); otherwise this waits for one.
int filter_columns(int ncols, const double* const* xin, double* const* yout,
                   const polparams* const* pols, bool f32, BlockWork& W, bool deferred = false) {
  Context& c = ctx();
  const int n = c.n;
  if (c.op != 1) {  // user operator: one column at a time through its MVFunc, FP64
    ChebWork cw;
    for (int j = 0; j < ncols; ++j)
      if (int e = cheb_av(pols[j], xin[j], yout[j], cw, EVSL_PREC_FP64)) return e;
    return 0;
  }
  int maxdeg = 0;
  for (int j = 0; j < ncols; ++j) maxdeg = std::max(maxdeg, pols[j]->deg);
  int mindeg = maxdeg;
  for (int j = 0; j < ncols; ++j) mindeg = std::min(mindeg, pols[j]->deg);
  FilterOp sop;
  if (mindeg > 0 && series_size(n, ncols))
    if (int e = make_filter_op(pols[0]->cc, pols[0]->dd, f32, &sop)) return e;
  if (series_fits(sop, ncols, mindeg)) {
    std::vector<const polparams*> key(pols, pols + ncols);
    BlockWork::CoefTab* ct = nullptr;
    // kind -2: the columns' coefficients one after the other
    if (int e = W.coef_table(key, -2, [&](std::vector<double>& tab, std::vector<size_t>& off) {
          for (const polparams* p : key) {
            off.push_back(tab.size());
            tab.insert(tab.end(), p->mu, p->mu + p->deg + 1);
          }
        }, &ct))
      return e;
    std::vector<SeriesCol> cols;
    for (int j = 0; j < ncols; ++j)
      cols.push_back({&sop, xin[j], yout[j], ct->mus.as<double>() + ct->off[j], 1,
                      pols[j]->deg});
    if (int e = series_launch(cols)) return e;
    if (deferred) return 0;
    EVSL_HIP(hipStreamSynchronize(c.stream));
    if (!series_failed()) return 0;
  }
  const int cap = filter_block_cap(c.A.view(), f32, evsl_dev::kCheb);
  for (int j0 = 0; j0 < ncols; j0 += cap) {
    const int b = std::min(cap, ncols - j0);
    const int B = kernel_width(b);
    if (int e = W.ensure(n, B, f32, maxdeg)) return e;
    std::vector<const double*> in(B);
    std::vector<double*> out(B);
    std::vector<const polparams*> key(pols + j0, pols + j0 + b);
    int md = 0;
    for (int cc = 0; cc < B; ++cc) {
      if (cc < b) {
        in[cc] = xin[j0 + cc];
        out[cc] = yout[j0 + cc];
        md = std::max(md, pols[j0 + cc]->deg);
      } else {
        in[cc] = W.zero.as<double>();
        out[cc] = W.junk.as<double>();
      }
    }
    if (md == 0) {  // degree-0 filters: y = mu0 x
      for (int cc = 0; cc < b; ++cc)
        EVSL_HIP(evsl_dev::scal_copy(n, pols[j0 + cc]->mu[0], in[cc], out[cc], c.stream));
      continue;
    }
    // mixed degrees in a block of at most 8 columns: run the series in
    // segments, dropping the columns whose degree is reached (every width
    // 1..8 has a kernel; wider blocks run all columns to the largest degree,
    // the others with zero coefficients)
    int dmin = md;
    for (int cc = 0; cc < b; ++cc) dmin = std::min(dmin, pols[j0 + cc]->deg);
    if (B == b && b > 1 && b <= 8 && dmin < md && dmin >= 3) {
      if (int e = filter_columns_phased(b, xin + j0, yout + j0, pols + j0, f32, W)) return e;
      continue;
    }
    BlockWork::CoefTab* ct = nullptr;
    if (int e = W.coef_table(key, B, [&](std::vector<double>& tab, std::vector<size_t>&) {
          tab.assign((size_t)(md + 1) * B, 0.0);
          for (int cc = 0; cc < b; ++cc)
            for (int d = 0; d <= key[cc]->deg; ++d) tab[(size_t)d * B + cc] = key[cc]->mu[d];
        }, &ct))
      return e;
    EVSL_HIP(evsl_dev::pack_cols(n, B, col_ptrs(in.data(), B), W.X0.p, f32, c.stream));
    void* bufs[3] = {W.buf(0, n, B), W.buf(1, n, B), W.buf(2, n, B)};
    FilterOp op;
    if (int e = make_filter_op(pols[j0]->cc, pols[j0]->dd, f32, &op)) return e;
    if (int e = block_filter(B, op, ct->mus.as<double>(), md, W.X0.p, bufs, W.Y.p)) return e;
    EVSL_HIP(evsl_dev::unpack_cols(n, B, W.Y.p, false, col_ptrs(out.data(), B), c.stream));
  }
  return 0;
}

// Cholesky of an m x m SPD matrix (column-major, upper factor R with G = R^T R)
bool cholesky_upper(int m, std::vector<double>& G) {
  for (int j = 0; j < m; ++j) {
    double d = G[(size_t)j * m + j];
    for (int k = 0; k < j; ++k) d -= G[(size_t)j * m + k] * G[(size_t)j * m + k];
    if (!(d > 0.0)) return false;
    d = std::sqrt(d);
    G[(size_t)j * m + j] = d;
    for (int i = j + 1; i < m; ++i) {
      double s = G[(size_t)i * m + j];
      for (int k = 0; k < j; ++k) s -= G[(size_t)j * m + k] * G[(size_t)i * m + k];
      G[(size_t)i * m + j] = s / d;  // R(j, i) stored at column i, row j
    }
  }
  return true;
}

// inverse of the upper-triangular R (column-major m x m) into Rinv (full, zeros below)
void invert_upper(int m, const std::vector<double>& R, std::vector<double>& Ri) {
  Ri.assign((size_t)m * m, 0.0);
  for (int j = 0; j < m; ++j) {
    Ri[(size_t)j * m + j] = 1.0 / R[(size_t)j * m + j];
    for (int i = j - 1; i >= 0; --i) {
      double s = 0.0;
      for (int k = i + 1; k <= j; ++k) s += R[(size_t)k * m + i] * Ri[(size_t)j * m + k];
      Ri[(size_t)j * m + i] = -s / R[(size_t)i * m + i];
    }
  }
}

// Column-wise W = A U (m columns, column-major n x m) via the blocked kernel
int apply_A_cols(int n, int m, const double* U, double* W, BlockWork& Wk) {
  Context& c = ctx();
  if (c.op != 1) {
    for (int j = 0; j < m; ++j)
      if (int e = apply_A(U + (size_t)j * n, W + (size_t)j * n)) return e;
    return 0;
  }
  const evsl_dev::Csr A = c.A.view();
  for (int j0 = 0; j0 < m; j0 += kBmaxPow) {
    const int b = std::min(kBmaxPow, m - j0);
    const int B = kernel_width(b);
    if (int e = Wk.ensure(n, B, false, 0)) return e;
    std::vector<const double*> in(B);
    std::vector<double*> out(B);
    for (int cc = 0; cc < B; ++cc) {
      in[cc] = cc < b ? U + (size_t)(j0 + cc) * n : Wk.zero.as<double>();
      out[cc] = cc < b ? W + (size_t)(j0 + cc) * n : Wk.junk.as<double>();
    }
    void* X = Wk.buf(0, n, B);
    void* Yb = Wk.buf(1, n, B);
    EVSL_HIP(evsl_dev::pack_cols(n, B, col_ptrs(in.data(), B), X, false, c.stream));
    EVSL_HIP(evsl_dev::cheb_spmm(A, B, false, evsl_dev::kPlain, X, nullptr, Yb, nullptr, nullptr,
                                 nullptr, nullptr, 1.0, 0.0, false, 0, nullptr, c.stream));
    EVSL_HIP(evsl_dev::unpack_cols(n, B, Yb, false, col_ptrs(out.data(), B), c.stream));
  }
  return 0;
}

// Per-slice Lanczos state
struct Slice {
  double intv[4];
  polparams* pol;
  DevBuf V;
  // FP32 copy of the basis read by the Gram-Schmidt passes (empty: they
  // read V); columns ld32 apart, ld32 even and >= n
  DevBuf V32;
  size_t ld32 = 0;
  std::vector<double> dT, eT;
  double beta = 0.0, wn = 0.0, tr0 = 0.0, old2 = 0.0, nrm = 0.0;
  int nwn = 0, kdim = 0, last_nconv = -1;
  bool active = true;
  double* vcol(int k, int n) const { return V.as<double>() + (size_t)k * n; }
  float* v32col(int k) const { return V32.as<float>() + (size_t)k * ld32; }
  bool has32() const { return V32.p != nullptr; }
};

// Z = p(A~) U for the m columns of U (FP64, column-major), in the form
// p(A~)U = U p(Theta~) + sum_k mu_k D_k with Theta~ the Rayleigh quotients
// of U, D_1 = R = A~U - U Theta~ (FP64) and
// D_{k+1} = 2 A~ D_k - D_{k-1} + 2 R T_k(Theta~).  The D recurrence runs in
// FP32 on the shifted matrix; its rounding scales with ||R||, not ||U||
// (relative error growing like k^1.5 eps_fp32).  A column whose residual is
// large (an unconverged or spurious Ritz vector: ||R|| > kFp64ResidualCut)
// would carry that much noise into the Rayleigh-Ritz space, where it couples
// to the converged vectors of nearby Rayleigh quotients; such columns are
// filtered in FP64 instead (p(A~)u directly).  On exit U holds Z; W is n x m
// scratch.
constexpr double kFp64ResidualCut = 1e-5;

int residual_filter(int n, int m, double* U, double* W, const polparams* pol, BlockWork& bw) {
  Context& c = ctx();
  const int deg = pol->deg;
  c.astats.n_refine_degcols += (size_t)m * deg;
  if (deg == 0) {
    for (int j = 0; j < m; ++j) EVSL_HIP(evsl_dev::scal(n, pol->mu[0], U + (size_t)j * n, c.stream));
    return 0;
  }
  const int nch = (n + 8191) / 8192;
  DevBuf part, th2, th, pv;
  EVSL_HIP(part.alloc((size_t)nch * m * sizeof(double)));
  EVSL_HIP(th2.alloc(m * sizeof(double)));
  EVSL_HIP(th.alloc(m * sizeof(double)));
  EVSL_HIP(pv.alloc(m * sizeof(double)));
  // W = A U, theta = (u.Au)/(u.u), R = (W - U theta)/dd  (R stored in W)
  if (int e = apply_A_cols(n, m, U, W, bw)) return e;
  EVSL_HIP(evsl_dev::col_dot(n, m, U, n, U, n, part.as<double>(), th2.as<double>(), c.stream));
  EVSL_HIP(evsl_dev::col_dot(n, m, W, n, U, n, part.as<double>(), th.as<double>(), c.stream));
  std::vector<double> uu(m), ua(m), thv(m), ths(m), rr(m);
  EVSL_HIP(hipMemcpy(uu.data(), th2.p, m * sizeof(double), hipMemcpyDeviceToHost));
  EVSL_HIP(hipMemcpy(ua.data(), th.p, m * sizeof(double), hipMemcpyDeviceToHost));
  for (int j = 0; j < m; ++j) {
    thv[j] = ua[j] / uu[j];
    ths[j] = (thv[j] - pol->cc) / pol->dd;
  }
  EVSL_HIP(hipMemcpy(th.p, thv.data(), m * sizeof(double), hipMemcpyHostToDevice));
  EVSL_HIP(evsl_dev::col_resid(n, m, W, n, U, n, th.as<double>(), 1.0 / pol->dd, W, n, c.stream));
  // residual norms (relative to the column's norm): the FP32 recurrence for
  // the small ones, FP64 filtering for the large ones
  EVSL_HIP(evsl_dev::col_dot(n, m, W, n, W, n, part.as<double>(), th2.as<double>(), c.stream));
  EVSL_HIP(hipMemcpy(rr.data(), th2.p, m * sizeof(double), hipMemcpyDeviceToHost));
  std::vector<int> small, big;
  for (int j = 0; j < m; ++j) {
    if (std::sqrt(std::max(rr[j], 0.0) / uu[j]) > kFp64ResidualCut)
      big.push_back(j);
    else
      small.push_back(j);
  }
  // p(theta~) per column (0 for the FP64-filtered columns: W then holds
  // their whole p(A~)u)
  std::vector<double> pth(m, 0.0);
  for (int j : small) evsl::chebxPltd(deg, pol->mu, 1, &ths[j], &pth[j]);
  EVSL_HIP(hipMemcpy(pv.p, pth.data(), m * sizeof(double), hipMemcpyHostToDevice));
  if (!big.empty()) {
    std::vector<const double*> in;
    std::vector<double*> out;
    std::vector<const polparams*> pp(big.size(), pol);
    for (int j : big) {
      in.push_back(U + (size_t)j * n);
      out.push_back(W + (size_t)j * n);
    }
    BlockWork bw64;
    if (int e = filter_columns((int)big.size(), in.data(), out.data(), pp.data(), false, bw64))
      return e;
    c.astats.n_refine_fp64_cols += big.size();
  }
  const int ms = (int)small.size();
  if (ms > 0) {
    FilterOp op;
    if (int e = make_filter_op(pol->cc, pol->dd, true, &op)) return e;
    // per-launch coefficient tables of every chunk, uploaded once:
    // g[chunk][k][c] = 2 T_k(theta~_c), k = 1..deg-1; pairs (mu_{k+1}, mu_1)
    const int cap = filter_block_cap(op.A, true, evsl_dev::kRes);
    const int nchunk = (ms + cap - 1) / cap;
    const size_t gstride = (size_t)(deg + 1) * cap;
    std::vector<double> g(gstride * nchunk, 0.0), mp((size_t)2 * (deg + 1), 0.0);
    for (int j0 = 0, ch = 0; j0 < ms; j0 += cap, ++ch) {
      const int b = std::min(cap, ms - j0);
      const int B = kernel_width(b);
      for (int cc = 0; cc < b; ++cc) {
        const double x = ths[small[j0 + cc]];
        double tkm1 = 1.0, tk = x;
        for (int k = 1; k < deg; ++k) {
          g[gstride * ch + (size_t)k * B + cc] = 2.0 * tk;
          const double tkp1 = 2.0 * x * tk - tkm1;
          tkm1 = tk;
          tk = tkp1;
        }
      }
    }
    for (int k = 1; k < deg; ++k) {
      mp[2 * k] = pol->mu[k + 1];
      mp[2 * k + 1] = pol->mu[1];
    }
    DevBuf g_d, mp_d;
    EVSL_HIP(g_d.alloc(g.size() * sizeof(double)));
    EVSL_HIP(mp_d.alloc(mp.size() * sizeof(double)));
    EVSL_HIP(hipMemcpy(g_d.p, g.data(), g.size() * sizeof(double), hipMemcpyHostToDevice));
    EVSL_HIP(hipMemcpy(mp_d.p, mp.data(), mp.size() * sizeof(double), hipMemcpyHostToDevice));
    for (int j0 = 0, ch = 0; j0 < ms; j0 += cap, ++ch) {
      const int b = std::min(cap, ms - j0);
      const int B = kernel_width(b);
      if (int e = bw.ensure(n, B, true, deg)) return e;
      // R columns -> FP32 block (xk of the first launch = D_1 = R); the same
      // block is the v0 operand (R) of every launch
      std::vector<const double*> in(B);
      std::vector<double*> out(B);
      for (int cc = 0; cc < B; ++cc) {
        in[cc] = cc < b ? W + (size_t)small[j0 + cc] * n : bw.zero.as<double>();
        out[cc] = cc < b ? W + (size_t)small[j0 + cc] * n : bw.junk.as<double>();
      }
      EVSL_HIP(evsl_dev::pack_cols(n, B, col_ptrs(in.data(), B), bw.X0.p, true, c.stream));
      void* X0 = bw.X0.p;  // R (FP32) = D_1
      void* bufs[3] = {bw.buf(0, n, B), bw.buf(1, n, B), bw.buf(2, n, B)};
      void* Yb = bw.Y.p;
      const double* gch = g_d.as<double>() + gstride * ch;
      if (deg == 1) {
        // Y = mu_1 R (W already holds R in FP64)
        for (int cc = 0; cc < b; ++cc)
          EVSL_HIP(evsl_dev::scal(n, pol->mu[1], W + (size_t)small[j0 + cc] * n, c.stream));
      } else {
        for (int k = 1; k < deg; ++k) {
          void* xkp1 = bufs[(k - 1) % 3];
          const void* xk = (k == 1) ? X0 : bufs[(k - 2) % 3];
          const void* xkm1 = (k == 1) ? nullptr : (k == 2 ? X0 : bufs[(k - 3) % 3]);
          const int yf = evsl_dev::y_flush(k, deg - 1);
          EVSL_HIP(evsl_dev::cheb_spmm(op.A, B, true, evsl_dev::kRes, xk, xkm1, xkp1, Yb, X0,
                                       gch + (size_t)k * B, mp_d.as<double>() + 2 * k, op.t2,
                                       op.cc, k == 1, yf, nullptr, c.stream));
          // the kCheb streams plus the residual block R
          c.astats.refine_bytes += c.A.mat_bytes(4, B) +
                                   (evsl_dev::cheb_vec_bytes(yf, k == 1, 4) + 4.0) * B * n;
        }
        EVSL_HIP(evsl_dev::unpack_cols(n, B, Yb, false, col_ptrs(out.data(), B), c.stream));
      }
    }
  }
  // U <- U p(theta~) + Y
  EVSL_HIP(evsl_dev::col_scale_add(n, m, U, n, pv.as<double>(), W, n, c.stream));
  return 0;
}

}  // namespace

// Ritz pairs of one converged slice.  FP64 mode: the reference's extraction
// (ritz of T above bar, SRC/cheblanNr.c:316-399).  Mixed mode: guard-extended
// Ritz block, FP64 filter pass(es), Cholesky QR and FP64 Rayleigh-Ritz.
int refine_extract(int n, int kdim, const double* dT, const double* eT, const double* V,
                   const polparams* pol, const double* intv, double tol, bool mixed,
                   int* nevOut, double** lamo, double** Wo, double** reso, FILE* fstats,
                   bool* stalled, double guard) {
  Context& c = ctx();
  if (stalled) *stalled = false;
  const double bar = pol->bar, aa = intv[0], bb = intv[1];
  std::vector<double> eval(kdim), e(kdim + 1, 0.0);
  std::memcpy(eval.data(), dT, kdim * sizeof(double));
  if (kdim > 1) std::memcpy(e.data(), eT, (kdim - 1) * sizeof(double));
  RotationLog rec;
  if (int err = tridiag_ql(kdim, eval.data(), e.data(), &rec)) return err;
  // guard threshold (default 0.8 bar): keep Ritz values of p(A) so that
  // eigenvectors just outside [a, b] are in the Rayleigh-Ritz space
  const double thr = mixed ? (guard > 0.0 ? guard : c.refine_guard) * bar : bar;
  std::vector<int> sel;
  for (int i = 0; i < kdim; ++i)
    if (!(eval[i] < thr)) sel.push_back(i);
  int m = (int)sel.size();
  if (mixed) c.astats.n_refine_cols += m;
  if (fstats) {
    int above = 0;
    for (int i = 0; i < kdim; ++i) above += !(eval[i] < bar);
    std::fprintf(fstats, "  extract: kdim %d, Ritz values >= bar %d, candidates %d (thr %.3f)\n",
                 kdim, above, m, thr);
  }
  const int alloc = std::max(kdim, m) + 1;
  double* Lam = (double*)std::malloc(alloc * sizeof(double));
  double* res = (double*)std::malloc(alloc * sizeof(double));
  *lamo = Lam;
  *reso = res;
  *Wo = nullptr;
  *nevOut = 0;
  if (m == 0) return 0;
  DevBuf Zsel, U, W, part, s2, tv, r2;
  EVSL_HIP(Zsel.alloc((size_t)kdim * m * sizeof(double)));
  if (int err = tridiag_rotations_to_device(kdim, rec, sel, Zsel.as<double>())) return err;
  EVSL_HIP(U.alloc((size_t)n * m * sizeof(double)));
  EVSL_HIP(W.alloc((size_t)n * m * sizeof(double)));
  double* Ud = U.as<double>();
  double* Wd = W.as<double>();
  EVSL_HIP(evsl_dev::gemm_nn(n, m, kdim, V, n, Zsel.as<double>(), kdim, Ud, n, c.stream));
  Zsel.release();
  BlockWork bw;
  const int nch = (n + 8191) / 8192;
  EVSL_HIP(part.alloc((size_t)nch * m * sizeof(double)));
  EVSL_HIP(s2.alloc(m * sizeof(double)));
  EVSL_HIP(tv.alloc(m * sizeof(double)));
  EVSL_HIP(r2.alloc(m * sizeof(double)));
  std::vector<double> hs2(m), ht(m), hr2(m);
  // Rayleigh quotients and residual norms of the columns of Ud (A U in Wd);
  // s2 holds the squared column norms, computed by the caller
  auto measure = [&]() -> int {
    EVSL_HIP(evsl_dev::col_dot(n, m, Wd, n, Ud, n, part.as<double>(), tv.as<double>(), c.stream));
    EVSL_HIP(evsl_dev::col_res2(n, m, Wd, n, Ud, n, tv.as<double>(), part.as<double>(),
                                r2.as<double>(), c.stream));
    EVSL_HIP(hipMemcpy(hs2.data(), s2.p, m * sizeof(double), hipMemcpyDeviceToHost));
    EVSL_HIP(hipMemcpy(ht.data(), tv.p, m * sizeof(double), hipMemcpyDeviceToHost));
    EVSL_HIP(hipMemcpy(hr2.data(), r2.p, m * sizeof(double), hipMemcpyDeviceToHost));
    return 0;
  };
  if (!mixed) {
    EVSL_HIP(evsl_dev::col_dot(n, m, Ud, n, Ud, n, part.as<double>(), s2.as<double>(), c.stream));
    EVSL_HIP(evsl_dev::col_scale_rsqrt(n, m, Ud, n, s2.as<double>(), c.stream));
    if (int err = apply_A_cols(n, m, Ud, Wd, bw)) return err;
    if (int err = measure()) return err;
  } else {
    // Refinement passes: filter the block with p(A) (FP32 residual
    // recurrence), re-orthonormalize (Cholesky QR twice) and extract Ritz
    // pairs with A in FP64.  Beyond the requested passes, more run while a
    // Ritz value inside [a, b] is close to converged (tol <= residual <
    // kRetryFactor * tol): a pass damps the components outside the guard set
    // by the guard ratio, so such a pair needs a few.  They go on while the
    // largest near-converged residual falls by kProgress per pass, at most
    // kMaxExtraPasses; then the slice counts as stalled.
    constexpr int kMaxExtraPasses = 8;
    constexpr double kRetryFactor = 1e3;
    constexpr double kProgress = 0.9;
    double last_near = 0.0;
    // the first pass's polynomial: the interval widened by refine_widen
    // slice widths on each side, same damping and thresholds (a lower
    // degree; the FP32-filtered basis carries rounding noise spread over
    // the whole spectrum, and the residual weighs a component by its
    // eigenvalue's distance, so the far part is what a pass must damp)
    polparams qpol = *pol;
    qpol.mu = nullptr;
    bool have_q = false;
    if (c.refine_widen > 0.0) {
      const double w = bb - aa, lmin = intv[2], lmax = intv[3];
      double qiv[4] = {std::max(lmin, aa - c.refine_widen * w),
                       std::min(lmax, bb + c.refine_widen * w), lmin, lmax};
      qpol.deg = 0;
      if (find_pol(qiv, &qpol) == 0 && qpol.deg < pol->deg && qpol.cc == pol->cc &&
          qpol.dd == pol->dd)
        have_q = true;
      else
        free_pol(&qpol);
    }
    struct PolGuard {
      polparams* p;
      ~PolGuard() { free_pol(p); }
    } qguard{&qpol};
    if (fstats) {
      // residuals of the Ritz vectors as the FP32-filtered basis gives them
      EVSL_HIP(evsl_dev::col_dot(n, m, Ud, n, Ud, n, part.as<double>(), s2.as<double>(),
                                 c.stream));
      if (int err = apply_A_cols(n, m, Ud, Wd, bw)) return err;
      if (int err = measure()) return err;
      double rmax = 0.0;
      int in_ab = 0, below = 0;
      for (int j = 0; j < m; ++j) {
        const double t = ht[j] / hs2[j];
        if (t < aa - kEpsM || t > bb + kEpsM) continue;
        const double r = std::sqrt(std::max(hr2[j], 0.0) / hs2[j]);
        ++in_ab;
        below += r < tol;
        rmax = std::max(rmax, r);
      }
      std::fprintf(fstats,
                   "  refinement: first pass degree %d (filter %d); before it %d Ritz values "
                   "in [a,b], %d below tol, max residual %.3e\n",
                   have_q ? qpol.deg : pol->deg, pol->deg, in_ab, below, rmax);
    }
    DevBuf G, gp, M, U2;
    EVSL_HIP(G.alloc((size_t)m * m * sizeof(double)));
    EVSL_HIP(gp.alloc(evsl_dev::gemm_tn_part_elems(n, m, m) * sizeof(double)));
    EVSL_HIP(M.alloc((size_t)m * m * sizeof(double)));
    EVSL_HIP(U2.alloc((size_t)n * m * sizeof(double)));
    const int min_pass = std::max(c.refine_passes, 1);
    for (int pass = 0;; ++pass) {
      if (int err = residual_filter(n, m, Ud, Wd, pass == 0 && have_q ? &qpol : pol, bw))
        return err;
      if (pass > 0) c.astats.n_refine_cols += m;
      // Cholesky QR: G = U^T U = R^T R, U <- U R^-1
      for (int qr = 0; qr < 2; ++qr) {
        EVSL_HIP(evsl_dev::gemm_tn(n, m, m, Ud, n, Ud, n, G.as<double>(), m, gp.as<double>(),
                                   c.stream));
        std::vector<double> Gh((size_t)m * m), Ri;
        EVSL_HIP(hipMemcpy(Gh.data(), G.p, Gh.size() * sizeof(double), hipMemcpyDeviceToHost));
        for (int j = 0; j < m; ++j)  // symmetrize
          for (int i = 0; i < j; ++i) {
            const double a = 0.5 * (Gh[(size_t)j * m + i] + Gh[(size_t)i * m + j]);
            Gh[(size_t)j * m + i] = Gh[(size_t)i * m + j] = a;
          }
        if (!cholesky_upper(m, Gh)) {
          set_error_msg("refinement: Ritz block lost rank in Cholesky QR");
          return EVSL_ERR_EIG;
        }
        invert_upper(m, Gh, Ri);
        EVSL_HIP(hipMemcpy(M.p, Ri.data(), Ri.size() * sizeof(double), hipMemcpyHostToDevice));
        EVSL_HIP(evsl_dev::gemm_nn(n, m, m, Ud, n, M.as<double>(), m, Wd, n, c.stream));
        std::swap(Ud, Wd);
      }
      // Rayleigh-Ritz with A in FP64: H = U^T A U
      if (int err = apply_A_cols(n, m, Ud, Wd, bw)) return err;
      EVSL_HIP(evsl_dev::gemm_tn(n, m, m, Ud, n, Wd, n, G.as<double>(), m, gp.as<double>(),
                                 c.stream));
      std::vector<double> Hh((size_t)m * m), Q((size_t)m * m), lam_rr(m);
      EVSL_HIP(hipMemcpy(Hh.data(), G.p, Hh.size() * sizeof(double), hipMemcpyDeviceToHost));
      for (int j = 0; j < m; ++j)
        for (int i = 0; i < j; ++i) {
          const double a = 0.5 * (Hh[(size_t)j * m + i] + Hh[(size_t)i * m + j]);
          Hh[(size_t)j * m + i] = Hh[(size_t)i * m + j] = a;
        }
      if (int err = sym_eig_host(m, Hh.data(), m, Q.data(), m, lam_rr.data())) return err;
      EVSL_HIP(hipMemcpy(M.p, Q.data(), Q.size() * sizeof(double), hipMemcpyHostToDevice));
      // rotate U and W = A U by Q: U2 = Ritz vectors, Ud = A * Ritz vectors
      EVSL_HIP(evsl_dev::gemm_nn(n, m, m, Ud, n, M.as<double>(), m, U2.as<double>(), n, c.stream));
      EVSL_HIP(evsl_dev::gemm_nn(n, m, m, Wd, n, M.as<double>(), m, Ud, n, c.stream));
      EVSL_HIP(hipMemcpyAsync(Wd, U2.p, (size_t)n * m * sizeof(double), hipMemcpyDeviceToDevice,
                              c.stream));
      std::swap(Ud, Wd);  // Ud = Ritz vectors, Wd = A * Ritz vectors
      EVSL_HIP(evsl_dev::col_dot(n, m, Ud, n, Ud, n, part.as<double>(), s2.as<double>(),
                                 c.stream));
      if (int err = measure()) return err;
      if (pass + 1 < min_pass) continue;
      int near = 0;
      double near_max = 0.0;
      for (int j = 0; j < m; ++j) {
        const double r = std::sqrt(std::max(hr2[j], 0.0));
        if (ht[j] >= aa - kEpsM && ht[j] <= bb + kEpsM && !(r < tol) &&
            r < kRetryFactor * tol) {
          ++near;
          near_max = std::max(near_max, r);
        }
      }
      if (fstats)
        std::fprintf(fstats, "  refinement pass %d: %d near-converged in [a,b] (max %.3e)\n",
                     pass + 1, near, near_max);
      if (near == 0) break;
      const bool progress = pass + 1 == min_pass || near_max < kProgress * last_near;
      last_near = near_max;
      if (pass + 1 >= min_pass + kMaxExtraPasses || !progress) {
        // the passes no longer close the gap to tol (a filter too weak to
        // separate the guard set): the caller may redo the slice in FP64
        if (stalled) *stalled = true;
        break;
      }
      ++c.astats.n_refine_extra;
    }
  }
  std::vector<int> keep;
  int nev = 0;
  for (int j = 0; j < m; ++j) {
    if (hs2[j] == 0.0) return 2;
    const double t = ht[j];
    if (t < aa - kEpsM || t > bb + kEpsM) continue;
    const double r = std::sqrt(std::max(hr2[j], 0.0));
    if (fstats && !(r < tol))
      std::fprintf(fstats, "  rejected in [a,b]: lambda %.12f residual %.3e\n", t, r);
    if (r < tol) {
      Lam[nev] = t;
      res[nev] = r;
      keep.push_back(j);
      ++nev;
    }
  }
  *nevOut = nev;
  if (nev > 0) {
    double* Y = (double*)_evsl_Malloc_device((size_t)n * nev * sizeof(double));
    if (!Y) return EVSL_ERR_ALLOC;
    DevBuf idx;
    EVSL_HIP(idx.alloc(nev * sizeof(int)));
    EVSL_HIP(hipMemcpy(idx.p, keep.data(), nev * sizeof(int), hipMemcpyHostToDevice));
    EVSL_HIP(evsl_dev::gather_cols(n, nev, Ud, n, idx.as<int>(), Y, n, c.stream));
    EVSL_HIP(hipStreamSynchronize(c.stream));
    *Wo = Y;
  }
  return 0;
}

// ---- LanczosGroup ----------------------------------------------------------
// Slices of one matrix (shared lmin, lmax) advance through the recurrence of
// ChebLanNr (SRC/cheblanNr.c:150-310) together: every step filters the
// current Lanczos vector of each active slice in one blocked pass (one per
// filter precision), then runs each slice's recurrence, DGKS
// re-orthogonalisation and (at its own test points) the convergence test.  A
// slice added between steps starts with the next step: its start vector is
// filtered with the other new slices' and normalised, then it takes its first
// Lanczos step.  Each slice counts its own steps, so its arithmetic (and
// result) does not depend on which other slices share the group or when they
// joined.
//
// In the mixed form a slice filters in FP32 only when its polynomial degree
// lies in a range (evsl_amd_set_mixed_degree_range, default [32, 20000]): a
// lower-degree filter carries few of the bytes (the re-orthogonalisation
// dominates) and separates the refinement's guard set too weakly (an end
// interval's degree-4 filter left every pair at ~2e-7 after three refinement
// passes).  At high degrees (7250 on the Anderson model at band centre) the
// FP64 sum of the series and the lower-degree first refinement pass keep the
// refinement's FP32 residual recurrence short and its noise low.  A mixed
// slice whose refinement still stalls above tol is run again from its start
// vector in FP64.

struct LanczosGroup::Impl {
  struct Slot {
    Slice L;
    int maxit = 0, k = 0;
    double tol = 0;
    bool f32 = false;
    const double* v0 = nullptr;
    SliceResult* out = nullptr;
    int state = 0;  // 0 free, 1 start pending, 2 active
  };
  bool mixed = false;
  FILE* fstats = nullptr;
  std::vector<std::unique_ptr<Slot>> slots;
  DevBuf gt_part, hbuf, scal_d, vrand, parts;
  int kcap = 0, scap = 0;
  size_t gt_stride = 0;
  BlockWork bw32, bw64;  // the FP32 and the FP64 blocked filter passes
  std::vector<int> st_cur, act_cur;  // slots of the phase in progress
  // filters the columns in -> out of this group's matrix, one pass per
  // precision
  int filter(const std::vector<LanczosGroup::FilterCol>& cols) {
    for (int pr = 0; pr < 2; ++pr) {
      std::vector<const double*> ii;
      std::vector<double*> oo;
      std::vector<const polparams*> pp;
      for (const auto& col : cols)
        if (col.f32 == (pr == 1)) {
          ii.push_back(col.in);
          oo.push_back(col.out);
          pp.push_back(col.pol);
        }
      if (ii.empty()) continue;
      if (int e = filter_columns((int)ii.size(), ii.data(), oo.data(), pp.data(), pr == 1,
                                 pr == 1 ? bw32 : bw64, true))
        return e;
    }
    return 0;
  }
  // (re)starts slot s: a fresh recurrence from its start vector
  int start(int s, bool f32) {
    Slot& sl = *slots[s];
    const int n = ctx().n;
    sl.L.dT.assign(sl.maxit, 0.0);
    sl.L.eT.assign(sl.maxit, 0.0);
    sl.L.beta = sl.L.wn = sl.L.tr0 = sl.L.old2 = sl.L.nrm = 0.0;
    sl.L.nwn = sl.L.kdim = 0;
    sl.L.last_nconv = -1;
    sl.L.active = true;
    sl.k = 0;
    sl.f32 = f32;
    sl.state = 1;
    EVSL_HIP(sl.L.V.alloc((size_t)n * (sl.maxit + 1) * sizeof(double)));
    if (f32 && ctx().fp32_basis) {
      sl.L.ld32 = ((size_t)n + 63) / 64 * 64;
      EVSL_HIP(sl.L.V32.alloc(sl.L.ld32 * (sl.maxit + 1) * sizeof(float)));
    } else {
      sl.L.V32.release();
      sl.L.ld32 = 0;
    }
    return 0;
  }
  // one Gram-Schmidt pass of vnew against the slice's first k + 1 basis
  // vectors (the FP32 copy when the slice has one); the partials of
  // ||vnew||^2 go to part, their count to *nparts
  int cgs_pass(Slice& L, int k, double* vnew, double* part, int* nparts) {
    const int n = ctx().n;
    hipStream_t st = ctx().stream;
    if (L.has32()) {
      EVSL_HIP(evsl_dev::gemv_t_f32(n, k + 1, L.V32.as<float>(), L.ld32, vnew,
                                    gt_part.as<double>(), hbuf.as<double>(), st));
      EVSL_HIP(evsl_dev::gemv_n_sub_nrm_f32(n, k + 1, L.V32.as<float>(), L.ld32,
                                            hbuf.as<double>(), vnew, part, st));
      *nparts = evsl_dev::gemv_n_sub_f32_blocks(n);
      return 0;
    }
    EVSL_HIP(evsl_dev::gemv_t(n, k + 1, L.V.as<double>(), n, vnew, gt_part.as<double>(),
                              hbuf.as<double>(), st));
    EVSL_HIP(evsl_dev::gemv_n_sub_nrm(n, k + 1, L.V.as<double>(), n, hbuf.as<double>(), vnew,
                                      part, st));
    *nparts = (n + evsl_dev::kWG - 1) / evsl_dev::kWG;
    return 0;
  }
  // bytes one Gram-Schmidt pass against k + 1 vectors reads and writes
  static double cgs_bytes(const Slice& L, int n, int k) {
    return (L.has32() ? 8.0 : 16.0) * n * (k + 1) + 24.0 * n;
  }
  // basis column k: scale by a, and write its FP32 copy when there is one
  int scal_col(Slice& L, int k, double a) {
    const int n = ctx().n;
    if (L.has32()) {
      EVSL_HIP(evsl_dev::scal_f32copy(n, a, L.vcol(k, n), L.v32col(k), ctx().stream));
    } else {
      EVSL_HIP(evsl_dev::scal(n, a, L.vcol(k, n), ctx().stream));
    }
    return 0;
  }
  // the column of slot s at its step k: vnew against the first k + 1 basis vectors
  evsl_dev::LanCol lan_col(int s) {
    Slot& sl = *slots[s];
    Slice& L = sl.L;
    const int n = ctx().n, k = sl.k;
    evsl_dev::LanCol q{};
    q.zold = k > 0 ? L.vcol(k - 1, n) : nullptr;
    q.v = L.vcol(k, n);
    q.vnew = L.vcol(k + 1, n);
    q.V = L.V.as<double>();
    q.V32 = L.V32.as<float>();
    q.ld32 = L.ld32;
    q.beta = L.beta;
    q.part = part_of(s);
    q.out = scal_d.as<double>() + 4 * s;
    q.k = k + 1;
    return q;
  }
  // runs `go(columns, count)` over the slots, at most kLanCols at a time
  template <typename Go>
  int by_cols(const std::vector<int>& ids, Go go) {
    for (size_t i0 = 0; i0 < ids.size(); i0 += evsl_dev::kLanCols) {
      evsl_dev::LanCols cols{};
      const int nc = (int)std::min((size_t)evsl_dev::kLanCols, ids.size() - i0);
      for (int j = 0; j < nc; ++j) {
        cols.c[j] = lan_col(ids[i0 + j]);
        cols.c[j].gt = gt_part.as<double>() + gt_stride * j;
      }
      if (int e = go(cols, nc, &ids[i0])) return e;
    }
    return 0;
  }
  // A Gram-Schmidt pass of the slots' new vectors and the sums of their norms
  // (second: of a further pass).  Small matrices: the slots of one basis
  // precision together; the others one after the other.
  int cgs_all(const std::vector<int>& ids, bool second) {
    Context& c = ctx();
    const int n = c.n;
    const bool small = evsl_dev::lan_small(n);
    for (int f32 = 0; f32 < 2; ++f32) {
      std::vector<int> sub;
      for (int s : ids)
        if (slots[s]->L.has32() == (f32 == 1)) sub.push_back(s);
      if (int e = by_cols(sub, [&](evsl_dev::LanCols& cols, int nc, const int* id) -> int {
            if (small) {
              EVSL_HIP(evsl_dev::lan_gram_schmidt(n, cols, nc, f32 == 1, c.stream));
            } else {
              for (int j = 0; j < nc; ++j)
                if (int e2 = cgs_pass(slots[id[j]]->L, slots[id[j]]->k, cols.c[j].vnew,
                                      cols.c[j].part + 2 * evsl_dev::kRedBlocks, &cols.c[j].np))
                  return e2;
            }
            EVSL_HIP(evsl_dev::lan_sums(n, cols, nc, second, c.stream));
            return 0;
          }))
        return e;
    }
    return 0;
  }
  hipEvent_t ev[3] = {nullptr, nullptr, nullptr};
  size_t part_stride() const { return evsl_dev::lan_part_elems(ctx().n); }
  double* part_of(int s) { return parts.as<double>() + (size_t)s * part_stride(); }
  int ensure(int maxit) {
    const int n = ctx().n;
    const int ns = (int)slots.size();
    // V^T w partials of kLanCols columns side by side where they run together
    kcap = std::max(kcap, maxit);
    gt_stride = (size_t)evsl_dev::gemv_t_chunks(n) * (kcap + 1);
    EVSL_HIP(gt_part.alloc(gt_stride * (evsl_dev::lan_small(n) ? evsl_dev::kLanCols : 1) *
                           sizeof(double)));
    EVSL_HIP(hbuf.alloc((size_t)(kcap + 1) * sizeof(double)));
    if (ns > scap) {
      EVSL_HIP(scal_d.alloc((size_t)4 * ns * sizeof(double)));
      EVSL_HIP(parts.alloc(part_stride() * ns * sizeof(double)));
      scap = ns;
    }
    EVSL_HIP(vrand.alloc((size_t)n * sizeof(double)));
    return 0;
  }
};

bool mixed_slice_fp32(const polparams* pol) {
  const Context& c = ctx();
  const bool capped =
      c.mixed_capped_fp64 && pol->max_deg > 0 && pol->deg >= pol->max_deg - 1;
  return !capped && pol->deg >= c.mixed_min_deg && pol->deg <= c.mixed_max_deg;
}

size_t slice_basis_bytes(int n, int maxit, bool mixed, const polparams* pol) {
  size_t b = (size_t)n * (maxit + 2) * sizeof(double);
  if (mixed && ctx().fp32_basis && mixed_slice_fp32(pol))
    b += ((size_t)n + 63) / 64 * 64 * (maxit + 1) * sizeof(float);
  return b;
}

LanczosGroup::LanczosGroup(bool mixed, FILE* fstats) : p_(new Impl) {
  p_->mixed = mixed;
  p_->fstats = fstats;
}

LanczosGroup::~LanczosGroup() {
  for (auto& e : p_->ev)
    if (e) (void)hipEventDestroy(e);
}

int LanczosGroup::active() const {
  int a = 0;
  for (auto& s : p_->slots) a += s->state != 0;
  return a;
}

int LanczosGroup::add(const double* intv, int maxit, double tol, const double* v0,
                      const polparams* pol, SliceResult* out) {
  Impl& g = *p_;
  Context& c = ctx();
  *out = SliceResult();
  if (intv[0] >= intv[1] || intv[0] >= intv[3] || intv[1] <= intv[2]) {
    out->done = true;  // empty result, as ChebLanNr on an invalid interval
    out->t_done = evsl_timer();
    return 0;
  }
  if (pol->gam > 1.0 || pol->gam < -1.0) {
    out->err = -1;
    out->done = true;
    out->t_done = evsl_timer();
    return 0;
  }
  int s = -1;
  for (int i = 0; i < (int)g.slots.size(); ++i)
    if (g.slots[i]->state == 0) {
      s = i;
      break;
    }
  if (s < 0) {
    g.slots.push_back(nullptr);
    s = (int)g.slots.size() - 1;
  }
  g.slots[s] = std::make_unique<Impl::Slot>();  // a fresh slot (a finished one is reused)
  Impl::Slot& sl = *g.slots[s];
  std::memcpy(sl.L.intv, intv, 4 * sizeof(double));
  sl.L.pol = const_cast<polparams*>(pol);
  sl.maxit = std::min(c.n, maxit);
  sl.tol = tol;
  sl.v0 = v0;
  sl.out = out;
  // FP32 filter only for degrees in the mixed range, and only for a filter
  // that met find_pol's damping thresholds: one that ran out of degrees
  // (deg = max_deg - 1, SRC/chebpoly.c:363-490) separates its interval
  // weakly, its slice tends to end at maxit, and there the FP32-filtered
  // basis leaves pairs just above tol and the slice would be redone in FP64
  const bool f32 = g.mixed && mixed_slice_fp32(pol);
  if (g.mixed && !f32) ++c.astats.n_fp64_slices;
  if (int e = g.start(s, f32)) return e;
  return g.ensure(sl.maxit);
}

int LanczosGroup::start_cols(std::vector<FilterCol>& cols) {
  Impl& g = *p_;
  const int n = ctx().n;
  g.st_cur.clear();
  for (int s = 0; s < (int)g.slots.size(); ++s)
    if (g.slots[s]->state == 1) {
      g.st_cur.push_back(s);
      Impl::Slot& sl = *g.slots[s];
      cols.push_back({sl.v0, sl.L.vcol(0, n), sl.L.pol, sl.f32});
    }
  return 0;
}

// the new slices' filtered start vectors: normalise, make the slices active
int LanczosGroup::start_done() {
  Impl& g = *p_;
  Context& c = ctx();
  const int n = c.n;
  if (g.st_cur.empty()) return 0;
  double* sc_d = g.scal_d.as<double>();
  for (int s : g.st_cur) {
    double* v = g.slots[s]->L.vcol(0, n);
    EVSL_HIP(evsl_dev::dot_partial(n, v, v, g.part_of(s), c.stream));
    EVSL_HIP(evsl_dev::sum_scalar(g.part_of(s), evsl_dev::kRedBlocks, sc_d + 4 * s, c.stream));
  }
  std::vector<double> nv(4 * g.slots.size());
  EVSL_HIP(hipMemcpy(nv.data(), sc_d, nv.size() * sizeof(double), hipMemcpyDeviceToHost));
  for (int s : g.st_cur) {
    if (int e = g.scal_col(g.slots[s]->L, 0, 1.0 / std::sqrt(nv[4 * s]))) return e;
    g.slots[s]->state = 2;
  }
  g.st_cur.clear();
  return 0;
}

int LanczosGroup::step_cols(std::vector<FilterCol>& cols) {
  Impl& g = *p_;
  const int n = ctx().n;
  g.act_cur.clear();
  for (int s = 0; s < (int)g.slots.size(); ++s)
    if (g.slots[s]->state == 2) {
      g.act_cur.push_back(s);
      Impl::Slot& sl = *g.slots[s];
      cols.push_back({sl.L.vcol(sl.k, n), sl.L.vcol(sl.k + 1, n), sl.L.pol, sl.f32});
    }
  return 0;
}

int LanczosGroup::filter_cols(const std::vector<FilterCol>& cols) { return p_->filter(cols); }

int LanczosGroup::step() {
  Impl& g = *p_;
  Context& c = ctx();
  if (!g.ev[0])
    for (auto& e : g.ev) EVSL_HIP(hipEventCreate(&e));
  auto elapsed = [](hipEvent_t a, hipEvent_t b) {
    float ms = 0.f;
    if (hipEventSynchronize(b) != hipSuccess || hipEventElapsedTime(&ms, a, b) != hipSuccess)
      return 0.0;
    return ms * 1e-3;
  };
  // new slices: filter their start vectors together, normalise
  std::vector<FilterCol> cols;
  if (int e = start_cols(cols)) return e;
  if (!cols.empty()) {
    do {  // once, or again by launches where a series launch has failed
      EVSL_HIP(hipEventRecord(g.ev[0], c.stream));
      if (int e = g.filter(cols)) return e;
      EVSL_HIP(hipEventRecord(g.ev[1], c.stream));
      c.astats.t_filter += elapsed(g.ev[0], g.ev[1]);
    } while (series_failed());
    if (int e = start_done()) return e;
  }
  // one blocked filter pass for all active slices
  cols.clear();
  if (int e = step_cols(cols)) return e;
  if (cols.empty()) return 0;
  do {
    EVSL_HIP(hipEventRecord(g.ev[0], c.stream));
    if (int e = g.filter(cols)) return e;
    EVSL_HIP(hipEventRecord(g.ev[1], c.stream));
    c.astats.t_filter += elapsed(g.ev[0], g.ev[1]);
  } while (series_failed());
  return step_done();
}

// the rest of the step once the active slices' vectors are filtered:
// recurrence, re-orthogonalisation, convergence tests, results
int LanczosGroup::step_done() {
  Impl& g = *p_;
  Context& c = ctx();
  const int n = c.n;
  FILE* fstats = g.fstats;
  if (!g.ev[0])
    for (auto& e : g.ev) EVSL_HIP(hipEventCreate(&e));
  auto elapsed = [](hipEvent_t a, hipEvent_t b) {
    float ms = 0.f;
    if (hipEventSynchronize(b) != hipSuccess || hipEventElapsedTime(&ms, a, b) != hipSuccess)
      return 0.0;
    return ms * 1e-3;
  };
  const double eta = 1.0 / std::sqrt(2.0);
  double* sc_d = g.scal_d.as<double>();
  const std::vector<int> act = g.act_cur;
  if (act.empty()) return 0;
  const int b = (int)act.size();
  EVSL_HIP(hipEventRecord(g.ev[1], c.stream));

  // ---- recurrence: vnew -= beta vold; alpha; vnew -= alpha v; ||vnew||^2;
  // first Gram-Schmidt pass -----
  if (int e = g.by_cols(act, [&](evsl_dev::LanCols& cols, int nc, const int*) -> int {
        EVSL_HIP(evsl_dev::lan_recurrence(n, cols, nc, c.stream));
        return 0;
      }))
    return e;
  if (int e = g.cgs_all(act, false)) return e;
  std::vector<double> hs(4 * g.slots.size());
  EVSL_HIP(hipMemcpy(hs.data(), sc_d, hs.size() * sizeof(double), hipMemcpyDeviceToHost));
  std::vector<int> second;
  for (int s : act) {
    Impl::Slot& sl = *g.slots[s];
    Slice& L = sl.L;
    const int k = sl.k;
    const double alpha = hs[4 * s], old_nrm = std::sqrt(hs[4 * s + 1]);
    L.dT[k] = alpha;
    L.wn += std::fabs(alpha);
    L.nrm = std::sqrt(hs[4 * s + 2]);
    c.astats.n_reorth_pass++;
    c.astats.reorth_bytes += Impl::cgs_bytes(L, n, k);
    if (!(L.nrm > eta * old_nrm)) second.push_back(s);
  }
  if (int e = g.cgs_all(second, true)) return e;
  for (int s : second) {
    c.astats.n_reorth_pass++;
    c.astats.reorth_bytes += Impl::cgs_bytes(g.slots[s]->L, n, g.slots[s]->k);
  }
  if (!second.empty()) {
    EVSL_HIP(hipMemcpy(hs.data(), sc_d, hs.size() * sizeof(double), hipMemcpyDeviceToHost));
    for (int s : second) g.slots[s]->L.nrm = std::sqrt(hs[4 * s + 3]);
  }
  std::vector<int> scaled;
  for (int s : act) {
    Impl::Slot& sl = *g.slots[s];
    Slice& L = sl.L;
    const int k = sl.k;
    double* vnew = L.vcol(k + 1, n);
    L.beta = L.nrm;
    L.wn += 2.0 * L.beta;
    L.nwn += 3;
    if (L.beta * L.nwn < kOrthTol * L.wn) {  // lucky breakdown: new filtered random vector
      rand_double_device(n, g.vrand.as<double>());
      ChebWork cw;
      if (int e = cheb_av(L.pol, g.vrand.as<double>(), vnew, cw, sl.f32 ? EVSL_PREC_MIXED : 0))
        return e;
      double d2[2];
      EVSL_HIP(evsl_dev::dot_partial(n, vnew, vnew, red_part(), c.stream));
      EVSL_HIP(evsl_dev::sum_scalar(red_part(), evsl_dev::kRedBlocks, red_scalar(0), c.stream));
      if (int e = read_scalars(red_scalar(0), 1, d2)) return e;
      double old = std::sqrt(d2[0]), nn = old;
      for (int it = 0; it < 2; ++it) {
        int np = 0;
        if (int e = g.cgs_pass(L, k, vnew, red_part(), &np)) return e;
        EVSL_HIP(evsl_dev::sum_scalar(red_part(), np, red_scalar(1), c.stream));
        if (int e = read_scalars(red_scalar(1), 1, d2)) return e;
        nn = std::sqrt(d2[0]);
        if (nn > eta * old) break;
        old = nn;
      }
      if (int e = g.scal_col(L, k + 1, 1.0 / nn)) return e;
      L.beta = 0.0;
    } else {
      scaled.push_back(s);
    }
    L.eT[k] = L.beta;
  }
  if (int e = g.by_cols(scaled, [&](evsl_dev::LanCols& cols, int nc, const int* id) -> int {
        for (int j = 0; j < nc; ++j) {
          Slice& L = g.slots[id[j]]->L;
          cols.c[j].beta = 1.0 / L.beta;
          cols.c[j].x32 = L.has32() ? L.v32col(g.slots[id[j]]->k + 1) : nullptr;
        }
        EVSL_HIP(evsl_dev::lan_scale(n, cols, nc, c.stream));
        return 0;
      }))
    return e;
  EVSL_HIP(hipEventRecord(g.ev[2], c.stream));
  c.astats.t_reorth += elapsed(g.ev[1], g.ev[2]);
  c.astats.n_lanczos += b;
  // ---- convergence tests (restricted trace, every 20 steps from 30) ---------
  const int Ntest = 30, cycle = 20;
  std::vector<int> tst;
  for (int s : act) {
    const int k = g.slots[s]->k;
    if (!((k < Ntest || (k - Ntest) % cycle != 0) && k != g.slots[s]->maxit - 1)) tst.push_back(s);
  }
  // the slices' tridiagonal eigenvalue problems are independent: one host
  // thread each (the device is idle until the next filter pass)
  const int nt = (int)tst.size();
  std::vector<double> tr1s(nt, 0.0);
  std::vector<int> nconvs(nt, 0), qlerr(nt, 0);
#pragma omp parallel for schedule(dynamic, 1) if (nt > 1)
  for (int j = 0; j < nt; ++j) {
    const Impl::Slot& sl = *g.slots[tst[j]];
    const Slice& L = sl.L;
    const int kdim = sl.k + 1;
    std::vector<double> ev(kdim), e(kdim + 1, 0.0);
    std::memcpy(ev.data(), L.dT.data(), kdim * sizeof(double));
    std::memcpy(e.data(), L.eT.data(), (kdim - 1) * sizeof(double));
    if (tridiag_ql(kdim, ev.data(), e.data(), nullptr)) {
      qlerr[j] = 1;
      continue;
    }
    for (int i = 0; i < kdim; ++i)
      if (ev[i] + kEpsM >= L.pol->bar) {
        tr1s[j] += ev[i];
        ++nconvs[j];
      }
  }
  for (int j = 0; j < nt; ++j) {
    const int s = tst[j];
    Impl::Slot& sl = *g.slots[s];
    Slice& L = sl.L;
    const int k = sl.k;
    if (qlerr[j]) return EVSL_ERR_EIG;
    const double tr1 = tr1s[j];
    const int nconv = nconvs[j];
    // FP64: the reference's test.  Mixed: the filtered operator is known to
    // ~1e-6, so the trace is compared at that level and the count of Ritz
    // values above bar must also be unchanged; both keep the reference's stop
    // when no Ritz value has reached bar at this test and the one before
    // (an empty trace, SRC/cheblanNr.c:269-309)
    const double dtr = std::fabs(tr1 - L.tr0);
    const bool empty = std::fabs(tr1) + std::fabs(L.tr0) < 1e-10;
    bool done = sl.f32 ? ((dtr < 1e-7 * std::max(1, nconv) && nconv == L.last_nconv) || empty)
                       : (dtr < 2e-12 || empty);
    if (fstats)
      std::fprintf(fstats, "slice %d k %4d: nconv %4d  tr1 %21.15e dtr %.3e\n", s, k, nconv, tr1,
                   dtr);
    L.tr0 = tr1;
    L.last_nconv = nconv;
    if (done || k == sl.maxit - 1) {
      L.kdim = k + 1;
      L.V32.release();  // the Ritz vectors and the refinement use the FP64 basis
      const double tr = evsl_timer();
      if (fstats) std::fprintf(fstats, "slice %d done at k %d\n", s, k);
      SliceResult* o = sl.out;
      bool stalled = false;
      int err = refine_extract(n, L.kdim, L.dT.data(), L.eT.data(), L.V.as<double>(), L.pol,
                               L.intv, sl.tol, sl.f32, &o->nev, &o->lam, &o->W, &o->res, fstats,
                               &stalled, -1.0);
      if (!err && stalled) {
        // once more with half the guard threshold: the eigenvectors whose
        // components a pass damps least lie just below the guard set, so a
        // wider Rayleigh-Ritz space takes them out
        if (fstats) std::fprintf(fstats, "slice %d: refinement stalled, again at half the guard\n", s);
        ++c.astats.n_refine_retries;
        std::free(o->lam);
        std::free(o->res);
        if (o->W) _evsl_Free_device(o->W);
        *o = SliceResult();
        stalled = false;
        err = refine_extract(n, L.kdim, L.dT.data(), L.eT.data(), L.V.as<double>(), L.pol,
                             L.intv, sl.tol, sl.f32, &o->nev, &o->lam, &o->W, &o->res, fstats,
                             &stalled, 0.5 * c.refine_guard);
      }
      c.astats.t_ritz += evsl_timer() - tr;
      if (!err && stalled) {
        // the FP32-filtered basis cannot reach tol: the slice again in FP64
        if (fstats) std::fprintf(fstats, "slice %d: refinement stalled, rerun in FP64\n", s);
        std::free(o->lam);
        std::free(o->res);
        if (o->W) _evsl_Free_device(o->W);
        *o = SliceResult();
        ++c.astats.n_fp64_reruns;
        if (int e = g.start(s, false)) return e;
        continue;
      }
      L.V.release();
      o->err = err;
      o->steps = L.kdim;
      o->done = true;
      o->t_done = evsl_timer();
      sl.state = 0;
      if (err) return err;
    }
  }
  for (int s : act)
    if (g.slots[s]->state == 2) ++g.slots[s]->k;
  return 0;
}

}  // namespace evsl

using namespace evsl;

extern "C" {

int ChebLanNr_batch(int nslices, double* intvs, int maxit, double tol, double* vinit,
                    polparams* pols, int* nevOut, double** lamo, double** Wo, double** reso,
                    FILE* fstats) {
  if (int e = ensure_started()) return e;
  Context& c = ctx();
  if (c.op == 0) return EVSL_ERR_NOMAT;
  if (nslices <= 0) return EVSL_ERR_ARG;
  const size_t nl = c.n;
  const bool mixed = (c.filter_prec == EVSL_PREC_MIXED) && c.op == 1;
  const double cc0 = pols[0].cc, dd0 = pols[0].dd;
  for (int s = 0; s < nslices; ++s) {
    nevOut[s] = 0;
    lamo[s] = reso[s] = Wo[s] = nullptr;
    if (pols[s].cc != cc0 || pols[s].dd != dd0) {
      set_error_msg("ChebLanNr_batch: slices must share [lmin, lmax]");
      return EVSL_ERR_ARG;
    }
    if (pols[s].gam > 1.0 || pols[s].gam < -1.0) return -1;
  }
  DevBuf vtmp;
  const double* v0;
  if (int e = as_device_vector(vinit, nl, vtmp, &v0)) return e;
  LanczosGroup grp(mixed, fstats);
  std::vector<SliceResult> out(nslices);
  for (int s = 0; s < nslices; ++s)
    if (int e = grp.add(intvs + 4 * s, maxit, tol, v0, &pols[s], &out[s])) return e;
  int err = 0;
  while (grp.active() > 0)
    if ((err = grp.step())) break;
  for (int s = 0; s < nslices; ++s) {
    nevOut[s] = out[s].nev;
    lamo[s] = out[s].lam;
    Wo[s] = out[s].W;
    reso[s] = out[s].res;
    if (!err && out[s].err) err = out[s].err;
  }
  return err;
}


// Polynomial-filtered subspace iteration (SRC/chebsi.c:39-336): a block of
// nev vectors is filtered with p(A) (one blocked SpMM per degree for up to 32
// columns), deflated against the locked columns, re-orthonormalised, and
// every cvcheck = 5 iterations Rayleigh-Ritz on p(A) rotates the block;
// columns whose p(A)-residual is below tol/100 and whose A-residual is below
// tol are locked.  The filter runs in FP64.  vinit holds nev vectors (n x nev,
// column-major, host or device).
int ChebSI(int nev, double* intv, int maxit, double tol, double* vinit, polparams* pol,
           int* nevo, double** lamo, double** Yo, double** reso, FILE* fstats) {
  if (int e = ensure_started()) return e;
  Context& c = ctx();
  if (c.op == 0) return EVSL_ERR_NOMAT;
  const double t_all = evsl_timer();
  const double tolP = tol * 0.01;
  const int n = c.n;
  const size_t nl = n;
  *nevo = 0;
  *lamo = *Yo = *reso = nullptr;
  if (check_intv(intv) < 0) return 0;
  const double aa = intv[0], bb = intv[1];
  const int cvcheck = 5, kNbuf = 2;
  const int deg = pol->deg;
  const double gamB = pol->gam, bar = pol->bar;
  if (fstats)
    std::fprintf(fstats, "Cheb Poly- deg = %d, gam = %.15e, bar: %.15e\n", deg, gamB, bar);
  if (gamB > 1.0 || gamB < -1.0) {
    std::fprintf(stdout, "gamB error %.15e\n", gamB);
    return -1;
  }
  if (nev <= 0 || nev > n) {
    set_error_msg("ChebSI: block size must be in [1, n]");
    return EVSL_ERR_ARG;
  }
  if (fstats) std::fprintf(fstats, "Step 2: ChebSI, block size = %d\n", nev);
  DevBuf Vb, PVb, Rb, Bb, Tb, Eb, gp, part, s2d, tvd, r2d, wcol, vtmp;
  const size_t blk = nl * nev * sizeof(double);
  EVSL_HIP(Vb.alloc(blk));
  EVSL_HIP(PVb.alloc(blk));
  EVSL_HIP(Rb.alloc(blk));
  EVSL_HIP(Bb.alloc(blk));
  EVSL_HIP(Tb.alloc((size_t)nev * nev * sizeof(double)));
  EVSL_HIP(Eb.alloc((size_t)nev * nev * sizeof(double)));
  EVSL_HIP(gp.alloc(evsl_dev::gemm_tn_part_elems(n, nev, nev) * sizeof(double)));
  const int nch8 = (n + 8191) / 8192;
  EVSL_HIP(part.alloc((size_t)nch8 * nev * sizeof(double)));
  EVSL_HIP(s2d.alloc(nev * sizeof(double)));
  EVSL_HIP(tvd.alloc(nev * sizeof(double)));
  EVSL_HIP(r2d.alloc(nev * sizeof(double)));
  EVSL_HIP(wcol.alloc(nl * sizeof(double)));
  double* V = Vb.as<double>();
  double* PV = PVb.as<double>();
  double* R = Rb.as<double>();
  double* buf = Bb.as<double>();
  auto col = [&](double* M, int j) { return M + (size_t)j * nl; };
  LanWork L;
  L.nch = evsl_dev::gemv_t_chunks(n);
  EVSL_HIP(L.gt_part.alloc((size_t)L.nch * (nev + 1) * sizeof(double)));
  EVSL_HIP(L.h.alloc((size_t)(nev + 1) * sizeof(double)));
  BlockWork bw;
  std::vector<double> T((size_t)nev * nev), evecT((size_t)nev * nev), evalT(nev), Lam(nev),
      res(nev);
  std::vector<int> act_idx(nev), lock_idx(nev);
  const double* v0;
  if (int e = as_device_vector(vinit, nl * nev, vtmp, &v0)) return e;
  // orth (SRC/misc_la.c:317-342): column-by-column CGS/DGKS into Vo
  auto orth = [&](const double* Vin, int k, double* Vo) -> int {
    EVSL_HIP(hipMemcpyAsync(Vo, Vin, nl * k * sizeof(double), hipMemcpyDeviceToDevice,
                            c.stream));
    double nrm;
    if (int e = nrm2_dev(n, Vo, &nrm)) return e;
    EVSL_HIP(evsl_dev::scal(n, 1.0 / nrm, Vo, c.stream));
    for (int i = 1; i < k; ++i) {
      double* vi = Vo + (size_t)i * nl;
      double old;
      if (int e = nrm2_dev(n, vi, &old)) return e;
      if (int e = cgs_dgks(n, i, Vo, vi, old * old, &nrm, L)) return e;
      EVSL_HIP(evsl_dev::scal(n, 1.0 / nrm, vi, c.stream));
    }
    return 0;
  };
  // PV(:, j0:j0+k) = p(A) V(:, j0:j0+k)
  auto filter = [&](int j0, int k) -> int {
    std::vector<const double*> in(k);
    std::vector<double*> out(k);
    std::vector<const polparams*> pp(k, pol);
    for (int j = 0; j < k; ++j) {
      in[j] = col(V, j0 + j);
      out[j] = col(PV, j0 + j);
    }
    return filter_columns(k, in.data(), out.data(), pp.data(), false, bw);
  };
  // X(:, nlock:nlock+nact) -= V(:, 0:nlock) V(:, 0:nlock)^T X(:, nlock:nlock+nact)
  auto deflate = [&](double* X, int nlock, int nact) -> int {
    EVSL_HIP(evsl_dev::gemm_tn(n, nlock, nact, V, n, col(X, nlock), n, Tb.as<double>(), nlock,
                               gp.as<double>(), c.stream));
    std::vector<double> Th((size_t)nlock * nact);
    EVSL_HIP(hipMemcpy(Th.data(), Tb.p, Th.size() * sizeof(double), hipMemcpyDeviceToHost));
    for (double& t : Th) t = -t;
    EVSL_HIP(hipMemcpy(Tb.p, Th.data(), Th.size() * sizeof(double), hipMemcpyHostToDevice));
    EVSL_HIP(evsl_dev::gemm_nn(n, nact, nlock, V, n, Tb.as<double>(), nlock, col(buf, nlock), n,
                               c.stream));
    std::vector<double> ones(nact, 1.0);
    EVSL_HIP(hipMemcpy(s2d.p, ones.data(), nact * sizeof(double), hipMemcpyHostToDevice));
    EVSL_HIP(evsl_dev::col_scale_add(n, nact, col(X, nlock), n, s2d.as<double>(),
                                     col(buf, nlock), n, c.stream));
    return 0;
  };
  if (int e = orth(v0, nev, V)) return e;
  if (int e = filter(0, nev)) return e;
  long nmv = (long)deg * nev;
  int it = 0, nlock = 0, nact = nev, nlock_ab = 0;
  bool find_more = true;
  while (it < maxit && find_more) {
    const size_t nnact = nl * nact;
    EVSL_HIP(hipMemcpyAsync(col(V, nlock), col(PV, nlock), nnact * sizeof(double),
                            hipMemcpyDeviceToDevice, c.stream));
    if (nlock > 0)
      if (int e = deflate(V, nlock, nact)) return e;
    if (int e = orth(col(V, nlock), nact, col(buf, nlock))) return e;
    EVSL_HIP(hipMemcpyAsync(col(V, nlock), col(buf, nlock), nnact * sizeof(double),
                            hipMemcpyDeviceToDevice, c.stream));
    if (int e = filter(nlock, nact)) return e;
    nmv += (long)deg * nact;
    if (nlock > 0)
      if (int e = deflate(PV, nlock, nact)) return e;
    if ((it + 1) % cvcheck == 0 || it + 1 == maxit) {
      // Rayleigh-Ritz on p(A): T = V_act^T PV_act, eigenpairs, rotate both blocks
      EVSL_HIP(evsl_dev::gemm_tn(n, nact, nact, col(V, nlock), n, col(PV, nlock), n,
                                 Tb.as<double>(), nact, gp.as<double>(), c.stream));
      EVSL_HIP(hipMemcpy(T.data(), Tb.p, (size_t)nact * nact * sizeof(double),
                         hipMemcpyDeviceToHost));
      for (int j = 0; j < nact; ++j)
        for (int i = 0; i < j; ++i) {
          const double a = 0.5 * (T[(size_t)j * nact + i] + T[(size_t)i * nact + j]);
          T[(size_t)j * nact + i] = T[(size_t)i * nact + j] = a;
        }
      if (int e = sym_eig_host(nact, T.data(), nact, evecT.data(), nact, &evalT[nlock]))
        return e;
      EVSL_HIP(hipMemcpy(Eb.p, evecT.data(), (size_t)nact * nact * sizeof(double),
                         hipMemcpyHostToDevice));
      EVSL_HIP(evsl_dev::gemm_nn(n, nact, nact, col(V, nlock), n, Eb.as<double>(), nact,
                                 col(buf, nlock), n, c.stream));
      EVSL_HIP(hipMemcpyAsync(col(V, nlock), col(buf, nlock), nnact * sizeof(double),
                              hipMemcpyDeviceToDevice, c.stream));
      EVSL_HIP(evsl_dev::gemm_nn(n, nact, nact, col(PV, nlock), n, Eb.as<double>(), nact,
                                 col(buf, nlock), n, c.stream));
      EVSL_HIP(hipMemcpyAsync(col(PV, nlock), col(buf, nlock), nnact * sizeof(double),
                              hipMemcpyDeviceToDevice, c.stream));
      // residual norms with respect to p(A): ||PV_i - evalT_i V_i||
      EVSL_HIP(hipMemcpy(tvd.p, &evalT[nlock], nact * sizeof(double), hipMemcpyHostToDevice));
      EVSL_HIP(evsl_dev::col_res2(n, nact, col(PV, nlock), n, col(V, nlock), n,
                                  tvd.as<double>(), part.as<double>(), r2d.as<double>(),
                                  c.stream));
      std::vector<double> rP2(nact);
      EVSL_HIP(hipMemcpy(rP2.data(), r2d.p, nact * sizeof(double), hipMemcpyDeviceToHost));
      int nlock_new = 0, nlock_ab_new = 0;
      const int nact_old = nact;
      nact = 0;
      for (int i = nlock; i < nev; ++i) {
        const double resP = std::sqrt(std::max(rP2[i - nlock], 0.0));
        bool locked = false;
        if (resP < tolP) {
          double* vi = col(V, i);
          if (int e = apply_A(vi, wcol.as<double>())) return e;
          ++nmv;
          EVSL_HIP(evsl_dev::col_dot(n, 1, vi, n, wcol.as<double>(), n, part.as<double>(),
                                     tvd.as<double>(), c.stream));
          EVSL_HIP(evsl_dev::col_res2(n, 1, wcol.as<double>(), n, vi, n, tvd.as<double>(),
                                      part.as<double>(), r2d.as<double>(), c.stream));
          double rq, rA2;
          EVSL_HIP(hipMemcpy(&rq, tvd.p, sizeof(double), hipMemcpyDeviceToHost));
          EVSL_HIP(hipMemcpy(&rA2, r2d.p, sizeof(double), hipMemcpyDeviceToHost));
          const double resA = std::sqrt(std::max(rA2, 0.0));
          if (resA < tol) {
            lock_idx[nlock_new] = i;
            res[nlock + nlock_new] = resA;
            Lam[nlock + nlock_new] = rq;
            ++nlock_new;
            if (rq >= aa - kEpsM && rq <= bb + kEpsM) ++nlock_ab_new;
            locked = true;
          }
        }
        if (!locked) act_idx[nact++] = i;
      }
      // newly locked columns first, then the active ones (via buf and R)
      for (int i = 0; i < nlock_new; ++i) {
        EVSL_HIP(hipMemcpyAsync(col(buf, nlock + i), col(V, lock_idx[i]), nl * sizeof(double),
                                hipMemcpyDeviceToDevice, c.stream));
        EVSL_HIP(hipMemcpyAsync(col(R, nlock + i), col(PV, lock_idx[i]), nl * sizeof(double),
                                hipMemcpyDeviceToDevice, c.stream));
      }
      for (int i = 0; i < nact; ++i) {
        EVSL_HIP(hipMemcpyAsync(col(buf, nlock + nlock_new + i), col(V, act_idx[i]),
                                nl * sizeof(double), hipMemcpyDeviceToDevice, c.stream));
        EVSL_HIP(hipMemcpyAsync(col(R, nlock + nlock_new + i), col(PV, act_idx[i]),
                                nl * sizeof(double), hipMemcpyDeviceToDevice, c.stream));
      }
      EVSL_HIP(hipMemcpyAsync(col(V, nlock), col(buf, nlock), nl * nact_old * sizeof(double),
                              hipMemcpyDeviceToDevice, c.stream));
      EVSL_HIP(hipMemcpyAsync(col(PV, nlock), col(R, nlock), nl * nact_old * sizeof(double),
                              hipMemcpyDeviceToDevice, c.stream));
      nlock += nlock_new;
      nlock_ab += nlock_ab_new;
      if (fstats)
        std::fprintf(fstats, "it %4d:   nMV %7ld,  nlock %3d, nlock_ab  %3d\n", it + 1, nmv,
                     nlock, nlock_ab);
      // stop when NBUF locked pairs lie outside [a, b] or the whole block is locked
      if (nlock - nlock_ab >= kNbuf || nlock == nev) {
        find_more = false;
        if (fstats)
          std::fprintf(fstats, "-------------------------------------\n No ev.s left to be "
                               "computed\n Number of evals found = %d\n", nlock_ab);
      }
    }
    ++it;
  }
  // keep the locked pairs inside [a, b], in locking order
  double* lam_o = (double*)std::malloc((size_t)nev * sizeof(double));
  double* res_o = (double*)std::malloc((size_t)nev * sizeof(double));
  double* Y_o = (double*)_evsl_Malloc_device(blk);
  if (!lam_o || !res_o || !Y_o) {
    std::free(lam_o);
    std::free(res_o);
    if (Y_o) _evsl_Free_device(Y_o);
    return EVSL_ERR_ALLOC;
  }
  int idx = 0;
  for (int i = 0; i < nlock; ++i) {
    const double t = Lam[i];
    if (t >= aa - kEpsM && t <= bb + kEpsM) {
      lam_o[idx] = t;
      res_o[idx] = res[i];
      EVSL_HIP(hipMemcpyAsync(Y_o + (size_t)idx * nl, col(V, i), nl * sizeof(double),
                              hipMemcpyDeviceToDevice, c.stream));
      ++idx;
    }
  }
  EVSL_HIP(hipStreamSynchronize(c.stream));
  *nevo = idx;
  *lamo = lam_o;
  *Yo = Y_o;
  *reso = res_o;
  const double tall = evsl_timer() - t_all;
  if (fstats)
    std::fprintf(fstats, "------This slice consumed: \nMatvecs :        %ld\ntotal  time :    %.2f\n",
                 nmv, tall);
  evslstat.t_iter = tall;
  return 0;
}


// Y(:, j) = p_j(A) X(:, j) for the ncols columns of the n x ncols
// column-major X (host or device; Y host or device likewise), with the
// blocked filter: at most 32 columns per series, columns of different degrees
// narrowed as their degrees are reached.  The block form of the reference's
// ChebAv (SRC/chebpoly.c:519-598), one p_j per column; every pols[j] must
// come from find_pol on the same outer bounds (same cc, dd).
int evsl_amd_cheb_av_cols(int ncols, const polparams* pols, const double* X, double* Y,
                          int prec) {
  if (int e = ensure_started()) return e;
  Context& c = ctx();
  if (c.op == 0) return EVSL_ERR_NOMAT;
  if (ncols <= 0 || !pols || !X || !Y || (prec != EVSL_PREC_FP64 && prec != EVSL_PREC_MIXED)) {
    set_error_msg("evsl_amd_cheb_av_cols: invalid arguments");
    return EVSL_ERR_ARG;
  }
  for (int j = 0; j < ncols; ++j)
    if (!pols[j].mu || pols[j].deg < 0 || pols[j].cc != pols[0].cc ||
        pols[j].dd != pols[0].dd) {
      set_error_msg("evsl_amd_cheb_av_cols: every filter needs coefficients and the same cc, dd");
      return EVSL_ERR_ARG;
    }
  const size_t nl = c.n, tot = nl * ncols;
  DevBuf xt, yt;
  const double* xd;
  if (int e = as_device_vector(X, tot, xt, &xd)) return e;
  double* yd = Y;
  hipPointerAttribute_t at;
  const bool ydev = hipPointerGetAttributes(&at, Y) == hipSuccess &&
                    (at.type == hipMemoryTypeDevice || at.type == hipMemoryTypeManaged);
  if (!ydev) {
    (void)hipGetLastError();  // clear the error of an unregistered host pointer
    EVSL_HIP(yt.alloc(tot * sizeof(double)));
    yd = yt.as<double>();
  }
  // X and Y may share memory.  A block's columns are packed before any of them is
  // written, which in place is all it takes; a series launch that fails has
  // written some outputs before its columns are filtered again, and in a shifted
  // range an output is a later block's input: X is copied for those.
  if (yd < xd + tot && xd < yd + tot && (xd != yd || series_size(c.n, ncols))) {
    EVSL_HIP(xt.alloc(tot * sizeof(double)));
    EVSL_HIP(hipMemcpyAsync(xt.p, xd, tot * sizeof(double), hipMemcpyDeviceToDevice, c.stream));
    xd = xt.as<double>();
  }
  std::vector<const double*> in(ncols);
  std::vector<double*> out(ncols);
  std::vector<const polparams*> pp(ncols);
  for (int j = 0; j < ncols; ++j) {
    in[j] = xd + (size_t)j * nl;
    out[j] = yd + (size_t)j * nl;
    pp[j] = pols + j;
  }
  BlockWork bw;
  if (int e = filter_columns(ncols, in.data(), out.data(), pp.data(),
                             prec == EVSL_PREC_MIXED, bw))
    return e;
  if (!ydev)
    EVSL_HIP(hipMemcpyAsync(Y, yd, tot * sizeof(double), hipMemcpyDeviceToHost, c.stream));
  EVSL_HIP(hipStreamSynchronize(c.stream));
  return 0;
}

// evsl_amd_cheb_av_cols with every work buffer in the library's static
// device scratch (evsl_dev::kNoAllocScratchBytes per GPU): no device memory
// is allocated or freed, for callers that cannot allocate.  X and Y must be
// device memory; the columns run in blocks of at most 32 whose interleaved
// input, recurrence ring (three blocks), FP64 output block and coefficient
// table fit the scratch.  The fused kernel runs the fixed layout policy (no
// layout tuning, whose timing events are resources), which gives the same
// bits as any tuned layout, so the result equals evsl_amd_cheb_av_cols's
// bit for bit.  Calls that overlap on one GPU share its scratch and race.
int evsl_amd_cheb_av_cols_noalloc(int ncols, const polparams* pols, const double* X, double* Y,
                                  int prec) {
  clear_error();
  Context& c = ctx();
  if (!c.started || c.op != 1) {
    set_error_msg("evsl_amd_cheb_av_cols_noalloc: no device matrix (EVSLStart, SetAMatrix)");
    return EVSL_ERR_NOMAT;
  }
  if (ncols <= 0 || !pols || !X || !Y || (prec != EVSL_PREC_FP64 && prec != EVSL_PREC_MIXED)) {
    set_error_msg("evsl_amd_cheb_av_cols_noalloc: invalid arguments");
    return EVSL_ERR_ARG;
  }
  for (int j = 0; j < ncols; ++j)
    if (!pols[j].mu || pols[j].deg < 0 || pols[j].cc != pols[0].cc ||
        pols[j].dd != pols[0].dd) {
      set_error_msg("evsl_amd_cheb_av_cols_noalloc: every filter needs coefficients and the "
                    "same cc, dd");
      return EVSL_ERR_ARG;
    }
  for (const void* p : {(const void*)X, (const void*)Y}) {
    hipPointerAttribute_t at;
    if (hipPointerGetAttributes(&at, p) != hipSuccess ||
        !(at.type == hipMemoryTypeDevice || at.type == hipMemoryTypeManaged)) {
      (void)hipGetLastError();
      set_error_msg("evsl_amd_cheb_av_cols_noalloc: X and Y must be device memory");
      return EVSL_ERR_ARG;
    }
  }
  const bool f32 = prec == EVSL_PREC_MIXED;
  if (!filter_op_ready(f32)) {
    set_error_msg("evsl_amd_cheb_av_cols_noalloc: the matrix's FP32 copy does not exist yet "
                  "(one mixed-precision call on this matrix creates it)");
    return EVSL_ERR_ARG;
  }
  void* base = nullptr;
  if (hipError_t he = evsl_dev::noalloc_scratch(&base); he != hipSuccess) {
    set_error("evsl_amd_cheb_av_cols_noalloc: scratch address", he);
    return EVSL_ERR_DEVICE;
  }
  const size_t n = c.n, vs = f32 ? 4 : 8, cap = evsl_dev::kNoAllocScratchBytes;
  auto up = [](size_t b) { return (b + 255) & ~(size_t)255; };
  // scratch bytes of a block of B columns filtered to degree md
  auto need = [&](int B, int md) {
    return up((size_t)(md + 1) * B * sizeof(double)) + 4 * up(n * B * vs) +
           up(n * B * sizeof(double));
  };
  FilterOp op;
  bool have_op = false;
  for (int j0 = 0; j0 < ncols;) {
    int B = 0, md = 0;
    for (int w : {32, 16, 8, 7, 6, 5, 4, 3, 2, 1}) {
      if (w > ncols - j0) continue;
      int d = 0;
      for (int j = j0; j < j0 + w; ++j) d = std::max(d, pols[j].deg);
      if (need(w, d) <= cap) {
        B = w;
        md = d;
        break;
      }
    }
    if (B == 0) {
      set_error_msg("evsl_amd_cheb_av_cols_noalloc: one column needs more than the scratch's " +
                    std::to_string(cap >> 20) + " MiB (n x (4 x vector size + 8) bytes plus " +
                    "(deg + 1) x 8)");
      return EVSL_ERR_ARG;
    }
    const double* in[evsl_dev::kMaxCols];
    double* out[evsl_dev::kMaxCols];
    for (int j = 0; j < B; ++j) {
      in[j] = X + (size_t)(j0 + j) * n;
      out[j] = Y + (size_t)(j0 + j) * n;
    }
    if (md == 0) {  // degree-0 filters: y = mu0 x
      for (int j = 0; j < B; ++j)
        EVSL_HIP(evsl_dev::scal_copy(n, pols[j0 + j].mu[0], in[j], out[j], c.stream));
      j0 += B;
      continue;
    }
    if (!have_op) {
      if (int e = make_filter_op(pols[0].cc, pols[0].dd, f32, &op)) return e;
      op.A.tune = nullptr;  // fixed layout policy
      have_op = true;
    }
    char* p = static_cast<char*>(base);
    double* tab = reinterpret_cast<double*>(p);
    p += up((size_t)(md + 1) * B * sizeof(double));
    void* X0 = p;
    p += up(n * B * vs);
    void* bufs[3];
    for (int i = 0; i < 3; ++i) {
      bufs[i] = p;
      p += up(n * B * vs);
    }
    void* Yb = p;
    // coefficient table: row d holds mu_d of each column, zero beyond a
    // column's degree (the column's sum is then the one of its own degree)
    EVSL_HIP(evsl_dev::fill((size_t)(md + 1) * B, 0.0, tab, c.stream));
    for (int j = 0; j < B; ++j)
      EVSL_HIP(hipMemcpy2DAsync(tab + j, B * sizeof(double), pols[j0 + j].mu, sizeof(double),
                                sizeof(double), pols[j0 + j].deg + 1, hipMemcpyHostToDevice,
                                c.stream));
    EVSL_HIP(evsl_dev::pack_cols(n, B, col_ptrs(in, B), X0, f32, c.stream));
    if (int e = block_filter(B, op, tab, md, X0, bufs, Yb)) return e;
    EVSL_HIP(evsl_dev::unpack_cols(n, B, Yb, false, col_ptrs(out, B), c.stream));
    // the next block reuses the scratch: the stream orders its launches
    // after these; the host's coefficient arrays are read by then
    EVSL_HIP(hipStreamSynchronize(c.stream));
    j0 += B;
  }
  EVSL_HIP(hipStreamSynchronize(c.stream));
  return 0;
}

}  // extern "C"
