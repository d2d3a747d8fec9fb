// lanczos.cpp -- filtered Lanczos on the device: ChebAv, CGS/DGKS,
// ChebLanNr, LanBounds and LanDos of the drop-in interface.
//
// Follows SRC/chebpoly.c:519-598 (ChebAv), SRC/misc_la.c:221-261 (CGS_DGKS),
// SRC/cheblanNr.c:57-434, SRC/lanbounds.c:21-144 and SRC/landos.c:37-196 of
// EVSL 1.1.1.  The Lanczos basis V stays in HBM (column-major, n x (maxit+1));
// all vector work runs in HIP kernels; the host keeps the scalar recurrence
// (alpha, beta), the tridiagonal eigenvalues and the control flow.  One
// device->host read per Lanczos step carries alpha and the DGKS norms.
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <future>
#include <system_error>
#include <vector>

#include "internal.h"

namespace evsl {

namespace {

constexpr double kOrthTol = 1e-14;  // INC/internal_header.h:21
const double kEpsM = EVSL_DBL_EPS_MULT * DBL_EPSILON;


}  // namespace

int check_intv(const double* intv) {
  if (intv[0] >= intv[1]) return -1;
  if (intv[0] >= intv[3] || intv[1] <= intv[2]) return -2;
  return 0;
}

int as_device_vector(const double* p, size_t n, DevBuf& tmp, const double** out) {
  hipPointerAttribute_t at;
  hipError_t e = hipPointerGetAttributes(&at, p);
  if (e == hipSuccess && (at.type == hipMemoryTypeDevice || at.type == hipMemoryTypeManaged)) {
    *out = p;
    return 0;
  }
  (void)hipGetLastError();  // clear the error of an unregistered host pointer
  EVSL_HIP(tmp.alloc(n * sizeof(double)));
  EVSL_HIP(hipMemcpy(tmp.p, p, n * sizeof(double), hipMemcpyHostToDevice));
  *out = tmp.as<double>();
  return 0;
}

namespace {

// HIP-event phase timing accumulated into the extension statistics
struct EventClock {
  hipEvent_t ev[4] = {nullptr, nullptr, nullptr, nullptr};
  bool ok = false;
  EventClock() {
    ok = true;
    for (auto& e : ev)
      if (hipEventCreate(&e) != hipSuccess) ok = false;
  }
  ~EventClock() {
    for (auto& e : ev)
      if (e) (void)hipEventDestroy(e);
  }
  void mark(int i) {
    if (ok) (void)hipEventRecord(ev[i], ctx().stream);
  }
  double secs(int a, int b) {
    float ms = 0.f;
    if (!ok || hipEventSynchronize(ev[b]) != hipSuccess ||
        hipEventElapsedTime(&ms, ev[a], ev[b]) != hipSuccess)
      return 0.0;
    return ms * 1e-3;
  }
};

// matrix bytes of one launch (values of sa bytes) plus vec_bytes per row
// and column of the B-column block
double filter_step_bytes(const Context& c, int B, int sa, double vec_bytes) {
  return c.A.mat_bytes((int)sa, B) + vec_bytes * B * c.n;
}

}  // namespace

// ---------------------------------------------------------------------
// y = p((A - cc)/dd) v  -- one fused SpMM launch per degree
// ---------------------------------------------------------------------
int cheb_av(const polparams* pol, const double* v, double* y, ChebWork& w, int prec,
            bool deferred) {
  Context& c = ctx();
  const int n = c.n, m = pol->deg;
  const double cc = pol->cc, t1 = 1.0 / pol->dd, t2 = 2.0 / pol->dd;
  (void)t1;
  (void)t2;
  if (w.deg_loaded != m || w.mu_src != pol->mu) {
    EVSL_HIP(w.mu_d.alloc((size_t)(m + 1) * sizeof(double)));
    EVSL_HIP(hipMemcpy(w.mu_d.p, pol->mu, (size_t)(m + 1) * sizeof(double),
                       hipMemcpyHostToDevice));
    w.deg_loaded = m;
    w.mu_src = pol->mu;
  }
  const double* mu_d = w.mu_d.as<double>();
  if (m == 0) {
    EVSL_HIP(evsl_dev::scal_copy(n, pol->mu[0], v, y, c.stream));
    return 0;
  }
  if (c.op == 2 && prec != EVSL_PREC_FP64) prec = EVSL_PREC_FP64;  // user operator: FP64 only
  if (c.op == 1) {
    const bool f32 = (prec == EVSL_PREC_MIXED);
    const size_t vs = f32 ? sizeof(float) : sizeof(double);
    FilterOp op;
    if (int e = make_filter_op(cc, pol->dd, f32, &op)) return e;
    if (series_fits(op, 1, m)) {
      if (int e = series_launch({{&op, v, y, mu_d, 1, m}})) return e;
      if (deferred) return 0;
      EVSL_HIP(hipStreamSynchronize(c.stream));
      if (!series_failed()) return 0;
    }
    // the kernel accumulates y in FP64 in both precisions, straight into
    // the caller's vector
    DevBuf& store = f32 ? w.b32 : w.bufs;
    const int nvec = f32 ? 4 : 3;
    EVSL_HIP(store.alloc((size_t)nvec * n * vs));
    char* base = store.as<char>();
    void* buf[3] = {base, base + (size_t)n * vs, base + 2 * (size_t)n * vs};
    const void* vin = v;
    void* yout = y;
    if (f32) {
      void* v32 = base + 3 * (size_t)n * vs;
      EVSL_HIP(evsl_dev::f64_to_f32(n, v, (float*)v32, c.stream));
      vin = v32;
    }
    for (int k = 1; k <= m; ++k) {
      void* xkp1 = buf[(k - 1) % 3];
      const void* xk = (k == 1) ? vin : buf[(k - 2) % 3];
      const void* xkm1 = (k == 1) ? nullptr : (k == 2 ? vin : buf[(k - 3) % 3]);
      const int yf = evsl_dev::y_flush(k, m);
      EVSL_HIP(evsl_dev::cheb_spmm(op.A, 1, f32, evsl_dev::kCheb, xk, xkm1, xkp1, yout, nullptr,
                                   mu_d + k, mu_d, k == 1 ? op.t1 : op.t2, op.cc, k == 1, yf,
                                   nullptr, c.stream));
      c.astats.filter_bytes +=
          filter_step_bytes(c, 1, (int)vs, evsl_dev::cheb_vec_bytes(yf, k == 1, (int)vs));
    }
    c.astats.n_filter_steps += m;
    c.astats.n_filter_cols += m;
    return 0;
  }
  // user operator: y = mu0 v; per degree vkp1 = A vk then a fused update
  EVSL_HIP(w.bufs.alloc((size_t)4 * n * sizeof(double)));
  double* b = w.bufs.as<double>();
  double* buf[3] = {b, b + n, b + 2 * (size_t)n};
  double* tmp = b + 3 * (size_t)n;
  EVSL_HIP(evsl_dev::scal_copy(n, pol->mu[0], v, y, c.stream));
  for (int k = 1; k <= m; ++k) {
    double* xkp1 = buf[(k - 1) % 3];
    const double* xk = (k == 1) ? v : buf[(k - 2) % 3];
    const double* xkm1 = (k == 1) ? nullptr : (k == 2 ? v : buf[(k - 3) % 3]);
    if (int e = apply_A(xk, tmp)) return e;
    // xkp1 = t*(tmp - cc*xk) - xkm1 ; y += mu_k xkp1
    const double t = (k == 1 ? t1 : t2);
    EVSL_HIP(evsl_dev::scal_copy(n, t, tmp, xkp1, c.stream));
    EVSL_HIP(evsl_dev::axpy_dot(n, -t * cc, xk, xkp1, nullptr, nullptr, c.stream));
    if (xkm1) EVSL_HIP(evsl_dev::axpy_dot(n, -1.0, xkm1, xkp1, nullptr, nullptr, c.stream));
    EVSL_HIP(evsl_dev::axpy_dot(n, pol->mu[k], xkp1, y, nullptr, nullptr, c.stream));
  }
  c.astats.n_filter_steps += m;
  c.astats.n_filter_cols += m;
  return 0;
}

namespace {

// one Gram-Schmidt pass of q.vnew against the q.k columns of q.V
int cgs_pass(int n, evsl_dev::LanCols& cols) {
  Context& c = ctx();
  evsl_dev::LanCol& q = cols.c[0];
  c.astats.n_reorth_pass++;
  c.astats.reorth_bytes += 16.0 * n * q.k + 24.0 * n;
  if (evsl_dev::lan_small(n)) {
    EVSL_HIP(evsl_dev::lan_gram_schmidt(n, cols, 1, false, c.stream));
    return 0;
  }
  double* h = const_cast<double*>(q.hvec);
  EVSL_HIP(evsl_dev::gemv_t(n, q.k, q.V, n, q.vnew, q.gt, h, c.stream));
  EVSL_HIP(evsl_dev::gemv_n_sub_nrm(n, q.k, q.V, n, h, q.vnew,
                                    q.part + 2 * evsl_dev::kRedBlocks, c.stream));
  q.np = (n + evsl_dev::kWG - 1) / evsl_dev::kWG;
  return 0;
}

evsl_dev::LanCols lan_col(int k, const double* V, double* vnew, LanWork& L) {
  evsl_dev::LanCols cols{};
  evsl_dev::LanCol& q = cols.c[0];
  q.V = V;
  q.k = k;
  q.vnew = vnew;
  q.hvec = L.h.as<double>();
  q.part = red_part();
  q.gt = L.gt_part.as<double>();
  q.out = red_scalar(0);
  return cols;
}

const double kDgksEta = 1.0 / std::sqrt(2.0);

// the second pass of the DGKS test where the first one, from norm old to *nrm,
// asks for it
int cgs_second(int n, evsl_dev::LanCols& cols, double old, double* nrm) {
  if (*nrm > kDgksEta * old) return 0;
  if (int e = cgs_pass(n, cols)) return e;
  EVSL_HIP(evsl_dev::lan_sums(n, cols, 1, true, ctx().stream));
  double s2;
  if (int e = read_scalars(red_scalar(3), 1, &s2)) return e;
  *nrm = std::sqrt(s2);
  return 0;
}

// vnew -= beta zold, alpha = vnew.v, vnew -= alpha v, then the first
// Gram-Schmidt pass against the k columns of V (SRC/misc_la.c:221-261): *alpha
// and the norms before and after the pass come back in one read
int lan_step(int n, int k, const double* V, double beta, const double* zold, const double* v,
             double* vnew, LanWork& L, double* alpha, double* old, double* nrm) {
  evsl_dev::LanCols cols = lan_col(k, V, vnew, L);
  cols.c[0].zold = zold;
  cols.c[0].v = v;
  cols.c[0].beta = beta;
  EVSL_HIP(evsl_dev::lan_recurrence(n, cols, 1, ctx().stream));
  if (int e = cgs_pass(n, cols)) return e;
  EVSL_HIP(evsl_dev::lan_sums(n, cols, 1, false, ctx().stream));
  double sc[3];
  if (int e = read_scalars(red_scalar(0), 3, sc)) return e;
  *alpha = sc[0];
  *old = std::sqrt(sc[1]);
  *nrm = std::sqrt(sc[2]);
  return 0;
}

}  // namespace

// CGS with the DGKS test, two GEMV passes at most (SRC/misc_la.c:221-261).
// On entry old2 = ||v||^2 (already known); returns ||v|| in *nrm.
int cgs_dgks(int n, int k, const double* Q, double* v, double old2, double* nrm, LanWork& L) {
  evsl_dev::LanCols cols = lan_col(k, Q, v, L);
  if (int e = cgs_pass(n, cols)) return e;
  EVSL_HIP(evsl_dev::lan_sums(n, cols, 1, true, ctx().stream));
  double s2;
  if (int e = read_scalars(red_scalar(3), 1, &s2)) return e;
  *nrm = std::sqrt(s2);
  return cgs_second(n, cols, std::sqrt(old2), nrm);
}

int nrm2_dev(int n, const double* x, double* out) {
  Context& c = ctx();
  EVSL_HIP(evsl_dev::dot_partial(n, x, x, red_part(), c.stream));
  EVSL_HIP(evsl_dev::sum_scalar(red_part(), evsl_dev::kRedBlocks, red_scalar(0), c.stream));
  double s;
  if (int e = read_scalars(red_scalar(0), 1, &s)) return e;
  *out = std::sqrt(s);
  return 0;
}


namespace {

// Lanczos with full modified Gram-Schmidt re-orthogonalisation (LanBounds,
// LanDos), enqueued without waiting: step j forms V(:, j+1) from V(:, 0..j) and
// leaves alpha_j, ||w||^2 and ||w|| in device arrays.  The host looks at them
// after the steps it asked for; a step past one where the recurrence ended has
// computed nothing that is used (a user's operator is asked for a step at a time,
// since it would be called with what that step divides by).  Up to `slots` runs from different vectors
// advance together, a column each of the step's launches, A applied to all of
// them as one interleaved block; the bits of a run do not depend on the others.
struct MgsChain {
  int n = 0, msteps = 0;
  size_t nch = 0;
  DevBuf V, scal, G, h, gt, part, xi, wi;
  double* col(int j, int s) const {
    return V.as<double>() + ((size_t)s * (msteps + 1) + j) * n;
  }
  size_t nscal() const { return 3 * (size_t)msteps + 2; }
  double* sc(int s) const { return scal.as<double>() + s * nscal(); }
  double* b2(int j, int s) const { return sc(s) + msteps + j; }
  double* b(int j, int s) const { return sc(s) + 2 * (size_t)msteps + j; }
  size_t npart() const {
    return std::max(evsl_dev::lan_part_elems(n), (size_t)3 * evsl_dev::kRedBlocks);
  }
  int init(int n_, int msteps_, int slots = 1) {
    n = n_;
    msteps = msteps_;
    nch = evsl_dev::gemv_t_chunks(n);
    const size_t S = slots * sizeof(double);
    EVSL_HIP(V.alloc((size_t)(msteps + 1) * n * S));
    EVSL_HIP(scal.alloc(nscal() * S));
    EVSL_HIP(G.alloc((size_t)msteps * msteps * S));
    EVSL_HIP(h.alloc((size_t)msteps * S));
    EVSL_HIP(gt.alloc(2 * nch * msteps * S));
    EVSL_HIP(part.alloc(npart() * S));
    if (slots > 1) {
      EVSL_HIP(xi.alloc((size_t)n * S));
      EVSL_HIP(wi.alloc((size_t)n * S));
    }
    return 0;
  }
  void release() {
    for (DevBuf* d : {&V, &scal, &G, &h, &gt, &part, &xi, &wi}) d->release();
  }
  // step j of the runs s0 .. s0 + cnt - 1
  evsl_dev::LanCols cols(int j, int s0, int cnt) const {
    evsl_dev::LanCols c{};
    for (int i = 0; i < cnt; ++i) {
      const int s = s0 + i;
      evsl_dev::LanCol& q = c.c[i];
      q.zold = j ? col(j - 1, s) : nullptr;
      q.beta_d = j ? b(j - 1, s) : nullptr;
      q.v = col(j, s);
      q.vnew = col(j + 1, s);
      q.V = col(0, s);
      q.hvec = h.as<double>() + (size_t)s * msteps;
      q.part = part.as<double>() + s * npart();
      q.gt = gt.as<double>() + (size_t)2 * s * nch * msteps;
      q.gt2 = q.gt + nch * msteps;
      q.out = sc(s) + j;
      q.G = G.as<double>() + (size_t)s * msteps * msteps;
      q.b2 = b2(j, s);
      q.b = b(j, s);
      q.k = j + 1;
      if (cnt > 1) {
        q.xi = xi.as<double>() + i;
        q.wi = wi.as<double>() + i;
        q.ldi = cnt;
      }
    }
    return c;
  }
  // V(:, 0), which holds a start vector, normalised
  int start(int s0, int cnt) {
    evsl_dev::LanCols c = cols(0, s0, cnt);
    for (int i = 0; i < cnt; ++i) {
      c.c[i].vnew = col(0, s0 + i);
      c.c[i].b2 = sc(s0 + i) + 3 * (size_t)msteps;
      c.c[i].b = c.c[i].b2 + 1;
    }
    EVSL_HIP(evsl_dev::lan_normalise(n, c, cnt, ctx().stream));
    return 0;
  }
  // V(:, j+1) minus its projections by a modified Gram-Schmidt sweep, normalised
  int sweep(int j, int s0 = 0, int cnt = 1) {
    evsl_dev::LanCols c = cols(j, s0, cnt);
    EVSL_HIP(evsl_dev::lan_mgs(n, c, cnt, msteps, ctx().stream));
    for (int i = 0; i < cnt; ++i) c.c[i].beta_d = c.c[i].b;
    EVSL_HIP(evsl_dev::lan_scale(n, c, cnt, ctx().stream));
    return 0;
  }
  // steps j0 .. j1 - 1 (more than one run: from step 0, after start())
  int run(int j0, int j1, int s0 = 0, int cnt = 1) {
    Context& c = ctx();
    for (int j = j0; j < j1; ++j) {
      if (cnt > 1) {
        EVSL_HIP(evsl_dev::cheb_spmm(c.A.view(), cnt, false, evsl_dev::kPlain, xi.p, nullptr, wi.p,
                                     nullptr, nullptr, nullptr, nullptr, 1.0, 0.0, false, 0,
                                     nullptr, c.stream));
      } else if (int e = apply_A(col(j, s0), col(j + 1, s0))) {
        return e;
      }
      EVSL_HIP(evsl_dev::lan_recurrence(n, cols(j, s0, cnt), cnt, c.stream));
      if (int e = sweep(j, s0, cnt)) return e;
    }
    return 0;
  }
  // alpha, ||w||^2 and ||w|| of every step of run s, nscal() apart (waits)
  int read(std::vector<double>& out, int s, int cnt = 1) {
    out.resize(std::max(out.size(), (s + cnt) * nscal()));
    EVSL_HIP(hipMemcpy(out.data() + s * nscal(), sc(s), cnt * nscal() * sizeof(double),
                       hipMemcpyDeviceToHost));
    return 0;
  }
};

}  // namespace

namespace {

// The restricted-trace test of ChebLanNr: the eigenvalues of T_kdim, found by a
// thread of their own while the device goes on with the next steps
struct TraceTest {
  int kdim = 0;  // 0: none under way
  int due = 0;   // the step at whose end its answer is looked at
  std::vector<double> eval, e;
  std::future<int> info;
  void set(int k, const std::vector<double>& dT, const std::vector<double>& eT) {
    kdim = k;
    eval.assign(dT.begin(), dT.begin() + k);
    e.assign(k + 1, 0.0);
    std::copy(eT.begin(), eT.begin() + (k - 1), e.begin());
  }
  int solve() { return tridiag_ql(kdim, eval.data(), e.data(), nullptr); }
};

// Steps that a test of kdim may lag.  The QL iteration takes about 0.022 kdim^2 us
// of one core (2.4 ms at 331); a step on a matrix of at most 65,536 rows takes
// about 80 us and 1 us for each degree of its filter.  Steps past the test that
// ends the run are lost, so a test lags no longer than it takes, and not at all
// where that is less than a step, on larger matrices or with a user's operator.
// A count, not a look at the clock: the steps of a run do not depend on timing.
int trace_test_lag(int kdim, int deg, int cycle) {
  Context& c = ctx();
  if (c.op != 1 || !evsl_dev::lan_small(c.n)) return 0;
  const double steps = 0.022 * kdim * kdim / (80.0 + deg);
  return std::min((int)steps, cycle - 1);
}

}  // namespace

// Ritz extraction shared by the filtered Lanczos solvers: given the
// tridiagonal T_kdim (dT, eT) and the basis V, compute Ritz pairs of A for
// the eigenvalues of T at or above bar, keep those in [a, b] with residual
// below tol (SRC/cheblanNr.c:316-399).
static int ritz_extract(int n, int kdim, const double* dT, const double* eT, const double* V,
                        double bar, double aa, double bb, double tol, int* nevOut,
                        double** lamo, double** Wo, double** reso, int maxit_alloc) {
  Context& c = ctx();
  std::vector<double> eval(kdim), e(kdim + 1, 0.0);
  std::memcpy(eval.data(), dT, kdim * sizeof(double));
  if (kdim > 1) std::memcpy(e.data(), eT, (kdim - 1) * sizeof(double));
  RotationLog rec;
  if (int err = tridiag_ql(kdim, eval.data(), e.data(), &rec)) return err;
  std::vector<int> sel;
  for (int i = 0; i < kdim; ++i)
    if (!(eval[i] < bar)) sel.push_back(i);
  const int m = (int)sel.size();
  double* Lam = (double*)std::malloc((size_t)std::max(maxit_alloc, 1) * sizeof(double));
  double* res = (double*)std::malloc((size_t)std::max(maxit_alloc, 1) * sizeof(double));
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
  const int nch = (n + 8191) / 8192;
  EVSL_HIP(part.alloc((size_t)nch * m * sizeof(double)));
  EVSL_HIP(s2.alloc(m * sizeof(double)));
  EVSL_HIP(tv.alloc(m * sizeof(double)));
  EVSL_HIP(r2.alloc(m * sizeof(double)));
  double* Ud = U.as<double>();
  double* Wd = W.as<double>();
  // U = V(:, 0:kdim) * Zsel
  EVSL_HIP(evsl_dev::gemm_nn(n, m, kdim, V, n, Zsel.as<double>(), kdim, Ud, n, c.stream));
  // normalise the columns
  EVSL_HIP(evsl_dev::col_dot(n, m, Ud, n, Ud, n, part.as<double>(), s2.as<double>(), c.stream));
  EVSL_HIP(evsl_dev::col_scale_rsqrt(n, m, Ud, n, s2.as<double>(), c.stream));
  // W = A U, Rayleigh quotients, residual norms
  for (int j = 0; j < m; ++j)
    if (int err = apply_A(Ud + (size_t)j * n, Wd + (size_t)j * n)) return err;
  EVSL_HIP(evsl_dev::col_dot(n, m, Wd, n, Ud, n, part.as<double>(), tv.as<double>(), c.stream));
  EVSL_HIP(evsl_dev::col_res2(n, m, Wd, n, Ud, n, tv.as<double>(), part.as<double>(),
                              r2.as<double>(), c.stream));
  std::vector<double> hs2(m), ht(m), hr2(m);
  EVSL_HIP(hipMemcpy(hs2.data(), s2.p, m * sizeof(double), hipMemcpyDeviceToHost));
  EVSL_HIP(hipMemcpy(ht.data(), tv.p, m * sizeof(double), hipMemcpyDeviceToHost));
  EVSL_HIP(hipMemcpy(hr2.data(), r2.p, m * sizeof(double), hipMemcpyDeviceToHost));
  std::vector<int> keep;
  int nev = 0;
  for (int j = 0; j < m; ++j) {
    if (hs2[j] == 0.0) return 2;  // zero Ritz vector (SRC/cheblanNr.c:362-364)
    const double t = ht[j];
    if (t < aa - kEpsM || t > bb + kEpsM) continue;
    const double r = std::sqrt(std::max(hr2[j], 0.0));
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

}  // namespace evsl

using namespace evsl;

extern "C" {

// SRC/cheblanNr.c:57-434
int ChebLanNr(double* intv, int maxit, double tol, double* vinit, polparams* pol, int* nevOut,
              double** lamo, double** Wo, double** reso, FILE* fstats) {
  if (int e = ensure_started()) return e;
  Context& c = ctx();
  if (c.op == 0) return EVSL_ERR_NOMAT;
  // MIXED filter precision on a CSR matrix: the one-slice case of the
  // batched solver, whose FP64 Rayleigh-Ritz refinement brings the
  // FP32-filtered Ritz pairs to tol
  if (c.filter_prec == EVSL_PREC_MIXED && c.op == 1)
    return ChebLanNr_batch(1, intv, maxit, tol, vinit, pol, nevOut, lamo, Wo, reso, fstats);
  const double t_all = evsl_timer();
  const int n = c.n;
  maxit = std::min(n, maxit);
  const double bar = pol->bar, gamB = pol->gam;
  if (check_intv(intv) < 0) {
    *nevOut = 0;
    *lamo = nullptr;
    *Wo = nullptr;
    *reso = nullptr;
    return 0;
  }
  const double aa = intv[0], bb = intv[1];
  if (fstats)
    std::fprintf(fstats, " ** Cheb Poly of deg = %d, gam = %.15e, bar: %.15e\n", pol->deg,
                 gamB, bar);
  if (gamB > 1.0 || gamB < -1.0) {
    std::fprintf(stdout, "gamB error %.15e\n", gamB);
    return -1;
  }
  const int prec = c.filter_prec;
  LanWork L;
  const size_t nl = n;
  EVSL_HIP(L.V.alloc(nl * (maxit + 1) * sizeof(double)));
  L.nch = evsl_dev::gemv_t_chunks(n);
  EVSL_HIP(L.gt_part.alloc((size_t)L.nch * (maxit + 1) * sizeof(double)));
  EVSL_HIP(L.h.alloc((size_t)(maxit + 1) * sizeof(double)));
  EVSL_HIP(L.vrand.alloc(nl * sizeof(double)));
  double* V = L.V.as<double>();
  std::vector<double> dT(maxit), eT(maxit);
  DevBuf vtmp;
  const double* v0;
  if (int e = as_device_vector(vinit, n, vtmp, &v0)) return e;
  EventClock clk;
  // filter the start vector and normalise it (FILTER_VINIT)
  clk.mark(0);
  if (int e = cheb_av(pol, v0, V, L.cw, prec)) return e;
  clk.mark(1);
  double nv;
  if (int e = nrm2_dev(n, V, &nv)) return e;
  c.astats.t_filter += clk.secs(0, 1);
  EVSL_HIP(evsl_dev::scal(n, 1.0 / nv, V, c.stream));
  double wn = 0.0, beta = 0.0, tr0 = 0.0;
  int nwn = 0, kdim = 0, k;
  const int Ntest = 30, cycle = 20;
  TraceTest test;
  // the answer of the test under way; 1: converged (SRC/cheblanNr.c:269-309)
  auto judge = [&](int info) -> int {
    kdim = test.kdim;
    test.kdim = 0;
    if (info) return EVSL_ERR_EIG;
    double tr1 = 0.0;
    int nconv = 0;
    for (double x : test.eval)
      if (x + kEpsM >= bar) {
        tr1 += x;
        ++nconv;
      }
    if (fstats)
      std::fprintf(fstats, "k %4d: nconv %4d  tr1 %21.15e\n", kdim - 1, nconv, tr1);
    const bool done = std::fabs(tr1 - tr0) < 2e-12 || std::fabs(tr1) + std::fabs(tr0) < 1e-10;
    tr0 = tr1;
    return done ? 1 : 0;
  };
  auto collect = [&]() -> int { return test.kdim ? judge(test.info.get()) : 0; };
  int done = 0;
  for (k = 0; k < maxit; ++k) {
    double* v = V + (size_t)k * nl;
    double* vnew = v + nl;
    const double* zold = k > 0 ? v - nl : nullptr;
    const double beta_prev = beta;
    double alpha, old;
    do {  // once, or again by launches where a series launch has failed
      clk.mark(0);
      if (int e = cheb_av(pol, v, vnew, L.cw, prec, true)) return e;
      clk.mark(1);
      // vnew -= beta*zold; alpha = v.vnew; vnew -= alpha*v; re-orthogonalise
      if (int e = lan_step(n, k + 1, V, beta_prev, zold, v, vnew, L, &alpha, &old,
                           &beta))
        return e;
    } while (series_failed());
    dT[k] = alpha;
    wn += std::fabs(alpha);
    {
      evsl_dev::LanCols cols = lan_col(k + 1, V, vnew, L);
      if (int e = cgs_second(n, cols, old, &beta)) return e;
    }
    clk.mark(2);
    wn += 2.0 * beta;
    nwn += 3;
    if (beta * nwn < kOrthTol * wn) {  // lucky breakdown (SRC/cheblanNr.c:225-256)
      if ((done = collect())) break;  // ends before this step: no draw
      if (fstats) std::fprintf(fstats, "it %4d: Lucky breakdown, beta = %.15e\n", k, beta);
      rand_double_device(n, L.vrand.as<double>());
      if (int e = cheb_av(pol, L.vrand.as<double>(), vnew, L.cw, prec)) return e;
      double nn;
      if (int e = nrm2_dev(n, vnew, &nn)) return e;
      if (int e = cgs_dgks(n, k + 1, V, vnew, nn * nn, &beta, L)) return e;
      EVSL_HIP(evsl_dev::scal(n, 1.0 / beta, vnew, c.stream));
      beta = 0.0;
    } else {
      EVSL_HIP(evsl_dev::scal(n, 1.0 / beta, vnew, c.stream));
    }
    eT[k] = beta;
    c.astats.t_filter += clk.secs(0, 1);
    c.astats.t_reorth += clk.secs(1, 2);
    c.astats.n_lanczos++;
    if (test.kdim && k >= test.due && (done = collect())) break;
    if ((k < Ntest || (k - Ntest) % cycle != 0) && k != maxit - 1) continue;
    // restricted-trace convergence test
    if ((done = collect())) break;
    const double te = evsl_timer();
    test.set(k + 1, dT, eT);
    const int lag = k == maxit - 1 ? 0 : trace_test_lag(test.kdim, pol->deg, cycle);
    bool started = false;
    if (lag > 0) {
      test.due = k + lag;
      try {
        test.info = std::async(std::launch::async, [&test] { return test.solve(); });
        started = true;
      } catch (const std::system_error&) {  // no thread to be had
      }
    }
    if (!started) done = judge(test.solve());
    c.astats.t_eig += evsl_timer() - te;
    if (done) break;
  }
  if (done < 0) return done;
  if (k >= maxit && fstats)
    std::fprintf(fstats, "The max number of iterations [%d] has been reached. The eigenvalues "
                         "computed may not have converged\n", maxit);
  const double tr = evsl_timer();
  int err = ritz_extract(n, kdim, dT.data(), eT.data(), V, bar, aa, bb, tol, nevOut, lamo, Wo,
                         reso, maxit);
  const double tnow = evsl_timer();
  c.astats.t_ritz += tnow - tr;
  evslstat.t_ritz = tnow - tr;
  evslstat.t_iter = tnow - t_all;
  return err;
}

// Lanczos with full (modified Gram-Schmidt) re-orthogonalization giving
// spectrum bounds (SRC/lanbounds.c:21-144).  v may be a host or device vector.
int LanBounds(int msteps, double* vin, double* lmin, double* lmax) {
  if (int e = ensure_started()) return e;
  Context& c = ctx();
  if (c.op == 0) return EVSL_ERR_NOMAT;
  const int n = c.n;
  msteps = std::min(n, msteps);
  std::vector<double> alp(msteps), bet(msteps), sc;
  DevBuf vtmp;
  MgsChain ch;
  if (int e = ch.init(n, msteps)) return e;
  const double* v;
  if (int e = as_device_vector(vin, n, vtmp, &v)) return e;
  double nv;
  if (int e = nrm2_dev(n, v, &nv)) return e;
  EVSL_HIP(evsl_dev::scal_copy(n, 1.0 / nv, v, ch.col(0, 0), c.stream));
  const bool ahead = c.op == 1;
  if (ahead) {
    if (int e = ch.run(0, msteps)) return e;
    if (int e = ch.read(sc, 0)) return e;
  }
  const int m0 = msteps;
  double wn = 0.0;
  for (int j = 0; j < msteps; ++j) {
    if (!ahead) {
      if (int e = ch.run(j, j + 1)) return e;
      if (int e = ch.read(sc, 0)) return e;
    }
    alp[j] = sc[j];
    bet[j] = sc[m0 + j];
    wn += alp[j] * alp[j];
    if (bet[j] * (j + 1) < kOrthTol * wn) {
      std::fprintf(stdout, "lanbounds: lucky break, j=%d, beta=%e, break\n", j, bet[j]);
      msteps = j + 1;
      break;
    }
    wn += 2.0 * bet[j];
    bet[j] = std::sqrt(bet[j]);
  }
  const double bottomBeta = bet[msteps - 1];
  std::vector<double> S((size_t)msteps * msteps), ritz(msteps);
  if (tridiag_eig_host(msteps, alp.data(), bet.data(), ritz.data(), S.data()))
    return EVSL_ERR_EIG;
  *lmin = ritz[0] - std::fabs(bottomBeta * S[msteps - 1]);
  *lmax = ritz[msteps - 1] + std::fabs(bottomBeta * S[(size_t)msteps * msteps - 1]);
  return 0;
}

// Lanczos DOS: nvec independent Lanczos runs with full re-orthogonalization,
// Gauss quadrature nodes/weights smoothed by Gaussians, Simpson integral
// (SRC/landos.c:37-196).  Random vectors are Box-Muller draws from libc
// rand() as in the reference.
int LanDos(const int nvec, int msteps, int npts, double* xdos, double* ydos, double* neig,
           const double* const intv) {
  if (int e = ensure_started()) return e;
  Context& c = ctx();
  if (c.op == 0) return EVSL_ERR_NOMAT;
  const int n = c.n;
  const size_t ml0 = msteps;
  std::vector<double> y(npts, 0.0), S(ml0 * ml0), gamma2(msteps), ritz(msteps);
  std::vector<int> ind(npts);
  const double lm = intv[2], lM = intv[3];
  const double tolBdwn = 1.e-13 * (std::fabs(lM) + std::fabs(lm));
  const double aa = std::max(intv[0], intv[2]), bb = std::min(intv[1], intv[3]);
  const double kappa = 1.25;
  const int M = std::min(msteps, 30);
  const double H = (lM - lm) / (M - 1);
  const double sigma = H / std::sqrt(8 * std::log(kappa));
  const double sigma2 = 2 * sigma * sigma;
  const double width = sigma * std::sqrt(-2.0 * std::log(1e-08));
  linspace(aa, bb, npts, xdos);
  // Runs from several vectors advance together on matrices whose step is launches
  // rather than bandwidth, in groups of 2, 4 and then 8: the first of them soon has
  // the device busy while the host draws the next group's vectors.
  int slots = 1;
  if (c.op == 1 && evsl_dev::lan_small(n))
    while (slots < evsl_dev::kLanCols && 2 * slots <= nvec) slots *= 2;
  std::vector<double> alp(msteps), bet(msteps), sc;
  // vectors drawn ahead of their use, in the order of the draws
  std::vector<std::vector<double>> drawn;
  auto draw = [&](size_t count) {
    while (drawn.size() < count) {
      drawn.emplace_back(n);
      randn_double(n, drawn.back().data());
    }
  };
  MgsChain ch;
  // as many runs as there is memory for (the bits of a run do not depend on it)
  while (int e = ch.init(n, msteps, slots)) {
    if (slots == 1) return e;
    slots /= 2;
    ch.release();
    (void)hipGetLastError();
    clear_error();
  }
  const int m0 = msteps;
  const bool ahead = c.op == 1;
  int have = 0, next = 0, group = 1;  // runs of the current group, the next one to look at
  for (int m = 0; m < nvec; ++m) {
    if (next == have) {
      auto size_of = [&](int left) {
        int g = std::min(slots, 2 * group);
        while (g > left) g /= 2;
        return g;
      };
      have = size_of(nvec - m);
      group = have;
      next = 0;
      draw(have);
      for (int s = 0; s < have; ++s)
        EVSL_HIP(hipMemcpy(ch.col(0, s), drawn[s].data(), n * sizeof(double),
                           hipMemcpyHostToDevice));
      drawn.erase(drawn.begin(), drawn.begin() + have);
      if (int e = ch.start(0, have)) return e;
      if (ahead) {
        if (int e = ch.run(0, msteps, 0, have)) return e;
        // the next group's draws while the device runs this one
        const int left = nvec - m - have;
        if (left > 0) draw(size_of(left));
      }
      if (int e = ch.read(sc, 0, have)) return e;
    }
    const int s = next++;
    const double* scs = sc.data() + s * ch.nscal();
    double wn = 0.0;
    for (int j = 0; j < msteps; ++j) {
      if (!ahead) {
        if (int e = ch.run(j, j + 1, s)) return e;
        if (int e = ch.read(sc, s)) return e;
      }
      alp[j] = scs[j];
      bet[j] = scs[m0 + j];
      wn += alp[j] * alp[j];
      if (bet[j] * (j + 1) < kOrthTol * wn) {
        std::fprintf(stdout, "lanbounds: lucky break, j=%d, beta=%e, break\n", j, bet[j]);
        msteps = j + 1;
        break;
      }
      if (bet[j] > tolBdwn) {
        wn += 2.0 * bet[j];
        bet[j] = std::sqrt(bet[j]);
      } else {
        // the reference draws the replacement into v, which is then unused
        // (SRC/landos.c:130-144); the stream of rand() calls is kept the same:
        // the replacement is the next draw, whose run is left out where there
        // is one already
        if (next < have) {
          ++next;
        } else {
          draw(1);
          drawn.erase(drawn.begin());
        }
        // another sweep of V(:, j+1), which stands normalised: its norm is
        // taken back into the squared norm of what it was
        if (int e = ch.sweep(j, s)) return e;
        const double was = bet[j];
        double again;
        if (int e = read_scalars(ch.b2(j, s), 1, &again)) return e;
        wn += 2.0 * was * again;
        bet[j] = 0;
        const double zero = 0.0;
        EVSL_HIP(hipMemcpy(ch.b(j, s), &zero, sizeof(double), hipMemcpyHostToDevice));
        if (ahead) {
          if (int e = ch.run(j + 1, msteps, s)) return e;
          if (int e = ch.read(sc, s)) return e;
        }
      }
    }
    if (tridiag_eig_host(msteps, alp.data(), bet.data(), ritz.data(), S.data()))
      return EVSL_ERR_EIG;
    for (int i = 0; i < msteps; ++i) gamma2[i] = S[i * ml0] * S[i * ml0];
    for (int i = 0; i < msteps; ++i) {
      const double t = ritz[i];
      int np = 0;
      for (int j = 0; j < npts; ++j)
        if (std::fabs(xdos[j] - t) < width) ind[np++] = j;
      for (int j = 0; j < np; ++j)
        y[ind[j]] += gamma2[i] * std::exp(-((xdos[ind[j]] - t) * (xdos[ind[j]] - t)) / sigma2);
    }
  }
  const double scaling = 1.0 / (nvec * std::sqrt(sigma2 * EVSL_PI));
  for (int j = 0; j < npts; ++j) y[j] *= scaling;
  std::memcpy(ydos, y.data(), npts * sizeof(double));
  // in-place Simpson integration (SRC/simpson.c:25-50)
  {
    double tc = 0.0, ti, tm, ysav = y[0];
    int i = 1;
    y[0] = 0;
    while (i < npts - 1) {
      ti = (xdos[i] - xdos[i - 1]) * (ysav + y[i]) / 2.0;
      tm = tc + ti;
      ti = (xdos[i + 1] - xdos[i - 1]) * (ysav + 4 * y[i] + y[i + 1]) / 6.0;
      tc += ti;
      y[i] = tm;
      ysav = y[i + 1];
      y[i + 1] = tc;
      i += 2;
    }
    if (i == npts - 1) y[i] = tc + (xdos[i] - xdos[i - 1]) * (y[i] + ysav) / 2.0;
  }
  *neig = y[npts - 1] * n;
  return 0;
}

// Thick-restart filtered Lanczos (SRC/cheblanTr.c:59-707).  The basis V
// (n x (lanm+1)), the locked block Y and the Ritz block live in HBM; the
// arrow-head matrix T and its dense eigensolve stay on the host.  The filter
// always runs in FP64: restarts lock Ritz pairs on their residual with A, so
// an FP32-filtered basis would never lock pairs below its rounding level.
int ChebLanTr(int lanm, int nev, double* intv, int maxit, double tol, double* vinit,
              polparams* pol, int* nev2, double** vals, double** W, double** resW,
              FILE* fstats) {
  if (int e = ensure_started()) return e;
  Context& c = ctx();
  if (c.op == 0) return EVSL_ERR_NOMAT;
  const double t_all = evsl_timer();
  const int n = c.n;
  const size_t nl = n;
  lanm = std::min(lanm, n);
  const int lanm1 = lanm + 1;
  const size_t L1 = lanm1;
  if (lanm == n) maxit = std::min(maxit, n);
  const double nevInc = 0.2;
  const int cycle = 50, min_inner_step = 5;
  if (check_intv(intv) < 0) {
    *nev2 = 0;
    *vals = nullptr;
    *W = nullptr;
    *resW = nullptr;
    return 0;
  }
  const double aa = intv[0], bb = intv[1];
  const double gamB = pol->gam, bar = pol->bar;
  if (gamB > 1.0 || gamB < -1.0) {
    if (fstats) std::fprintf(fstats, "gamB error %.15e\n", gamB);
    return -1;
  }
  if (lanm < 1) {
    set_error_msg("ChebLanTr: lanm must be positive");
    return EVSL_ERR_ARG;
  }
  if (fstats) std::fprintf(fstats, " Cheb-LanTR, dim %d  cycle %d  \n", lanm, cycle);
  const int prec = EVSL_PREC_FP64;
  int ycap = std::max(nev, 1);
  LanWork L;
  L.nch = evsl_dev::gemv_t_chunks(n);
  int gcap = 0;  // columns the Gram-Schmidt scratch holds
  auto ensure_gs = [&](int cols) -> int {
    if (cols <= gcap) return 0;
    gcap = cols;
    EVSL_HIP(L.gt_part.alloc((size_t)L.nch * (gcap + 1) * sizeof(double)));
    EVSL_HIP(L.h.alloc((size_t)(gcap + 1) * sizeof(double)));
    return 0;
  };
  if (int e = ensure_gs(std::max(lanm1, ycap))) return e;
  EVSL_HIP(L.V.alloc(nl * L1 * sizeof(double)));
  EVSL_HIP(L.vrand.alloc(nl * sizeof(double)));
  DevBuf Yd, Rvec, Wblk, Ed, part, s2d, tvd, r2d;
  EVSL_HIP(Yd.alloc(nl * ycap * sizeof(double)));
  EVSL_HIP(Rvec.alloc(nl * lanm * sizeof(double)));
  constexpr int kChunk = 64;  // Ritz columns per A-application block
  EVSL_HIP(Wblk.alloc(nl * std::min(kChunk, lanm) * sizeof(double)));
  const int nch8 = (n + 8191) / 8192;
  EVSL_HIP(part.alloc((size_t)nch8 * lanm * sizeof(double)));
  EVSL_HIP(s2d.alloc(lanm * sizeof(double)));
  EVSL_HIP(tvd.alloc(lanm * sizeof(double)));
  EVSL_HIP(r2d.alloc(lanm * sizeof(double)));
  double* V = L.V.as<double>();
  std::vector<double> T(L1 * L1, 0.0), EvecT(L1 * L1), Rval(lanm), resi(lanm), s(lanm);
  std::vector<double> Lam(ycap), res(ycap);
  DevBuf vtmp;
  const double* v0;
  if (int e = as_device_vector(vinit, n, vtmp, &v0)) return e;
  EventClock clk;
  int lock = 0, trlen = 0, prtrlen = -1, it = 0;
  // filter the start vector and normalise it (FILTER_VINIT)
  if (int e = cheb_av(pol, v0, V, L.cw, prec)) return e;
  double nv;
  if (int e = nrm2_dev(n, V, &nv)) return e;
  EVSL_HIP(evsl_dev::scal(n, 1.0 / nv, V, c.stream));
  // deflation against the locked block: v -= Y Y^T v (two CGS passes at most)
  auto deflate = [&](double* vnew) -> int {
    if (lock == 0) return 0;
    double nn, dummy;
    if (int e = nrm2_dev(n, vnew, &nn)) return e;
    return cgs_dgks(n, lock, Yd.as<double>(), vnew, nn * nn, &dummy, L);
  };
  // lucky breakdown: a filtered random vector orthogonalised against Y and V(:,0:k)
  auto breakdown = [&](int k, double* vnew, double* beta) -> int {
    rand_double_device(n, L.vrand.as<double>());
    if (int e = cheb_av(pol, L.vrand.as<double>(), vnew, L.cw, prec)) return e;
    if (int e = deflate(vnew)) return e;
    double nn;
    if (int e = nrm2_dev(n, vnew, &nn)) return e;
    if (int e = cgs_dgks(n, k, V, vnew, nn * nn, beta, L)) return e;
    EVSL_HIP(evsl_dev::scal(n, 1.0 / *beta, vnew, c.stream));
    *beta = 0.0;
    return 0;
  };
  while (it < maxit) {
    double wn = 0.0, beta = 0.0;
    int nwn = 0;
    int k = trlen > 0 ? trlen + 1 : 0;
    if (k + min_inner_step > lanm1) {  // the reference exits here
      if (fstats) std::fprintf(fstats, "Krylov dim too small for this problem. Try a larger dim\n");
      set_error_msg("ChebLanTr: Krylov dimension too small for the restart set");
      return EVSL_ERR_ARG;
    }
    if (trlen > 0) {  // thick-restart special step (SRC/cheblanTr.c:224-319)
      const int k1 = k - 1;
      double* v = V + (size_t)k1 * nl;
      double* vnew = v + nl;
      clk.mark(0);
      if (int e = cheb_av(pol, v, vnew, L.cw, prec)) return e;
      clk.mark(1);
      c.astats.t_filter += clk.secs(0, 1);
      if (int e = deflate(vnew)) return e;
      for (int i = 0; i < trlen; ++i) {
        T[i * L1 + i] = Rval[i];
        wn += std::fabs(Rval[i]);
      }
      EVSL_HIP(evsl_dev::dot_partial(n, v, vnew, red_part(), c.stream));
      EVSL_HIP(evsl_dev::sum_scalar(red_part(), evsl_dev::kRedBlocks, red_scalar(0), c.stream));
      if (int e = read_scalars(red_scalar(0), 1, &s[k1])) return e;
      // vnew -= V(:, 0:k) s(0:k), with ||vnew||^2
      EVSL_HIP(hipMemcpy(L.h.p, s.data(), (size_t)k * sizeof(double), hipMemcpyHostToDevice));
      const int nb = (n + evsl_dev::kWG - 1) / evsl_dev::kWG;
      EVSL_HIP(evsl_dev::gemv_n_sub_nrm(n, k, V, n, L.h.as<double>(), vnew, red_part(), c.stream));
      EVSL_HIP(evsl_dev::sum_scalar(red_part(), nb, red_scalar(1), c.stream));
      for (int i = 0; i < k1; ++i) {
        T[trlen * L1 + i] = s[i];
        T[i * L1 + trlen] = s[i];
        wn += 2.0 * std::fabs(s[i]);
      }
      T[trlen * L1 + trlen] = s[k1];
      wn += std::fabs(s[k1]);
      double b2;
      if (int e = read_scalars(red_scalar(1), 1, &b2)) return e;
      beta = std::sqrt(b2);
      wn += 2.0 * beta;
      nwn += 3 * k;
      if (beta * nwn < kOrthTol * wn) {
        if (fstats) std::fprintf(fstats, "it %4d: Lucky breakdown, beta = %.15e\n", k, beta);
        if (int e = breakdown(k, vnew, &beta)) return e;
      } else {
        EVSL_HIP(evsl_dev::scal(n, 1.0 / beta, vnew, c.stream));
      }
      T[k1 * L1 + k] = beta;
      T[k * L1 + k1] = beta;
    }
    const int Ntest = std::max(20, nev - lock + 10);
    int last_jl = 0;
    double last_tr = 0.0;
    const double* zold = k > 0 ? V + (size_t)(k - 1) * nl : nullptr;
    while (k < lanm && it < maxit) {  // Lanczos inner loop (SRC/cheblanTr.c:331-503)
      ++k;
      double* v = V + (size_t)(k - 1) * nl;
      double* vnew = v + nl;
      clk.mark(0);
      if (int e = cheb_av(pol, v, vnew, L.cw, prec)) return e;
      clk.mark(1);
      ++it;
      if (int e = deflate(vnew)) return e;
      // vnew -= beta*zold; alpha = v.vnew; vnew -= alpha*v; re-orthogonalise
      double alpha, old;
      if (int e = lan_step(n, k, V, beta, zold, v, vnew, L, &alpha, &old, &beta)) return e;
      T[(k - 1) * L1 + (k - 1)] = alpha;
      wn += std::fabs(alpha);
      {
        evsl_dev::LanCols cols = lan_col(k, V, vnew, L);
        if (int e = cgs_second(n, cols, old, &beta)) return e;
      }
      clk.mark(2);
      wn += 2.0 * beta;
      nwn += 3;
      zold = v;
      if (beta * nwn < kOrthTol * wn) {
        if (fstats) std::fprintf(fstats, "it %4d: Lucky breakdown, beta = %.15e\n", it, beta);
        if (int e = breakdown(k, vnew, &beta)) return e;
      } else {
        EVSL_HIP(evsl_dev::scal(n, 1.0 / beta, vnew, c.stream));
      }
      T[k * L1 + (k - 1)] = beta;
      T[(k - 1) * L1 + k] = beta;
      c.astats.t_filter += clk.secs(0, 1);
      c.astats.t_reorth += clk.secs(1, 2);
      c.astats.n_lanczos++;
      const int k1 = k - trlen - Ntest;
      if (((k1 >= 0) && (k1 % cycle == 0)) || (k == lanm) || it == maxit) {
        const double te = evsl_timer();
        if (int e = sym_eig_host(k, T.data(), lanm1, EvecT.data(), lanm1, Rval.data())) return e;
        c.astats.t_eig += evsl_timer() - te;
        if (k == lanm || it == maxit) break;
        int jl = 0;
        double tr = 0.0;
        for (int i = 0; i < k; ++i)
          if (Rval[i] + kEpsM >= bar) {
            ++jl;
            tr += Rval[i];
          }
        if (std::fabs(tr - last_tr) <= 2e-12 && jl == last_jl) {
          if (fstats)
            std::fprintf(fstats,
                         "break: [it %d, k %d]: last_tr %.15e, tr %.15e, last_jl %d  jl %d\n", it,
                         k, last_tr, tr, last_jl, jl);
          break;
        }
        if (fstats)
          std::fprintf(fstats, "[it %d, k %d] testing: last_tr %.15e, tr %.15e, last_jl %d  jl %d\n",
                       it, k, last_tr, tr, last_jl, jl);
        last_tr = tr;
        last_jl = jl;
      }
    }
    const double tr0 = evsl_timer();
    // pass 1: Ritz values of p(A) at or above bar, moved to the front
    int jl = 0;
    for (int i = 0; i < k; ++i) {
      if (Rval[i] + kEpsM >= bar) {
        if (i != jl) {
          std::memcpy(&EvecT[jl * L1], &EvecT[i * L1], (size_t)k * sizeof(double));
          Rval[jl] = Rval[i];
        }
        resi[jl] = std::fabs(beta * EvecT[i * L1 + (k - 1)]);
        ++jl;
      }
    }
    // Rvec(:, 0:jl) = V(:, 0:k) EvecT(0:k, 0:jl)
    double* R = Rvec.as<double>();
    std::vector<double> hs2(jl), ht(jl), hr2(jl);
    if (jl > 0) {
      std::vector<double> Eh((size_t)k * jl);
      for (int j = 0; j < jl; ++j)
        std::memcpy(&Eh[(size_t)j * k], &EvecT[j * L1], (size_t)k * sizeof(double));
      EVSL_HIP(Ed.alloc(Eh.size() * sizeof(double)));
      EVSL_HIP(hipMemcpy(Ed.p, Eh.data(), Eh.size() * sizeof(double), hipMemcpyHostToDevice));
      EVSL_HIP(evsl_dev::gemm_nn(n, jl, k, V, n, Ed.as<double>(), k, R, n, c.stream));
      EVSL_HIP(evsl_dev::col_dot(n, jl, R, n, R, n, part.as<double>(), s2d.as<double>(), c.stream));
      EVSL_HIP(hipMemcpy(hs2.data(), s2d.p, jl * sizeof(double), hipMemcpyDeviceToHost));
      for (int i = 0; i < jl; ++i)
        if (hs2[i] == 0.0) return 2;  // zero Ritz vector (SRC/cheblanTr.c:562-564)
      EVSL_HIP(evsl_dev::col_scale_rsqrt(n, jl, R, n, s2d.as<double>(), c.stream));
      // Rayleigh quotients and residuals, kChunk columns at a time
      double* Wb = Wblk.as<double>();
      for (int j0 = 0; j0 < jl; j0 += kChunk) {
        const int m = std::min(kChunk, jl - j0);
        for (int j = 0; j < m; ++j)
          if (int e = apply_A(R + (size_t)(j0 + j) * nl, Wb + (size_t)j * nl)) return e;
        EVSL_HIP(evsl_dev::col_dot(n, m, Wb, n, R + (size_t)j0 * nl, n, part.as<double>(),
                                   tvd.as<double>() + j0, c.stream));
        EVSL_HIP(evsl_dev::col_res2(n, m, Wb, n, R + (size_t)j0 * nl, n, tvd.as<double>() + j0,
                                    part.as<double>(), r2d.as<double>() + j0, c.stream));
      }
      EVSL_HIP(hipMemcpy(ht.data(), tvd.p, jl * sizeof(double), hipMemcpyDeviceToHost));
      EVSL_HIP(hipMemcpy(hr2.data(), r2d.p, jl * sizeof(double), hipMemcpyDeviceToHost));
    }
    // pass 2: Ritz values of A in [a, b] are locked or kept for the restart
    int ll = 0;
    prtrlen = trlen;
    trlen = 0;
    for (int i = 0; i < jl; ++i) {
      const double t3 = ht[i];
      if (!(t3 >= aa - kEpsM && t3 <= bb + kEpsM)) continue;
      ++ll;
      const double res0 = std::sqrt(std::max(hr2[i], 0.0));
      const double* y = R + (size_t)i * nl;
      if (res0 < tol) {
        if (lock >= nev) {  // grow the locked block by 1 + 20%
          nev += 1 + (int)(nev * nevInc);
          if (fstats) std::fprintf(fstats, "-- More eigval found: realloc space for %d evs\n", nev);
        }
        if (lock >= ycap) {
          const int ncap = std::max(nev, lock + 1);
          DevBuf Y2;
          EVSL_HIP(Y2.alloc(nl * ncap * sizeof(double)));
          EVSL_HIP(hipMemcpyAsync(Y2.p, Yd.p, nl * lock * sizeof(double),
                                  hipMemcpyDeviceToDevice, c.stream));
          std::swap(Yd.p, Y2.p);
          std::swap(Yd.bytes, Y2.bytes);
          ycap = ncap;
          Lam.resize(ycap);
          res.resize(ycap);
          if (int e = ensure_gs(std::max(lanm1, ycap))) return e;
        }
        EVSL_HIP(hipMemcpyAsync(Yd.as<double>() + (size_t)lock * nl, y, nl * sizeof(double),
                                hipMemcpyDeviceToDevice, c.stream));
        Lam[lock] = t3;
        res[lock] = res0;
        ++lock;
      } else {
        Rval[trlen] = Rval[i];
        EVSL_HIP(hipMemcpyAsync(V + (size_t)trlen * nl, y, nl * sizeof(double),
                                hipMemcpyDeviceToDevice, c.stream));
        s[trlen] = beta * EvecT[i * L1 + (k - 1)];
        ++trlen;
      }
    }
    c.astats.t_ritz += evsl_timer() - tr0;
    if (fstats)
      std::fprintf(fstats, "it %4d:  k %3d, jl %3d, ll %3d, lock %3d, trlen %3d\n", it, k, jl, ll,
                   lock, trlen);
    if (prtrlen == 0 && ll == 0) {
      if (fstats)
        std::fprintf(fstats, "--------------------------------------------------\n"
                             " --> No ev.s left to be computed\n");
      break;
    }
    if (it == maxit) {
      if (fstats)
        std::fprintf(fstats, "--------------------------------------------------\n"
                             " --> Max its reached without convergence\n");
      break;
    }
    std::fill(T.begin(), T.end(), 0.0);
    if (trlen != k)
      EVSL_HIP(hipMemcpyAsync(V + (size_t)trlen * nl, V + (size_t)k * nl, nl * sizeof(double),
                              hipMemcpyDeviceToDevice, c.stream));
  }
  if (fstats)
    std::fprintf(fstats, "     Number of evals found = %d\n"
                         "--------------------------------------------------\n", lock);
  EVSL_HIP(hipStreamSynchronize(c.stream));
  // outputs: host Lam/res (evsl_Malloc), device Y (evsl_Malloc_device)
  double* lam_o = (double*)std::malloc((size_t)std::max(lock, 1) * sizeof(double));
  double* res_o = (double*)std::malloc((size_t)std::max(lock, 1) * sizeof(double));
  double* Y_o = (double*)_evsl_Malloc_device(nl * std::max(lock, 1) * sizeof(double));
  if (!lam_o || !res_o || !Y_o) {
    std::free(lam_o);
    std::free(res_o);
    if (Y_o) _evsl_Free_device(Y_o);
    return EVSL_ERR_ALLOC;
  }
  if (lock > 0) {
    std::memcpy(lam_o, Lam.data(), lock * sizeof(double));
    std::memcpy(res_o, res.data(), lock * sizeof(double));
    EVSL_HIP(hipMemcpy(Y_o, Yd.p, nl * lock * sizeof(double), hipMemcpyDeviceToDevice));
  }
  *nev2 = lock;
  *vals = lam_o;
  *W = Y_o;
  *resW = res_o;
  evslstat.t_iter = evsl_timer() - t_all;
  return 0;
}


// Thick-restart Lanczos spectrum bounds (SRC/lanTrbounds.c:35-421): Lanczos
// on A with full reorthogonalization, restarted from the two extreme Ritz
// pairs until the bound corrections fall below tol * (|lmin| + |lmax|).
// bndtype <= 1: simple bounds |beta s|; otherwise Kato-Temple.
int LanTrbounds(int lanm, int maxit, double tol, double* vinit, int bndtype, double* lammin,
                double* lammax, FILE* fstats) {
  if (int e = ensure_started()) return e;
  Context& c = ctx();
  if (c.op == 0) return EVSL_ERR_NOMAT;
  const int n = c.n;
  const size_t nl = n;
  lanm = std::min(lanm, n);
  const int lanm1 = lanm + 1;
  const size_t L1 = lanm1;
  if (lanm == n) maxit = std::min(maxit, n);
  const int min_inner_step = 5;
  if (fstats) std::fprintf(fstats, " LanTR for bounds: dim %d, maxits %d\n", lanm, maxit);
  LanWork L;
  L.nch = evsl_dev::gemv_t_chunks(n);
  EVSL_HIP(L.gt_part.alloc((size_t)L.nch * (lanm1 + 1) * sizeof(double)));
  EVSL_HIP(L.h.alloc((size_t)(lanm1 + 1) * sizeof(double)));
  EVSL_HIP(L.V.alloc(nl * L1 * sizeof(double)));
  DevBuf Rvec, Ed;
  EVSL_HIP(Rvec.alloc(2 * nl * sizeof(double)));
  double* V = L.V.as<double>();
  std::vector<double> T(L1 * L1, 0.0), EvecT(L1 * L1), Rval(std::max(lanm, 2));
  double s[3] = {0.0, 0.0, 0.0};
  DevBuf vtmp;
  const double* v0;
  if (int e = as_device_vector(vinit, n, vtmp, &v0)) return e;
  EVSL_HIP(hipMemcpyAsync(V, v0, nl * sizeof(double), hipMemcpyDeviceToDevice, c.stream));
  double nv;
  if (int e = nrm2_dev(n, V, &nv)) return e;
  EVSL_HIP(evsl_dev::scal(n, 1.0 / nv, V, c.stream));
  const int nb = (n + evsl_dev::kWG - 1) / evsl_dev::kWG;
  // lucky breakdown: a random vector orthogonalised against V(:, 0:k)
  auto breakdown = [&](int k, double* vnew, double* beta) -> int {
    rand_double_device(n, vnew);
    double nn;
    if (int e = nrm2_dev(n, vnew, &nn)) return e;
    if (int e = cgs_dgks(n, k, V, vnew, nn * nn, beta, L)) return e;
    EVSL_HIP(evsl_dev::scal(n, 1.0 / *beta, vnew, c.stream));
    *beta = 0.0;
    return 0;
  };
  double lmin = 0.0, lmax = 0.0;
  int it = 0, trlen = 0;
  while (it < maxit) {
    double wn = 0.0, beta = 0.0;
    int nwn = 0;
    int k = trlen > 0 ? trlen + 1 : 0;
    if (k + min_inner_step > lanm1) {  // the reference exits here
      set_error_msg("LanTrbounds: Krylov dimension too small");
      return EVSL_ERR_ARG;
    }
    if (trlen > 0) {  // thick-restart special step (SRC/lanTrbounds.c:145-215)
      const int k1 = k - 1;
      double* v = V + (size_t)k1 * nl;
      double* vnew = v + nl;
      if (int e = apply_A(v, vnew)) return e;
      for (int i = 0; i < trlen; ++i) {
        T[i * L1 + i] = Rval[i];
        wn += std::fabs(Rval[i]);
      }
      EVSL_HIP(evsl_dev::dot_partial(n, v, vnew, red_part(), c.stream));
      EVSL_HIP(evsl_dev::sum_scalar(red_part(), evsl_dev::kRedBlocks, red_scalar(0), c.stream));
      if (int e = read_scalars(red_scalar(0), 1, &s[k1])) return e;
      EVSL_HIP(hipMemcpy(L.h.p, s, (size_t)k * sizeof(double), hipMemcpyHostToDevice));
      EVSL_HIP(evsl_dev::gemv_n_sub_nrm(n, k, V, n, L.h.as<double>(), vnew, red_part(), c.stream));
      EVSL_HIP(evsl_dev::sum_scalar(red_part(), nb, red_scalar(1), c.stream));
      for (int i = 0; i < k1; ++i) {
        T[trlen * L1 + i] = s[i];
        T[i * L1 + trlen] = s[i];
        wn += 2.0 * std::fabs(s[i]);
      }
      T[trlen * L1 + trlen] = s[k1];
      wn += std::fabs(s[k1]);
      double b2;
      if (int e = read_scalars(red_scalar(1), 1, &b2)) return e;
      beta = std::sqrt(b2);
      wn += 2.0 * beta;
      nwn += 3 * k;
      if (beta * nwn < kOrthTol * wn) {
        if (int e = breakdown(k, vnew, &beta)) return e;
      } else {
        EVSL_HIP(evsl_dev::scal(n, 1.0 / beta, vnew, c.stream));
      }
      T[k1 * L1 + k] = beta;
      T[k * L1 + k1] = beta;
    }
    const double* zold = k > 0 ? V + (size_t)(k - 1) * nl : nullptr;
    while (k < lanm && it < maxit) {  // Lanczos inner loop (SRC/lanTrbounds.c:222-300)
      ++k;
      double* v = V + (size_t)(k - 1) * nl;
      double* vnew = v + nl;
      if (int e = apply_A(v, vnew)) return e;
      ++it;
      double alpha, old;
      if (int e = lan_step(n, k, V, beta, zold, v, vnew, L, &alpha, &old, &beta)) return e;
      T[(k - 1) * L1 + (k - 1)] = alpha;
      wn += std::fabs(alpha);
      {
        evsl_dev::LanCols cols = lan_col(k, V, vnew, L);
        if (int e = cgs_second(n, cols, old, &beta)) return e;
      }
      wn += 2.0 * beta;
      nwn += 3;
      zold = v;
      if (beta * nwn < kOrthTol * wn) {
        if (fstats) std::fprintf(fstats, "it %4d: Lucky breakdown, beta = %.15e\n", it, beta);
        if (int e = breakdown(k, vnew, &beta)) return e;
      } else {
        EVSL_HIP(evsl_dev::scal(n, 1.0 / beta, vnew, c.stream));
      }
      T[k * L1 + (k - 1)] = beta;
      T[(k - 1) * L1 + k] = beta;
      c.astats.n_lanczos++;
    }
    if (k < 2) {
      set_error_msg("LanTrbounds: fewer than two Lanczos steps");
      return EVSL_ERR_ARG;
    }
    if (int e = sym_eig_host(k, T.data(), lanm1, EvecT.data(), lanm1, Rval.data())) return e;
    // spikes: beta times the last components of the extreme eigenvectors
    s[0] = beta * EvecT[k - 1];
    s[1] = beta * EvecT[(size_t)(k - 1) * L1 + (k - 1)];
    double t1, t2;
    if (bndtype <= 1) {
      t1 = std::fabs(s[0]);
      t2 = std::fabs(s[1]);
    } else {  // Kato-Temple
      t1 = 2.0 * s[0] * s[0] / (Rval[1] - Rval[0]);
      t2 = 2.0 * s[1] * s[1] / (Rval[k - 1] - Rval[k - 2]);
    }
    lmin = Rval[0] - t1;
    lmax = Rval[k - 1] + t2;
    // the two extreme Ritz vectors become the restart set
    std::vector<double> Eh((size_t)2 * k);
    std::memcpy(Eh.data(), &EvecT[0], (size_t)k * sizeof(double));
    std::memcpy(Eh.data() + k, &EvecT[(size_t)(k - 1) * L1], (size_t)k * sizeof(double));
    EVSL_HIP(Ed.alloc(Eh.size() * sizeof(double)));
    EVSL_HIP(hipMemcpy(Ed.p, Eh.data(), Eh.size() * sizeof(double), hipMemcpyHostToDevice));
    EVSL_HIP(evsl_dev::gemm_nn(n, 2, k, V, n, Ed.as<double>(), k, Rvec.as<double>(), n,
                               c.stream));
    trlen = 2;
    EVSL_HIP(hipMemcpyAsync(V, Rvec.p, 2 * nl * sizeof(double), hipMemcpyDeviceToDevice,
                            c.stream));
    Rval[1] = Rval[k - 1];
    if (fstats)
      std::fprintf(fstats, "it %4d, k %3d: ritz %.15e %.15e, t1,t2 %e %e, res %.15e %.15e\n", it,
                   k, Rval[0], Rval[1], t1, t2, std::fabs(s[0]), std::fabs(s[1]));
    if (t1 + t2 < tol * (std::fabs(lmin) + std::fabs(lmax))) break;
    std::fill(T.begin(), T.end(), 0.0);
    EVSL_HIP(hipMemcpyAsync(V + (size_t)trlen * nl, V + (size_t)k * nl, nl * sizeof(double),
                            hipMemcpyDeviceToDevice, c.stream));
  }
  EVSL_HIP(hipStreamSynchronize(c.stream));
  *lammin = lmin;
  *lammax = lmax;
  return 0;
}

}  // extern "C"
