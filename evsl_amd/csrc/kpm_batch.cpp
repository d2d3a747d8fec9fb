// kpm_batch.cpp -- KPM densities of many matrices in one batched run.
//
// Each request is kpmdos (SRC/spslice.c:29-148) on its own matrix and
// interval: nvec seeded device random vectors in column blocks of up to 32,
// a three-term Chebyshev recurrence per block, and the moments
// mu_k ~ sum_m v_m^T T_k(A~) v_m.  The requests advance together: one grouped
// launch per degree runs the row blocks of every matrix (owner table ->
// matrix entry), so small matrices fill the device beside large ones, and
// one grouped reduction per degree sums each matrix's block partials in the
// order the one-matrix path uses.  In FP64 a request's moments equal
// kpmdos_ex on its matrix with the same seed bit for bit; EVSL_PREC_MIXED
// runs the recurrence in FP32 on (A - ctr I) * 2^-s with the moment dots
// accumulated in FP64.
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstring>
#include <map>
#include <memory>
#include <string>
#include <vector>

#include "internal.h"

namespace evsl {
namespace {

// Places in one allocation, 256 bytes apart: a call's buffers are many and small,
// and an allocation and a free of its own for each cost more than the kernels.
struct Places {
  size_t end = 0;
  size_t take(size_t bytes) {
    const size_t at = end;
    end += (bytes + 255) / 256 * 256;
    return at;
  }
};

// one distinct matrix of the batch, resident for the call
struct BatchMatrix {
  const csrMat* host = nullptr;
  int n = 0, nnz = 0;
  bool full_diag = false;
  bool regular = false;
  size_t ia_at = 0, ja_at = 0, a64_at = 0;
  const int *ia = nullptr, *ja = nullptr;
  const double* a64 = nullptr;
  std::map<int, std::vector<int>> table;  // row-block table by lanes per row
  evsl_dev::Csr view() const {
    evsl_dev::Csr v;
    v.n = n;
    v.nnz = nnz;
    v.ia = ia;
    v.ja = ja;
    v.a64 = a64;
    return v;
  }
  const std::vector<int>& row_blocks(int lanes) {
    std::vector<int>& rbp = table[lanes];
    if (rbp.empty()) {
      std::vector<int> rb = make_row_blocks(host->ia, n, evsl_dev::rows_cap_for(lanes));
      rbp.resize(2 * rb.size());
      for (size_t i = 0; i < rb.size(); ++i) {
        rbp[2 * i] = rb[i];
        rbp[2 * i + 1] = host->ia[rb[i]];
      }
    }
    return rbp;
  }
};

// FP32 values of a matrix, shared by the requests with its centre and scale
struct BatchValues {
  BatchMatrix* mat = nullptr;
  double ctr = 0, scale = 0;  // scale 0: the values as they are
  size_t at = 0;
};

// one request
struct BatchRequest {
  BatchMatrix* mat = nullptr;
  const double* intv = nullptr;
  unsigned long long seed = 0;
  double ctr = 0, wid = 0, t0 = 0, t = 0, cc = 0;
  int a32 = -1;  // its BatchValues
  std::vector<double> raw;
};

}  // namespace
}  // namespace evsl

using namespace evsl;

extern "C" {

int kpmdos_batch(int nreq, csrMat* const* mats, const double* intvs, int Mdeg, int damping,
                 int nvec, int vec_kind, const unsigned long long* seeds, int prec, double* mu,
                 double* ecnt) {
  if (int e = ensure_started()) return e;
  Context& c = ctx();
  if (nreq <= 0 || !mats || !intvs || !mu || !ecnt || Mdeg < 0 || nvec <= 0 ||
      (prec != EVSL_PREC_FP64 && prec != EVSL_PREC_MIXED)) {
    set_error_msg("kpmdos_batch: invalid arguments");
    return EVSL_ERR_ARG;
  }
  if (vec_kind != EVSL_VEC_RADEMACHER && vec_kind != EVSL_VEC_GAUSSIAN) {
    set_error_msg("kpmdos_batch: vec_kind must be EVSL_VEC_RADEMACHER or EVSL_VEC_GAUSSIAN");
    return EVSL_ERR_UNSUPP;
  }
  for (int r = 0; r < nreq; ++r) {
    const csrMat* A = mats[r];
    if (!A || A->nrows <= 0 || A->nrows != A->ncols || !A->ia || (A->ia[A->nrows] > 0 && (!A->ja || !A->a))) {
      set_error_msg("kpmdos_batch: request " + std::to_string(r) + " has no square CSR matrix");
      return EVSL_ERR_ARG;
    }
    const double* iv = intvs + 4 * r;
    if (iv[0] >= iv[1] || iv[0] >= iv[3] || iv[1] <= iv[2]) {
      set_error_msg("kpmdos_batch: request " + std::to_string(r) + " has an invalid interval");
      return -1;
    }
  }
  const bool f32 = prec == EVSL_PREC_MIXED;
  const size_t vs = f32 ? 4 : 8;
  // distinct matrices, and FP32 values, on the device
  std::vector<std::unique_ptr<BatchMatrix>> mat;
  std::map<const csrMat*, BatchMatrix*> by_ptr;
  std::vector<BatchValues> values;
  std::vector<BatchRequest> req(nreq);
  Places mp;
  for (int r = 0; r < nreq; ++r) {
    const csrMat* A = mats[r];
    auto it = by_ptr.find(A);
    if (it == by_ptr.end()) {
      auto m = std::make_unique<BatchMatrix>();
      m->host = A;
      m->n = A->nrows;
      m->nnz = A->ia[A->nrows];
      m->ia_at = mp.take((size_t)(m->n + 1) * sizeof(int));
      m->ja_at = mp.take((size_t)m->nnz * sizeof(int));
      m->a64_at = mp.take((size_t)m->nnz * sizeof(double));
      bool full = true;
      for (int i = 0; i < m->n && full; ++i) {
        bool has = false;
        for (int k = A->ia[i]; k < A->ia[i + 1]; ++k)
          if (A->ja[k] == i) {
            has = true;
            break;
          }
        full = has;
      }
      m->full_diag = full;
      m->regular = regular_rows(m->n, A->ia, A->ja);
      it = by_ptr.emplace(A, m.get()).first;
      mat.push_back(std::move(m));
    }
    BatchRequest& q = req[r];
    q.mat = it->second;
    q.intv = intvs + 4 * r;
    q.seed = seeds ? seeds[r] : (unsigned long long)r;
    q.ctr = (q.intv[3] + q.intv[2]) / 2.0;
    q.wid = (q.intv[3] - q.intv[2]) / 2.0;
    q.t0 = 1.0 / q.wid;
    q.t = 2.0 / q.wid;
    q.cc = q.ctr;
    q.raw.assign(Mdeg + 1, 0.0);
    if (f32 && q.mat->nnz > 0) {
      BatchValues v;
      v.mat = q.mat;
      if (q.mat->full_diag) {
        // as the mixed filter: round (A - ctr I) * 2^-s, not A, to FP32
        v.ctr = q.ctr;
        v.scale = std::ldexp(1.0, -(int)std::lround(std::log2(q.wid)));
        q.t0 /= v.scale;
        q.t /= v.scale;
        q.cc = 0.0;
      }
      for (size_t i = 0; i < values.size() && q.a32 < 0; ++i)
        if (values[i].mat == v.mat && values[i].ctr == v.ctr && values[i].scale == v.scale)
          q.a32 = (int)i;
      if (q.a32 < 0) {
        v.at = mp.take((size_t)q.mat->nnz * sizeof(float));
        q.a32 = (int)values.size();
        values.push_back(v);
      }
    }
  }
  DevBuf md;
  EVSL_HIP(md.alloc(mp.end));
  for (auto& m : mat) {
    char* base = md.as<char>();
    m->ia = reinterpret_cast<const int*>(base + m->ia_at);
    m->ja = reinterpret_cast<const int*>(base + m->ja_at);
    m->a64 = reinterpret_cast<const double*>(base + m->a64_at);
    EVSL_HIP(hipMemcpy(base + m->ia_at, m->host->ia, (size_t)(m->n + 1) * sizeof(int),
                       hipMemcpyHostToDevice));
    if (m->nnz == 0) continue;
    EVSL_HIP(hipMemcpy(base + m->ja_at, m->host->ja, (size_t)m->nnz * sizeof(int),
                       hipMemcpyHostToDevice));
    EVSL_HIP(hipMemcpy(base + m->a64_at, m->host->a, (size_t)m->nnz * sizeof(double),
                       hipMemcpyHostToDevice));
  }
  for (auto& v : values) {
    float* a32 = reinterpret_cast<float*>(md.as<char>() + v.at);
    if (v.scale != 0.0)
      EVSL_HIP(evsl_dev::shift_scale_f32(v.mat->view(), v.ctr, v.scale, a32, c.stream));
    else
      EVSL_HIP(evsl_dev::f64_to_f32(v.mat->nnz, v.mat->a64, a32, c.stream));
  }
  DevBuf work;
  std::vector<char> up;
  std::vector<double> hdots;
  // the requests whose column blocks start at one width share their launches
  for (int width : {32, 16, 8}) {
    std::vector<BatchRequest*> reqs;
    for (auto& q : req)
      if (evsl_dev::kpm_max_width(q.mat->n, !f32 && q.mat->regular) == width) reqs.push_back(&q);
    const int nr = (int)reqs.size();
    int done = nr ? 0 : nvec;
    while (done < nvec) {
      int B = width;
      while (B > nvec - done) B >>= 1;
      const int V = evsl_dev::cheb_spmm_vec(B, f32, evsl_dev::kKpm);
      const int R = evsl_dev::cheb_spmm_rows(B, f32, evsl_dev::kKpm);
      if (V <= 0 || R <= 0) return EVSL_ERR_ARG;
      const int lanes = B / V / R;
      size_t pv = 0;
      int maxn = 0, total = 0;
      std::vector<int> nblk(nr), G(nr), owner, owner1, first1(nr), owner2;
      for (int r = 0; r < nr; ++r) {
        BatchMatrix& m = *reqs[r]->mat;
        nblk[r] = (int)(m.row_blocks(lanes).size() / 2) - 1;
        G[r] = evsl_dev::sum_levels_blocks(nblk[r], B);
        pv = std::max(pv, (size_t)nblk[r] * B);
        maxn = std::max(maxn, m.n);
        owner.insert(owner.end(), nblk[r], r);
        first1[r] = (int)owner1.size();
        owner1.insert(owner1.end(), G[r], r);
        if (G[r] > 1) owner2.push_back(r);
      }
      const int nd = std::max(1, std::min(evsl_dev::kpm_sum_degrees(pv), Mdeg));
      // what the host fills in comes first and goes over in one copy
      Places p;
      const size_t tab_at = p.take(nr * sizeof(evsl_dev::KpmGroupEntry));
      const size_t sums_at = p.take(nr * sizeof(evsl_dev::KpmSumEntry));
      const size_t start_at = p.take(nr * sizeof(evsl_dev::KpmStartEntry));
      const size_t owner_at = p.take(owner.size() * sizeof(int));
      const size_t owner1_at = p.take(owner1.size() * sizeof(int));
      const size_t first1_at = p.take(first1.size() * sizeof(int));
      const size_t owner2_at = p.take(owner2.size() * sizeof(int));
      std::map<BatchMatrix*, size_t> rbp_at;
      for (int r = 0; r < nr; ++r)
        if (!rbp_at.count(reqs[r]->mat))
          rbp_at[reqs[r]->mat] = p.take(reqs[r]->mat->row_blocks(lanes).size() * sizeof(int));
      const size_t up_bytes = p.end, dots1 = (size_t)(Mdeg + 1) * B;
      const size_t dots_at = p.take(nr * dots1 * sizeof(double));
      struct At {
        size_t x0, ring, part, scratch, npart, nrm2;
      };
      std::vector<At> at(nr);
      for (int r = 0; r < nr; ++r) {
        const size_t n = reqs[r]->mat->n, nb = n * B;
        at[r].x0 = p.take(nb * vs);
        at[r].ring = p.take(3 * nb * vs);
        at[r].part = p.take((size_t)nd * nblk[r] * B * sizeof(double));
        at[r].scratch = p.take(G[r] > 1 ? (size_t)nd * G[r] * B * sizeof(double) : 0);
        at[r].npart = p.take((size_t)evsl_dev::kpm_start_blocks(n, B) * B * sizeof(double));
        at[r].nrm2 = p.take(B * sizeof(double));
      }
      EVSL_HIP(work.alloc(p.end));
      char* d = work.as<char>();
      up.assign(up_bytes, 0);
      auto* tab = reinterpret_cast<evsl_dev::KpmGroupEntry*>(up.data() + tab_at);
      auto* sums = reinterpret_cast<evsl_dev::KpmSumEntry*>(up.data() + sums_at);
      auto* start = reinterpret_cast<evsl_dev::KpmStartEntry*>(up.data() + start_at);
      for (int r = 0; r < nr; ++r) {
        BatchRequest& q = *reqs[r];
        BatchMatrix& m = *q.mat;
        // start block: the kpmdos_ex vectors of this request's seed, unit columns
        evsl_dev::KpmStartEntry& b = start[r];
        b.x0 = d + at[r].x0;
        b.part = reinterpret_cast<double*>(d + at[r].npart);
        b.nrm2 = reinterpret_cast<double*>(d + at[r].nrm2);
        b.seed = q.seed;
        b.n = m.n;
        b.g = evsl_dev::kpm_start_blocks(m.n, B);
        evsl_dev::KpmGroupEntry& e = tab[r];
        e.ia = m.ia;
        e.ja = m.ja;
        e.a = m.a64;
        if (f32) e.a = q.a32 < 0 ? nullptr : md.as<char>() + values[q.a32].at;
        e.rbp = reinterpret_cast<const int*>(d + rbp_at[q.mat]);
        e.x0 = b.x0;
        e.ring = d + at[r].ring;
        e.part = reinterpret_cast<double*>(d + at[r].part);
        e.t0 = q.t0;
        e.t = q.t;
        e.cc = q.cc;
        e.n = m.n;
        e.blk0 = total;
        e.k0 = 0;
        e.part_step = nblk[r] * B;
        total += nblk[r];
        evsl_dev::KpmSumEntry& s = sums[r];
        s.part = e.part;
        s.scratch = G[r] > 1 ? reinterpret_cast<double*>(d + at[r].scratch) : nullptr;
        s.dots = reinterpret_cast<double*>(d + dots_at) + r * dots1;
        s.nblk = nblk[r];
        s.G = G[r];
        s.k0 = 0;
        s.pad = 0;
      }
      auto fill = [&](size_t to, const std::vector<int>& v) {
        if (!v.empty()) std::memcpy(up.data() + to, v.data(), v.size() * sizeof(int));
      };
      fill(owner_at, owner);
      fill(owner1_at, owner1);
      fill(first1_at, first1);
      fill(owner2_at, owner2);
      for (auto& t : rbp_at) fill(t.second, t.first->row_blocks(lanes));
      EVSL_HIP(hipMemcpy(d, up.data(), up_bytes, hipMemcpyHostToDevice));
      EVSL_HIP(evsl_dev::kpm_group_start(
          f32, B, reinterpret_cast<const evsl_dev::KpmStartEntry*>(d + start_at), nr, maxn,
          vec_kind == EVSL_VEC_RADEMACHER ? 0 : 1, done, c.stream));
      double step_bytes = 0.0;
      for (int r = 0; r < nr; ++r)
        step_bytes += (double)reqs[r]->mat->nnz * (vs + 4) + 4.0 * (reqs[r]->mat->n + 1) +
                      4.0 * reqs[r]->mat->n * B * vs;
      auto ints = [&](size_t from) { return reinterpret_cast<const int*>(d + from); };
      for (int k = 0; k < Mdeg; ++k) {
        EVSL_HIP(evsl_dev::kpm_group_step(
            f32, B, reinterpret_cast<const evsl_dev::KpmGroupEntry*>(d + tab_at), ints(owner_at),
            total, k, k % nd, c.stream));
        if ((k + 1) % nd == 0 || k + 1 == Mdeg) {
          const int have = k % nd + 1;
          EVSL_HIP(evsl_dev::kpm_group_sums(
              B, reinterpret_cast<const evsl_dev::KpmSumEntry*>(d + sums_at), k + 1 - have,
              have, ints(owner1_at), ints(first1_at), (int)owner1.size(), ints(owner2_at),
              (int)owner2.size(), c.stream));
        }
        c.astats.filter_bytes += step_bytes;
      }
      c.astats.n_filter_steps += Mdeg;
      c.astats.n_filter_cols += (size_t)Mdeg * B * nr;
      hdots.resize(nr * dots1);
      EVSL_HIP(hipMemcpy(hdots.data(), d + dots_at, hdots.size() * sizeof(double),
                         hipMemcpyDeviceToHost));
      for (int r = 0; r < nr; ++r)
        kpm_add_dots(Mdeg, B, hdots.data() + r * dots1, reqs[r]->raw.data());
      done += B;
    }
  }
  for (int r = 0; r < nreq; ++r)
    kpm_moments(Mdeg, damping, nvec, req[r].intv, req[r].mat->n, req[r].raw.data(),
                mu + (size_t)r * (Mdeg + 1), ecnt + r);
  return 0;
}

}  // extern "C"
