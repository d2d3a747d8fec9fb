// series.cpp -- host side of the series launches (series.hip): when a filter
// runs as one, the launches' memory, and how a failed one is noticed.
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <vector>

#include "internal.h"

namespace evsl {

// Row-mask matrices of at most 65,536 rows (two a lane) whose rows are paired.
// Eight columns run side by side, an XCD each, and further ones take turns; by
// launches a step takes (us; 8 / 16 / 24 / 32 columns, FP64) 3.5 / 4.1 / 4.8 /
// 4.7 on a 100 x 97 grid, 5.2 / 5.8 / 8.1 / 8.1 on 31 x 32 x 33 and 5.6 / 7.9 /
// 14.2 / 14.4 on 40^3, as series 0.8 / 1.6 / 2.3 / 3.1, 1.4 / 2.5 / 3.7 / 4.9 and
// 2.3 / 4.5 / 6.7 / 9.0; FP32 likewise (40^3: 4.5 / 6.0 / 8.8 / 8.8 against 2.0 /
// 3.9 / 5.9 / 7.8).  So any number of columns does.  Larger matrices are left to
// the launches, which use all XCDs for one column.  Eight degrees pay for the
// launch.  A forced lane layout asks for the CSR kernel, whose launches the blocks
// of any width then are.
bool series_fits(const FilterOp& op, int ncols, int deg) {
  const SeriesState& s = ctx().series;
  if (s.off || s.limit == 0 || !op.A.rmask || !op.A.pairs) return false;
  if (op.A.tune && evsl_dev::spmm_tuner_any_forced(op.A.tune, op.f32, evsl_dev::kCheb)) return false;
  return deg >= 8 && series_size(op.A.n, ncols) &&
         std::max(op.A.nneg, op.A.npair - op.A.nneg) <= evsl_dev::kSeriesMaxHalf;
}

bool series_size(int n, int ncols) {
  return ncols <= SeriesState::kSlots / 2 * evsl_dev::kSeriesMaxJobs &&
         evsl_dev::series_rows_per_lane(n) <= evsl_dev::kSeriesMaxRows;
}

namespace {

constexpr size_t kSetWords = (size_t)evsl_dev::kSeriesXcds * evsl_dev::kSeriesStride;

// memory of the series launches, made on the first one
int ensure_series() {
  Context& c = ctx();
  SeriesState& s = c.series;
  if (!s.status) {
    EVSL_HIP(s.words.alloc(SeriesState::kSets * kSetWords * sizeof(unsigned)));
    const size_t words = (size_t)SeriesState::kSlots * (1 + evsl_dev::kSeriesMaxJobs);
    EVSL_HIP(hipHostMalloc((void**)&s.status, words * sizeof(unsigned), hipHostMallocDefault));
    EVSL_HIP(hipHostGetDevicePointer((void**)&s.status_d, s.status, 0));
    std::fill(s.status, s.status + words, 0u);
    s.id = 0;
  }
  return 0;
}

// reads the outcome of the pending launches, which have ended
void collect() {
  SeriesState& s = ctx().series;
  for (size_t i = 0; i < s.pending.size(); ++i) {
    const volatile unsigned* st = s.status + i * (1 + evsl_dev::kSeriesMaxJobs);
    bool bad = st[0] == s.pending[i].id;
    for (int j = 0; j < s.pending[i].njobs; ++j) bad = bad || st[1 + j] != s.pending[i].id;
    s.failures += bad;
    s.failed = s.failed || bad;
  }
  s.pending.clear();
  s.off = s.off || s.failed;
}

}  // namespace

int series_launch(const std::vector<SeriesCol>& cols) {
  Context& c = ctx();
  SeriesState& s = c.series;
  if (int e = ensure_series()) return e;
  for (size_t j0 = 0; j0 < cols.size(); j0 += evsl_dev::kSeriesMaxJobs) {
    if ((int)s.pending.size() == SeriesState::kSlots) {  // many matrices, each on its own
      EVSL_HIP(hipStreamSynchronize(c.stream));
      collect();
    }
    // each launch has its own counters, cleared kSets launches at a time
    if (s.id % SeriesState::kSets == 0)
      EVSL_HIP(evsl_dev::fill_u32(SeriesState::kSets * kSetWords, 0u, s.words.as<unsigned>(),
                                  c.stream));
    evsl_dev::SeriesArgs a{};
    a.njobs = (int)std::min((size_t)evsl_dev::kSeriesMaxJobs, cols.size() - j0);
    a.parts = evsl_dev::kSeriesParts;
    a.grid = s.workgroups;
    a.limit = (unsigned)s.limit;
    a.words = s.words.as<unsigned>() + (size_t)(s.id % SeriesState::kSets) * kSetWords;
    a.id = ++s.id;
    a.status = s.status_d + s.pending.size() * (1 + evsl_dev::kSeriesMaxJobs);
    // rings and tags: a cell's tag is one that no earlier launch has stored
    const bool f32 = cols[j0].op->f32;
    size_t cells = 0;
    int deg = 0;
    for (int j = 0; j < a.njobs; ++j) {
      cells += (size_t)2 * cols[j0 + j].op->A.n;
      deg = std::max(deg, cols[j0 + j].deg);
    }
    const size_t bytes = cells * evsl_dev::series_cell(f32);
    const bool grow = s.ring.bytes < bytes;
    if (grow) EVSL_HIP(s.ring.alloc(bytes));
    if (grow || s.tag > ~0u - (unsigned)deg - 2u) {
      EVSL_HIP(evsl_dev::fill_u32(s.ring.bytes / sizeof(unsigned), 0u, s.ring.as<unsigned>(),
                                  c.stream));
      s.tag = 0;
    }
    a.tag = s.tag + 1;
    s.tag += (unsigned)deg + 1;
    char* ring = s.ring.as<char>();
    int half = 0, row = 0, rpl = 1;
    for (int j = 0; j < a.njobs; ++j) {
      const SeriesCol& col = cols[j0 + j];
      const evsl_dev::Csr& A = col.op->A;
      evsl_dev::SeriesJob& q = a.job[j];
      q.in = col.in;
      q.out = col.out;
      q.mu = col.mu;
      q.rmask = A.rmask;
      q.dg = col.op->f32 ? (const void*)A.dg32 : (const void*)A.dg64;
      q.ring = ring;
      ring += (size_t)2 * A.n * evsl_dev::series_cell(f32);
      q.pairs = A.pairs;
      q.t1 = col.op->t1;
      q.t2 = col.op->t2;
      q.cc = col.op->cc;
      q.n = A.n;
      q.deg = col.deg;
      q.mu_step = col.mu_step;
      q.mbytes = A.mbytes;
      half = std::max(half, std::max(A.nneg, A.npair - A.nneg));
      row = std::max(row, A.mrow);
      rpl = std::max(rpl, evsl_dev::series_rows_per_lane(A.n));
      c.astats.filter_bytes += A.n * (A.mbytes + (col.op->f32 ? 4.0 : 8.0)) * col.deg;
      c.astats.n_filter_steps += col.deg;
      c.astats.n_filter_cols += col.deg;
    }
    EVSL_HIP(evsl_dev::cheb_series(f32, a, half, row, rpl, c.stream));
    s.pending.push_back({a.id, a.njobs});
    ++s.launched;
  }
  return 0;
}

bool series_failed() {
  SeriesState& s = ctx().series;
  collect();
  const bool bad = s.failed;
  s.failed = false;
  return bad;
}

}  // namespace evsl
