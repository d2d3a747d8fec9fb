// series.cpp -- host side of the series launches (series.hip): when a filter
// runs as one, the meeting's memory, and how a failed launch is noticed.
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <vector>

#include "internal.h"

namespace evsl {

// Up to eight columns (an XCD each) of a row-mask matrix of at most 65,536 rows
// (four a lane): there a step takes 1.7 to 3.8 us against 3.3 to 5.6 by
// launches (series.hip), less than the launches' own 3.5 us wherever the rows
// are few, and at least as fast at the upper end in both precisions.  Larger
// matrices are left to the launches, which use all XCDs for one column; more
// columns would take turns on the XCDs.  Eight degrees pay for the launch and
// its meetings' first trip.
bool series_fits(const FilterOp& op, int ncols, int deg) {
  const SeriesState& s = ctx().series;
  if (s.off || s.limit == 0 || !op.A.rmask || !op.A.pairs) return false;
  if (deg < 8 || ncols > 8) return false;
  if (std::max(op.A.nneg, op.A.npair - op.A.nneg) > evsl_dev::kSeriesMaxHalf) return false;
  return evsl_dev::series_rows_per_lane(op.A.n) <= evsl_dev::kSeriesMaxRows;
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

}  // namespace

int series_launch(const std::vector<SeriesCol>& cols) {
  Context& c = ctx();
  SeriesState& s = c.series;
  if (int e = ensure_series()) return e;
  for (size_t j0 = 0; j0 < cols.size(); j0 += evsl_dev::kSeriesMaxJobs) {
    if ((int)s.pending.size() == SeriesState::kSlots) {  // none of the callers comes near
      set_error_msg("series_launch: too many launches before a check");
      return EVSL_ERR_DEVICE;
    }
    // each launch has its own counters, cleared kSets launches at a time
    if (s.id % SeriesState::kSets == 0)
      EVSL_HIP(evsl_dev::fill_u32(SeriesState::kSets * kSetWords, 0u, s.words.as<unsigned>(),
                                  c.stream));
    evsl_dev::SeriesArgs a{};
    a.njobs = (int)std::min((size_t)evsl_dev::kSeriesMaxJobs, cols.size() - j0);
    a.parts = evsl_dev::kSeriesParts;
    a.limit = (unsigned)s.limit;
    a.words = s.words.as<unsigned>() + (size_t)(s.id % SeriesState::kSets) * kSetWords;
    a.id = ++s.id;
    a.status = s.status_d + s.pending.size() * (1 + evsl_dev::kSeriesMaxJobs);
    int half = 0, rpl = 1;
    for (int j = 0; j < a.njobs; ++j) {
      const SeriesCol& col = cols[j0 + j];
      const evsl_dev::Csr& A = col.op->A;
      evsl_dev::SeriesJob& q = a.job[j];
      q.in = col.in;
      q.out = col.out;
      q.mu = col.mu;
      q.rmask = A.rmask;
      q.dg = col.op->f32 ? (const void*)A.dg32 : (const void*)A.dg64;
      q.ring = col.ring;
      q.pairs = A.pairs;
      q.t1 = col.op->t1;
      q.t2 = col.op->t2;
      q.cc = col.op->cc;
      q.n = A.n;
      q.deg = col.deg;
      q.mu_step = col.mu_step;
      q.mbytes = A.mbytes;
      half = std::max(half, std::max(A.nneg, A.npair - A.nneg));
      rpl = std::max(rpl, evsl_dev::series_rows_per_lane(A.n));
      c.astats.filter_bytes += A.n * (A.mbytes + (col.op->f32 ? 4.0 : 8.0)) * col.deg;
      c.astats.n_filter_steps += col.deg;
      c.astats.n_filter_cols += col.deg;
    }
    EVSL_HIP(evsl_dev::cheb_series(cols[j0].op->f32, a, half, rpl, c.stream));
    s.pending.push_back({a.id, a.njobs});
  }
  return 0;
}

bool series_failed() {
  SeriesState& s = ctx().series;
  bool bad = false;
  for (size_t i = 0; i < s.pending.size(); ++i) {
    const volatile unsigned* st = s.status + i * (1 + evsl_dev::kSeriesMaxJobs);
    bad = bad || st[0] == s.pending[i].id;
    for (int j = 0; j < s.pending[i].njobs; ++j) bad = bad || st[1 + j] != s.pending[i].id;
  }
  s.pending.clear();
  s.off = s.off || bad;
  return bad;
}

}  // namespace evsl
