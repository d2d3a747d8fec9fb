// spmm_mask.hip -- launches of the row-mask step kernel, one object per
// precision (EVSL_MASK_FP32).
#include "spmm_mask.h"

namespace evsl_dev {

#if EVSL_MASK_FP32
using MaskVT = float;
#define EVSL_MASK_ENTRY cheb_spmm_mask_f32
#else
using MaskVT = double;
#define EVSL_MASK_ENTRY cheb_spmm_mask_f64
#endif

hipError_t EVSL_MASK_ENTRY(const Csr& A, int B, Mode mode, const void* xk, const void* xkm1,
                           void* xkp1, void* y, const void* v0, const double* s,
                           const double* mu0, double t, double cc, bool first, int yflush,
                           double* part, hipStream_t st) {
#define EVSL_MASK_CASE(BB, MODE_)                                                             \
  case BB:                                                                                    \
    return launch_mask<MaskVT, BB, mask_layout(sizeof(MaskVT), BB, MODE_) / 10,               \
                       mask_layout(sizeof(MaskVT), BB, MODE_) % 10, MODE_>(                   \
        A, xk, xkm1, xkp1, y, v0, s, mu0, t, cc, first, yflush, part, st);
#define EVSL_MASK_POW2(MODE_) \
  EVSL_MASK_CASE(1, MODE_)    \
  EVSL_MASK_CASE(2, MODE_)    \
  EVSL_MASK_CASE(4, MODE_)    \
  EVSL_MASK_CASE(8, MODE_)    \
  EVSL_MASK_CASE(16, MODE_)   \
  EVSL_MASK_CASE(32, MODE_)
#define EVSL_MASK_ALL(MODE_) \
  EVSL_MASK_POW2(MODE_)      \
  EVSL_MASK_CASE(3, MODE_)   \
  EVSL_MASK_CASE(5, MODE_)   \
  EVSL_MASK_CASE(6, MODE_)   \
  EVSL_MASK_CASE(7, MODE_)
  switch (mode) {
    case kCheb:
      switch (B) { EVSL_MASK_ALL(kCheb) default: break; }
      break;
    case kRes:
      switch (B) { EVSL_MASK_ALL(kRes) default: break; }
      break;
#if !EVSL_MASK_FP32
    case kPlain:
      switch (B) { EVSL_MASK_ALL(kPlain) default: break; }
      break;
    case kKpm:
      switch (B) { EVSL_MASK_POW2(kKpm) default: break; }
      break;
#endif
    default:
      break;
  }
  return hipErrorInvalidValue;
}

}  // namespace evsl_dev
