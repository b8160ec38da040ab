// mw3_step_f64.hip -- the step kernels of mw3_step.h for FP64.
#include "mw3_step.h"

namespace mw3 {

hipError_t step_build_f64(Ctx* c) { return step::build<double>(c); }

hipError_t step_update_f64(Ctx* c, const step::UpArgs& a, int nk1, int cpl, int aux, int mode) {
  return step::update<double>(c, a, nk1, cpl, aux, mode);
}

hipError_t step_rad_rr(Ctx* c, const step::RrArgs& a) {
  switch (c->rr_np) {
    case 1: step::launch_rr<1>(c, a); break;
    case 2: step::launch_rr<2>(c, a); break;
    case 3: step::launch_rr<3>(c, a); break;
    case 4: step::launch_rr<4>(c, a); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace mw3
