// mw3_step_f32.hip -- the step kernels of mw3_step.h for FP32 operator terms (mixed precision).
#include "mw3_step.h"

namespace mw3 {

hipError_t step_build_f32(Ctx* c) { return step::build<float>(c); }

hipError_t step_update_f32(Ctx* c, const step::UpArgs& a, int nk1, int cpl, int aux, int mode) {
  return step::update<float>(c, a, nk1, cpl, aux, mode);
}

}  // namespace mw3
