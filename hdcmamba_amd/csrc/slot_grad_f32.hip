// fp32 instantiations of the slot memory's gradient passes (hdcm_slot_grad is in slot_grad.hip).
#include "slot_grad_kernels.h"

int hdcm_slot::grad_launch_f32(const GradCall& g, const SlotPlan& pl, hipStream_t s) {
#define HDCM_GRAD_CASE(HDV) \
  if (pl.HD == HDV) return launch_grad<float, HDV>(g, pl, s);
  HDCM_GRAD_CASE(16) HDCM_GRAD_CASE(32) HDCM_GRAD_CASE(48) HDCM_GRAD_CASE(64)
  HDCM_GRAD_CASE(80) HDCM_GRAD_CASE(96) HDCM_GRAD_CASE(112) HDCM_GRAD_CASE(128)
#undef HDCM_GRAD_CASE
  return HDCM_EUNSUPPORTED;
}
