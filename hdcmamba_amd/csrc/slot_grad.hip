// Gradient of the slot memory + GroupNorm + gate: the entry points and the bf16 instantiations
// (the passes are in slot_grad_kernels.h).
#include "slot_grad_kernels.h"

namespace {

size_t align256(size_t n) { return (n + 255) / 256 * 256; }

// workspace: dy [B L, dm], the reverse pass's segment states, the partial column sums
size_t dy_bytes(int64_t B, int64_t L, int64_t dm, int dtype) { return align256((size_t)B * L * dm * hdcm_elt_size(dtype)); }
size_t part_bytes(int64_t B, int64_t dm, const SlotPlan& pl) { return (size_t)B * pl.nseg * 2 * dm * sizeof(float); }

}  // namespace

int hdcm_slot::grad_launch_bf16(const GradCall& g, const SlotPlan& pl, hipStream_t s) {
#define HDCM_GRAD_CASE(HDV) \
  if (pl.HD == HDV) return launch_grad<bf16_t, HDV>(g, pl, s);
  HDCM_GRAD_CASE(16) HDCM_GRAD_CASE(32) HDCM_GRAD_CASE(48) HDCM_GRAD_CASE(64)
  HDCM_GRAD_CASE(80) HDCM_GRAD_CASE(96) HDCM_GRAD_CASE(112) HDCM_GRAD_CASE(128)
#undef HDCM_GRAD_CASE
  return HDCM_EUNSUPPORTED;
}

extern "C" size_t hdcm_slot_grad_workspace_bytes(int64_t B, int64_t L, int64_t dm, int64_t H, int64_t C, int dtype) {
  SlotPlan pl;
  if (slot_plan(B, L, dm, H, C, dtype, &pl) != HDCM_OK) return 0;
  return dy_bytes(B, L, dm, dtype) + align256(slot_ws_bytes(B, H, pl)) + part_bytes(B, dm, pl);
}

extern "C" int hdcm_slot_grad(const void* projs, int64_t proj_row_stride, int64_t q_col, const void* gamma,
                              const void* gn_w, const void* gn_b, float gn_eps, const void* ws_fwd, size_t ws_fwd_bytes,
                              const void* dout, int64_t dout_row_stride, void* dprojs, int64_t dprojs_row_stride,
                              float* dgn_w, float* dgn_b, void* ws, size_t ws_bytes, int64_t B, int64_t L, int64_t dm,
                              int64_t H, int64_t C, int dtype, void* stream) {
  SlotPlan pl;
  int st = slot_plan(B, L, dm, H, C, dtype, &pl);
  if (st) return st;
  const bool empty = B == 0 || L == 0;
  st = check_projs(projs, proj_row_stride, q_col, dm, dtype, empty);
  if (st) return st;
  HDCM_CHECK_ARG(gamma && gn_w && gn_b && dgn_w && dgn_b && ((dout && dprojs) || empty), HDCM_EINVAL);
  const int E = 16 / hdcm_elt_size(dtype);
  HDCM_CHECK_ARG(empty || (dout_row_stride >= dm && dprojs_row_stride >= q_col + 4 * dm), HDCM_EINVAL);
  HDCM_CHECK_ARG(hdcm_aligned16(dout) && hdcm_aligned16(dprojs) &&
                     (empty || (dout_row_stride % E == 0 && dprojs_row_stride % E == 0)),
                 HDCM_EALIGN);
  hipStream_t s = (hipStream_t)stream;
  if (empty)  // no rows: zero parameter gradients
    return hdcm_colsum(nullptr, 0, 0, 2 * (int)dm, 2 * (int)dm, 0, dgn_w, (int)dm, dgn_b, s);
  HDCM_CHECK_ARG(ws_fwd && ws_fwd_bytes >= slot_ws_bytes(B, H, pl) && ws &&
                     ws_bytes >= hdcm_slot_grad_workspace_bytes(B, L, dm, H, C, dtype),
                 HDCM_EWORKSPACE);
  HDCM_CHECK_ARG(hdcm_aligned16(ws_fwd) && hdcm_aligned16(ws), HDCM_EALIGN);
  hdcm_slot::GradCall g;
  g.projs = projs, g.gamma = gamma, g.gn_w = gn_w, g.gn_b = gn_b, g.ws_fwd = ws_fwd, g.dout = dout;
  g.prs = proj_row_stride, g.q_col = q_col, g.dors = dout_row_stride, g.dprs = dprojs_row_stride;
  g.dprojs = dprojs, g.gn_eps = gn_eps, g.dgn_w = dgn_w, g.dgn_b = dgn_b;
  g.dy = ws;
  g.ws_rev = (char*)ws + dy_bytes(B, L, dm, dtype);
  g.part = (float*)((char*)g.ws_rev + align256(slot_ws_bytes(B, H, pl)));
  g.B = B, g.L = L, g.dm = dm, g.H = H, g.C = C;
  return dtype == HDCM_BF16 ? hdcm_slot::grad_launch_bf16(g, pl, s) : hdcm_slot::grad_launch_f32(g, pl, s);
}
