// fp32 instantiations of the LayerNorm + causal conv forward (hdcm_norm_conv_fwd is in norm_conv.hip).
#include "norm_conv_kernels.h"

int hdcm_norm_conv_launch_f32(const void* x, int64_t x_bs, int64_t x_rs, const void* ln_w, const void* ln_b,
                              const void* conv_w, const void* conv_b, void* out, int64_t o_bs, int64_t o_rs, int64_t B,
                              int64_t L, int64_t D, float eps, hipStream_t s) {
  return launch<float>(x, x_bs, x_rs, ln_w, ln_b, conv_w, conv_b, out, o_bs, o_rs, B, L, D, eps, s);
}
