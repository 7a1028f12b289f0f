// Small row helpers of the block's host path: left padding, the decay buffer, and the ordering of
// one stream after another.
#include <math.h>

#include "hdcm_common.h"

using namespace hdcm;

namespace {

constexpr int kThreads = 256;

// dst[b, i] = i < pad ? 0 : src[b, i - pad], rows of G 16-byte groups.  One thread per group:
// the zero fill and the strided copy of a padded batch in one launch (2 x 3001 rows of 768 bf16:
// 14 us as a fill and a copy).
__global__ __launch_bounds__(kThreads) void pad_rows_kernel(const char* __restrict__ src, int64_t s_bs, int64_t s_rs,
                                                            char* __restrict__ dst, int64_t rows, int L, int pad,
                                                            int G) {
  const int64_t n = rows * G;
  const int P = L + pad;
  for (int64_t k = (int64_t)blockIdx.x * kThreads + threadIdx.x; k < n; k += (int64_t)gridDim.x * kThreads) {
    const int64_t row = k / G;
    const int g = (int)(k - row * G);
    const int64_t b = row / P;
    const int i = (int)(row - b * P);
    const uint4 v = i < pad ? make_uint4(0, 0, 0, 0) : ldg16(src + b * s_bs + (int64_t)(i - pad) * s_rs + 16 * g);
    *reinterpret_cast<uint4*>(dst + row * 16 * G + 16 * g) = v;
  }
}

// gamma = exp(-softplus(decay_log)), each step rounded to T as the tensor operations round it.
template <typename T>
__global__ __launch_bounds__(kThreads) void gamma_kernel(const T* __restrict__ decay_log, T* __restrict__ gamma, int H) {
  const int h = blockIdx.x * kThreads + threadIdx.x;
  if (h >= H) return;
  const float x = to_f<T>(decay_log[h]);
  const float sp = rnd<T>(x > 20.0f ? x : log1pf(expf(x)));
  gamma[h] = from_f<T>(expf(-sp));
}

}  // namespace

extern "C" int hdcm_pad_rows_fwd(const void* src, int64_t src_batch_stride, int64_t src_row_stride, void* dst, int64_t B,
                                 int64_t L, int64_t pad, int64_t D, int dtype, void* stream) {
  HDCM_CHECK_ARG(dtype == HDCM_F32 || dtype == HDCM_BF16, HDCM_EUNSUPPORTED);
  HDCM_CHECK_ARG(B >= 0 && L >= 0 && pad >= 0 && D > 0, HDCM_EINVAL);
  HDCM_CHECK_ARG(L + pad < (int64_t)1 << 30 && D < (int64_t)1 << 30, HDCM_EUNSUPPORTED);
  if (B == 0 || L + pad == 0) return HDCM_OK;
  HDCM_CHECK_ARG((src || L == 0) && dst && (L <= 1 || src_row_stride >= D), HDCM_EINVAL);
  const int esz = hdcm_elt_size(dtype), E = 16 / esz;
  HDCM_CHECK_ARG(D % E == 0 && src_batch_stride % E == 0 && src_row_stride % E == 0 && hdcm_aligned16(src) &&
                     hdcm_aligned16(dst),
                 HDCM_EALIGN);
  const int64_t rows = B * (L + pad), G = D / E;
  const int64_t blocks = (rows * G + kThreads - 1) / kThreads;
  HDCM_LAUNCH(pad_rows_kernel, dim3((unsigned)(blocks < 8192 ? blocks : 8192)), dim3(kThreads), 0, (hipStream_t)stream,
              (const char*)src, src_batch_stride * esz, src_row_stride * esz, (char*)dst, rows, (int)L, (int)pad, (int)G);
  return hdcm_launch_status();
}

extern "C" int hdcm_gamma_fwd(const void* decay_log, void* gamma, int64_t H, int dtype, void* stream) {
  HDCM_CHECK_ARG(dtype == HDCM_F32 || dtype == HDCM_BF16, HDCM_EUNSUPPORTED);
  HDCM_CHECK_ARG(H >= 0 && H < (int64_t)1 << 30 && ((decay_log && gamma) || H == 0), HDCM_EINVAL);
  if (H == 0) return HDCM_OK;
  const dim3 grid((unsigned)((H + kThreads - 1) / kThreads));
  if (dtype == HDCM_F32)
    HDCM_LAUNCH((gamma_kernel<float>), grid, dim3(kThreads), 0, (hipStream_t)stream, (const float*)decay_log,
                (float*)gamma, (int)H);
  else
    HDCM_LAUNCH((gamma_kernel<bf16_t>), grid, dim3(kThreads), 0, (hipStream_t)stream, (const bf16_t*)decay_log,
                (bf16_t*)gamma, (int)H);
  return hdcm_launch_status();
}

// An event of the call's own, on the streams' device: a wait holds what it needs of the event, which is given
// back here (nothing is kept per thread, and a captured event is never recorded again outside its capture).
extern "C" int hdcm_stream_after(void* stream, void* after, int device) {
  if (stream == after) return HDCM_OK;
  HDCM_CHECK_ARG(device >= 0, HDCM_EINVAL);
  int current = device;
  if (hipGetDevice(&current) != hipSuccess || (current != device && hipSetDevice(device) != hipSuccess)) return HDCM_ELAUNCH;
  hipEvent_t e = nullptr;
  bool ok = hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
  if (ok) {
    ok = hipEventRecord(e, (hipStream_t)after) == hipSuccess && hipStreamWaitEvent((hipStream_t)stream, e, 0) == hipSuccess;
    (void)hipEventDestroy(e);
  }
  if (current != device) (void)hipSetDevice(current);
  return ok ? HDCM_OK : HDCM_ELAUNCH;
}
