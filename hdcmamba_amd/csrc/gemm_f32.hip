// Tiled fp32 GEMM for gfx950: out[t, o] = sum_k X[t, k] W[o, k] (+ bias[o]) (+ res[t, o]), X [M, K]
// rows, W [N, K] an nn.Linear weight, products and sums in fp32 on v_mfma_f32_16x16x4_f32.
//
// The bound is the fp32 matrix rate (256 flops per clock and CU, 1/16 of bf16's), so the operands'
// way there is cheap and the split decides: a tile that leaves CUs idle costs in full.  A workgroup is 2
// x 2 waves with a tile of 64 or 32 outputs x tokens (tile_choice); 128-wide tiles were never faster.
// Rows of 32 values (128 bytes) go to LDS directly from memory, double-buffered, chunk c of row r at
// c ^ (r & 7), as in gemm.hip.  A lane reads 16 bytes of a row, four consecutive k, and step e of
// four MFMAs takes value e of each lane: an MFMA sums k = e, 4 + e, 8 + e, 12 + e of 16, in A and B alike.
// The MFMAs' sums are folded into a second accumulator every 128 values of K: the error against 64
// bits is 1.4-1.6e-7 at any K, where one running sum (and the library) has 2.1e-7 at K = 256 and
// 5.7e-7 at 2048.
//
// Measured against the library (M x N x K, us): 2048 x 2240 x 512 48 against 72; 256 x 256 x 320 6
// against 83 (it takes one 256-wide tile); 1000 x 4480 x 1024 89 against 99; 8192 x 4480 x 1024 575
// against 602 (131 TFLOP/s of about 157).
#include <algorithm>

#include "gemm_tile.h"
#include "hdcm_common.h"

using namespace hdcm;

namespace {

constexpr int kBK = 32;
constexpr int kChunks = kBK / 4;  // 16-byte chunks per tile row
constexpr int kSub = 4;           // K steps per partial sum
using Tile64 = Tile<2, 2, 2, 2>;
using Tile32 = Tile<2, 2, 1, 1>;

template <class TL>
__global__ __launch_bounds__(TL::threads, 4) void gemm_f32_kernel(
    const float* __restrict__ X, int64_t x_rs, const float* __restrict__ W, int64_t w_rs,
    const float* __restrict__ bias, const float* res, int64_t r_rs, float* out, int64_t o_rs, int M, int N, int K,
    int n_otiles) {
  constexpr int kBO = TL::BO, kBT = TL::BT, NI = TL::ni, NJ = TL::nj;
  // four arrays, so that the loads filling one buffer are known not to alias the reads of the other
  __shared__ uint4 sW0[kBO * kChunks], sW1[kBO * kChunks], sX0[kBT * kChunks], sX1[kBT * kChunks];
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int w = __builtin_amdgcn_readfirstlane(tid / kWave);
  int ot, tt;
  tile_of(n_otiles, ot, tt);
  const int o0 = ot * kBO, t0 = tt * kBT;
  const int nw = min(N - o0, kBO), nx = min(M - t0, kBT);
  // rows past M or N and columns past K read as zeros (range checking)
  const __amdgpu_buffer_rsrc_t wsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(W + (int64_t)o0 * w_rs), (short)0, (int)(((int64_t)(nw - 1) * w_rs + K) * 4), kBufferFlags);
  const __amdgpu_buffer_rsrc_t xsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(X + (int64_t)t0 * x_rs), (short)0, (int)(((int64_t)(nx - 1) * x_rs + K) * 4), kBufferFlags);
  const int jr = lane >> 3, jc = (lane & 7) ^ jr;
  const int wvb = (int)(((int64_t)(w * 8 * TL::WL + jr) * w_rs + jc * 4) * 4);
  const int xvb = (int)(((int64_t)(w * 8 * TL::XL + jr) * x_rs + jc * 4) * 4);
  const int wst = (int)(8 * w_rs * 4), xst = (int)(8 * x_rs * 4);
  auto issue = [&](uint4* dw, uint4* dx, int k0) {
    const bool kin = k0 + jc * 4 < K;
    const unsigned wv = kin ? (unsigned)(wvb + 4 * k0) : 0x80000000u;
    const unsigned xv = kin ? (unsigned)(xvb + 4 * k0) : 0x80000000u;
#pragma unroll
    for (int i = 0; i < TL::WL; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(wsrc, (lds_ptr_t)(dw + 8 * (w * TL::WL + i) * kChunks), 16,
                                               (int)(wv + (unsigned)(i * wst)), 0, 0, 0);
#pragma unroll
    for (int i = 0; i < TL::XL; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xsrc, (lds_ptr_t)(dx + 8 * (w * TL::XL + i) * kChunks), 16,
                                               (int)(xv + (unsigned)(i * xst)), 0, 0, 0);
  };

  const int wo0 = (w % TL::nwo) * NI * 16, wt0 = (w / TL::nwo) * NJ * 16;  // this wave's corner of the tile
  const int l16 = lane & 15, g = lane >> 4;
  f32x4_t acc[NI][NJ], tot[NI][NJ];  // the partial sum, the sums before it
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = tot[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto fold = [&] {
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        tot[i][j] += acc[i][j];
        acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
  };
  auto compute = [&](const uint4* bw, const uint4* bx) {
    f32x4_t fa[2][NI], fb[2][NJ];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int pc = (kk * 4 + g) ^ (l16 & 7);
#pragma unroll
      for (int i = 0; i < NI; ++i) fa[kk][i] = __builtin_bit_cast(f32x4_t, bw[(wo0 + i * 16 + l16) * kChunks + pc]);
#pragma unroll
      for (int j = 0; j < NJ; ++j) fb[kk][j] = __builtin_bit_cast(f32x4_t, bx[(wt0 + j * 16 + l16) * kChunks + pc]);
    }
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
          for (int j = 0; j < NJ; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[kk][i][e], fb[kk][j][e], acc[i][j], 0, 0, 0);
  };

  const int nk = (K + kBK - 1) / kBK;
  issue(sW0, sX0, 0);
  for (int kt = 0; kt < nk; ++kt) {
    const bool odd = kt & 1;
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's loads of tile kt are in LDS
    __syncthreads();                     // everyone's; and tile kt-1's buffer is free again
    if (kt + 1 < nk) issue(odd ? sW0 : sW1, odd ? sX0 : sX1, (kt + 1) * kBK);
    compute(odd ? sW1 : sW0, odd ? sX1 : sX0);
    if (kt % kSub == kSub - 1) fold();
  }
  fold();

  // lane holds out[t][o .. o+3], t = t0 + wt0 + 16 j + l16, o = o0 + wo0 + 16 i + 4 g
  float4 b[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i)
    b[i] = bias ? *reinterpret_cast<const float4*>(bias + min(o0 + wo0 + i * 16 + 4 * g, N - 4))
                : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int t = t0 + wt0 + j * 16 + l16;
    if (t >= M) continue;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int o = o0 + wo0 + i * 16 + 4 * g;
      if (o >= N) continue;
      float4 v = make_float4(tot[i][j][0] + b[i].x, tot[i][j][1] + b[i].y, tot[i][j][2] + b[i].z, tot[i][j][3] + b[i].w);
      if (res) {
        const float4 r = *reinterpret_cast<const float4*>(res + (int64_t)t * r_rs + o);
        v = make_float4(v.x + r.x, v.y + r.y, v.z + r.z, v.w + r.w);
      }
      *reinterpret_cast<float4*>(out + (int64_t)t * o_rs + o) = v;
    }
  }
}

// A workgroup's rows span at most 64 row strides of bytes, addressed with 32-bit offsets.
bool fits32(int64_t row_stride) { return row_stride <= ((int64_t)1 << 30) / (4 * Tile64::BO); }

// Tile width by estimated time per K step in hundredths of a microsecond, fitted to measurements (M x N x
// K, us with 64, with 32): 256 x 1216 x 256 8.2, 6.3; 1000 x 768 x 832 20.4, 17.5; 256 x 4480 x 1024
// 39, 33; 1000 x 1024 x 1152 26.7, 28.9; 2048 x 3264 x 768 89, 105; 8192 x 2240 x 512 154, 187.
int tile_choice(int64_t M, int64_t N) {
  const auto per_cu = [](int64_t tiles) { return (tiles + 255) / 256; };
  const int64_t t64 = 18 + 51 * per_cu(tiles_of<Tile64>(M, N)), t32 = 25 + 15 * per_cu(tiles_of<Tile32>(M, N));
  return t64 <= t32 ? 64 : 32;
}

template <class TL>
void launch_tile(const float* x, int64_t x_rs, const float* w, int64_t w_rs, const float* bias, const float* res,
                 int64_t r_rs, float* out, int64_t o_rs, int64_t M, int64_t N, int64_t K, hipStream_t s) {
  HDCM_LAUNCH((gemm_f32_kernel<TL>), dim3((unsigned)tiles_of<TL>(M, N)), dim3(TL::threads), 0, s, x, x_rs, w, w_rs,
              bias, res, r_rs, out, o_rs, (int)M, (int)N, (int)K, (int)((N + TL::BO - 1) / TL::BO));
}

}  // namespace

// Up to M N K of 4e10 and K of 1152 (d_model 1024's projections).  Beyond that many products the library is
// as fast (M x N x K, us, library and this: 16384 x 3264 x 768 607, 628; 16384 x 4480 x 1024 1103, 1133).  At
// wider K it wins below 2048 rows and gives away little above: 64 x 6336 x 1536 18.5, 22.8; 256 rows 50, 56; 512 x
// 1408 x 1472 25, 33; 512 x 1280 x 1344 22, 30; 1536 x 5312 x 1280 155, 165; 4096 x 6336 x 1536 618, 609.  Within
// the line its time is uneven, and single sizes lie behind it (128 x 4480 x 1024 19, 23; 384 rows 32, 38; 512 x
// 3264 x 768 28, 30) among neighbours ahead (256 rows 35, 31; 1000 x 3264 x 768 64, 56).  A few rows (decode
// steps) stay with it too: 16 x 8576 x 2048 is 21 us against 29.
extern "C" int hdcm_gemm_f32_preferred(int64_t M, int64_t N, int64_t K) {
  return M >= 64 && N > 0 && N % 4 == 0 && K > 0 && K <= 1152 && K % 4 == 0 && M <= (int64_t)40000000000 / K / N;
}

extern "C" int hdcm_gemm_f32_fwd(const float* x, int64_t x_row_stride, const float* w, int64_t w_row_stride,
                                 const float* bias, const float* res, int64_t res_row_stride, float* out,
                                 int64_t out_row_stride, int64_t M, int64_t N, int64_t K, void* stream) {
  HDCM_CHECK_ARG(M >= 0 && N > 0 && K > 0, HDCM_EINVAL);
  HDCM_CHECK_ARG(w != nullptr && ((x && out) || M == 0), HDCM_EINVAL);
  HDCM_CHECK_ARG(w_row_stride >= K && (M == 0 || (x_row_stride >= K && out_row_stride >= N)), HDCM_EINVAL);
  HDCM_CHECK_ARG(!res || M == 0 || res_row_stride >= N, HDCM_EINVAL);
  HDCM_CHECK_ARG(K % 4 == 0 && N % 4 == 0 && x_row_stride % 4 == 0 && w_row_stride % 4 == 0 && out_row_stride % 4 == 0 &&
                     hdcm_aligned16(x) && hdcm_aligned16(w) && hdcm_aligned16(out) && hdcm_aligned16(bias) &&
                     (!res || (res_row_stride % 4 == 0 && hdcm_aligned16(res))),
                 HDCM_EALIGN);
  HDCM_CHECK_ARG(M <= INT32_MAX - 128 && N <= INT32_MAX - 128 && K <= INT32_MAX - 128 && fits32(x_row_stride) &&
                     fits32(w_row_stride) && tiles_of<Tile32>(M, N) <= INT32_MAX / 64,
                 HDCM_EUNSUPPORTED);
  if (M == 0) return HDCM_OK;
  const auto go = tile_choice(M, N) == 64 ? launch_tile<Tile64> : launch_tile<Tile32>;
  go(x, x_row_stride, w, w_row_stride, bias, res, res_row_stride, out, out_row_stride, M, N, K, (hipStream_t)stream);
  return hdcm_launch_status();
}
