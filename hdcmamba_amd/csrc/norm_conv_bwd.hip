// Backward of the fused LayerNorm + causal depthwise conv (width 4) for gfx950.
//
// Forward (norm_conv_kernels.h; hdcmamba/model.py:22-72): xh[t] = (x[t] - mu_t) * r_t,
// u[t] = xh[t] * g + b for t >= 0 and u[t] = b for t < 0 (the LayerNorm of a zero row),
// out[t] = sum_k w_k u[t-3+k] + cb.  With go = dL/dout this computes the exact gradients
// of that forward (hdcmamba/model.py:74-166 is the reference's backward, which drops the
// b terms of dw and db and works from bf16-rounded statistics; see the oracle):
//   gu[t]  = sum_k w_k go[t+3-k]                     (t >= 0; go past L is 0)
//   dx[t]  = r_t (gh - mean(gh) - xh[t] mean(gh xh[t])),  gh = gu[t] g
//   dcb    = sum_t go[t] = G
//   dw_k   = sum_t go[t] u[t-3+k] = g X_k + b G,     X_k = sum_{t>=0} xh[t] go[t+3-k]
//   dg     = sum_{t>=0} gu[t] xh[t] = sum_k w_k X_k
//   db     = sum_{t, k} w_k go[t] = G sum_k w_k      (rows t < 0 included)
// so a column's parameter gradients follow from five sums over the rows, X_0 .. X_3 and G, taken
// by the pass that computes dx: x and go are read once.
//
// norm_conv_bwd_kernel: WPR waves (1, 2 or 4) walk a run of rows, lanes owning 16-byte column
// groups (as the forward) with their five sums and four taps in registers; rows come through rings (each go
// row unpacked once, nothing moved between steps), the next ones in flight.  Eight columns per lane leave room for two waves per SIMD, so rows take one wave
// up to 512 columns, two up to 1024 and four beyond (row sums then finish across the waves in
// LDS), up to the forward's 768 groups per row.  Runs are sized for about 2048 waves.  Each
// workgroup leaves one row of sums [5][D]; norm_conv_bwd_sum_kernel adds them in a fixed order
// (the result does not depend on scheduling) and forms the gradients.
// dx may take the gradient of the residual branch with it (res), in place of an addition of its own (23 us at
// 32768 x 768, bf16).
// Bound: the vector ALU (about 40 operations a value), then HBM (x, go read, dx written; go 3 rows more per
// run).  This kernel alone, bf16 8 x 4095 rows of 1024: 50 us, 4.0 TB/s of that traffic; 60 with three chained
// reductions a row, 56 with one and registers moved every row; fp32 2 x 1024 x 512 18, 20, 17 us.
// The sums' launch adds 8 us there; two passes (dx, then the sums) and three launches were 135 in all.
#include <algorithm>
#include <type_traits>

#include "hdcm_common.h"

using namespace hdcm;

namespace {

constexpr int kWpb = 4;            // waves per workgroup
constexpr int kMinRun = 16;        // fewest rows per run (3 more rows of go are read per run)
constexpr int kTargetWaves = 2048;

template <typename T, int NG, int WPR>
__global__ __launch_bounds__(kWpb* kWave, NG * Vec<T>::N > 8 ? 1 : 2) void norm_conv_bwd_kernel(
    const T* __restrict__ go, int64_t g_bs, int64_t g_rs, const T* __restrict__ x, int64_t x_bs, int64_t x_rs,
    const T* __restrict__ ln_w, const T* __restrict__ conv_w, T* __restrict__ dx, int64_t d_bs, int64_t d_rs,
    const T* __restrict__ res, int64_t r_bs, int64_t r_rs, float* __restrict__ part, int L, int D, float eps, int run_rows, int runs_per_seq, int nruns) {
  constexpr int E = Vec<T>::N;
  constexpr int CW = WPR * kWave;   // column lanes of a row
  constexpr int SL = kWpb / WPR;    // runs of a workgroup
  constexpr int W = NG * CW * E;    // columns those lanes span
  __shared__ __attribute__((aligned(16))) float red[2][kWpb][4];
  __shared__ __attribute__((aligned(16))) float cols[SL > 1 ? 5 * W : 4];
  const int wave = threadIdx.x / kWave, slice = wave / WPR;
  const int lane = threadIdx.x % CW;  // column lane
  const int run = (int)blockIdx.x * SL + slice;
  const int G = D / E;
  // Row totals of four values: within the wave, then (WPR > 1) across the waves through LDS.  Two
  // buffers used in turn: a buffer is written again only two reductions later, after the barrier
  // of the reduction between, which every thread passes after reading it.
  int parity = 0;
  auto row_totals = [&](float4 v) {
    v = make_float4(wave_total(v.x), wave_total(v.y), wave_total(v.z), wave_total(v.w));
    if constexpr (WPR > 1) {
      if ((threadIdx.x & (kWave - 1)) == 0) *reinterpret_cast<float4*>(red[parity][wave]) = v;
      __syncthreads();
      v = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
      for (int k = 0; k < WPR; ++k) {
        const float4 u = *reinterpret_cast<const float4*>(red[parity][slice * WPR + k]);
        v = make_float4(v.x + u.x, v.y + u.y, v.z + u.z, v.w + u.w);
      }
      parity ^= 1;
    }
    return v;
  };

  float X[4][NG][E], Gs[NG][E];
#pragma unroll
  for (int i = 0; i < NG; ++i)
#pragma unroll
    for (int e = 0; e < E; ++e) X[0][i][e] = X[1][i][e] = X[2][i][e] = X[3][i][e] = Gs[i][e] = 0.f;

  // A workgroup past the last run has none (its slices walk zero rows); with WPR > 1 every slice
  // walks run_rows rows, so that all waves meet at the barriers: rows past a slice's end (and a
  // run past the last one, which reads run 0) are taken as zeros and not stored.
  const bool live = run < nruns;
  const int rr = live ? run : 0;
  const int b = rr / runs_per_seq;
  const int t0 = (rr - b * runs_per_seq) * run_rows, t1 = live ? min(L, t0 + run_rows) : t0;
  const float invD = 1.0f / (float)D;
  const T* gb = go + (int64_t)b * g_bs;
  const T* xb = x + (int64_t)b * x_bs;
  T* db = dx + (int64_t)b * d_bs;
  const T* rb = res ? res + (int64_t)b * r_bs : nullptr;
  // raw 16-byte groups of one row; rows past the sequence read its last row (used as zeros)
  auto fetch = [&](uint4 (&v)[NG], const T* base, int64_t rs, int t) {
    const T* row = base + (int64_t)min(t, L - 1) * rs;
#pragma unroll
    for (int i = 0; i < NG; ++i) v[i] = ldg16(row + (int64_t)min(lane + CW * i, G - 1) * E);
  };
  bool own[NG];
#pragma unroll
  for (int i = 0; i < NG; ++i) own[i] = lane + CW * i < G;
  // sum of a row, and of its squared distances from the mean
  auto sum_of = [&](const uint4 (&raw)[NG]) {
    float v[E], s = 0.f;
#pragma unroll
    for (int i = 0; i < NG; ++i) {
      unpack16<T>(raw[i], v);
#pragma unroll
      for (int e = 0; e < E; ++e) s += own[i] ? v[e] : 0.f;
    }
    return s;
  };
  auto squares_of = [&](const uint4 (&raw)[NG], float mean) {
    float v[E], q = 0.f;
#pragma unroll
    for (int i = 0; i < NG; ++i) {
      unpack16<T>(raw[i], v);
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const float c = own[i] ? v[e] - mean : 0.f;
        q += c * c;
      }
    }
    return q;
  };
  // Rings over rows, indexed by the row's number in the run modulo 4 (2 for gr), so that no step moves
  // registers: gf = go[t .. t+3] unpacked, gr = go[t+4], go[t+5] and x = x[t .. t+3] as loaded, the last in
  // flight; r = res[t], res[t+1]
  float gf[4][NG][E];
  uint4 gr[2][NG], xr[4][NG], r[2][NG];
  // go[t] unpacked; columns past the row and rows past the sequence are zeros
  auto unpack_go = [&](float (&f)[NG][E], const uint4 (&raw)[NG], int t) {
#pragma unroll
    for (int i = 0; i < NG; ++i) {
      const bool ok = own[i] && t < L;
      const uint4 v = raw[i];
      unpack16<T>(ok ? v : make_uint4(0, 0, 0, 0), f[i]);
    }
  };
  fetch(xr[0], xb, x_rs, t0);
  fetch(xr[1], xb, x_rs, t0 + 1);
  {
    uint4 g[4][NG];
#pragma unroll
    for (int k = 0; k < 4; ++k) fetch(g[k], gb, g_rs, t0 + k);
    fetch(xr[2], xb, x_rs, t0 + 2);
    fetch(gr[0], gb, g_rs, t0 + 4);
    fetch(xr[3], xb, x_rs, t0 + 3);
    fetch(gr[1], gb, g_rs, t0 + 5);
    if (rb) fetch(r[0], rb, r_rs, t0);
#pragma unroll
    for (int k = 0; k < 4; ++k) unpack_go(gf[k], g[k], t0 + k);
  }
  float gw[NG][E], cw[4][NG][E];
#pragma unroll
  for (int i = 0; i < NG; ++i) {
    const int g = min(lane + CW * i, G - 1);
    float c4[4 * E];
    load16<T>(ln_w + (int64_t)g * E, gw[i]);
#pragma unroll
    for (int k = 0; k < 4; ++k) load16<T>(conv_w + (int64_t)g * E * 4 + k * E, c4 + k * E);
#pragma unroll
    for (int e = 0; e < E; ++e)
#pragma unroll
      for (int k = 0; k < 4; ++k) cw[k][i][e] = c4[4 * e + k];
  }
  // A row's reductions (mean, variance, the two gradient sums) form a chain, so each step takes one
  // round for three rows: the gradient sums of t, the variance of t + 1 and the mean of t + 2.
  float mean, mean1, rstd;
  {
    const float4 m = row_totals(make_float4(sum_of(xr[0]), sum_of(xr[1]), 0.f, 0.f));
    mean = m.x * invD, mean1 = m.y * invD;
    rstd = rsqrtf(row_totals(make_float4(squares_of(xr[0], mean), 0.f, 0.f, 0.f)).x * invD + eps);
  }
  const int t_end = WPR > 1 ? t0 + run_rows : t1;
  // row t, whose number in the run is M modulo 4
  auto step = [&](auto M_, int t) {
    constexpr int M = decltype(M_)::value;
    if (rb) fetch(r[(M + 1) % 2], rb, r_rs, t + 1);
    const bool in_run = t < t1;
    float xv[NG][E], gh[NG][E];
    const float rx = in_run ? rstd : 0.f, in = in_run ? 1.f : 0.f;
    float s1 = 0.f, s2 = 0.f;
#pragma unroll
    for (int i = 0; i < NG; ++i) {
      unpack16<T>(xr[M][i], xv[i]);
#pragma unroll
      for (int e = 0; e < E; ++e) xv[i][e] = own[i] ? (xv[i][e] - mean) * rx : 0.f;  // xh
    }
    fetch(xr[M], xb, x_rs, t + 4);
#pragma unroll
    for (int i = 0; i < NG; ++i)
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const float f0 = gf[M][i][e], f1 = gf[(M + 1) % 4][i][e], f2 = gf[(M + 2) % 4][i][e], f3 = gf[(M + 3) % 4][i][e];
        X[3][i][e] += xv[i][e] * f0;
        X[2][i][e] += xv[i][e] * f1;
        X[1][i][e] += xv[i][e] * f2;
        X[0][i][e] += xv[i][e] * f3;
        Gs[i][e] += in * f0;
        gh[i][e] = (cw[3][i][e] * f0 + cw[2][i][e] * f1 + cw[1][i][e] * f2 + cw[0][i][e] * f3) * gw[i][e];
        s1 += gh[i][e];
        s2 += gh[i][e] * xv[i][e];
      }
    const float4 tot = row_totals(make_float4(s1, s2, squares_of(xr[(M + 1) % 4], mean1), sum_of(xr[(M + 2) % 4])));
    const float m1 = tot.x * invD, m2 = tot.y * invD;
#pragma unroll
    for (int i = 0; i < NG; ++i) {
      float o[E];
#pragma unroll
      for (int e = 0; e < E; ++e) o[e] = rstd * (gh[i][e] - m1 - xv[i][e] * m2);
      if (rb) {
        float rv[E];
        unpack16<T>(r[M % 2][i], rv);
#pragma unroll
        for (int e = 0; e < E; ++e) o[e] += rv[e];
      }
      if (own[i] && in_run) store16<T>(db + (int64_t)t * d_rs + (int64_t)(lane + CW * i) * E, o);
    }
    unpack_go(gf[M], gr[M % 2], t + 4);
    fetch(gr[M % 2], gb, g_rs, t + 6);
    mean = mean1, mean1 = tot.w * invD;
    rstd = rsqrtf(tot.z * invD + eps);
  };
#pragma unroll 1
  for (int t = t0; t < t_end; t += 4) {
    step(std::integral_constant<int, 0>{}, t);
    if (t + 1 < t_end) step(std::integral_constant<int, 1>{}, t + 1);
    if (t + 2 < t_end) step(std::integral_constant<int, 2>{}, t + 2);
    if (t + 3 < t_end) step(std::integral_constant<int, 3>{}, t + 3);
  }

  // this workgroup's sums: part[block][5][D] (X_0 .. X_3, G)
  float* pp = part + (int64_t)blockIdx.x * 5 * D;
  if constexpr (SL > 1) {  // the slices' sums added in LDS in order
    for (int sl = 0; sl < SL; ++sl) {
      if (slice == sl) {
#pragma unroll
        for (int j = 0; j < 5; ++j)
#pragma unroll
          for (int i = 0; i < NG; ++i) {
            float* c = cols + j * W + (lane + CW * i) * E;
#pragma unroll
            for (int e = 0; e < E; ++e) {
              const float v = j < 4 ? X[j < 4 ? j : 0][i][e] : Gs[i][e];
              c[e] = sl == 0 ? v : c[e] + v;
            }
          }
      }
      __syncthreads();
    }
    for (int j = 0; j < 5; ++j)
      for (int i = threadIdx.x; i < D; i += kWpb * kWave) pp[(int64_t)j * D + i] = cols[j * W + i];
  } else {
#pragma unroll
    for (int j = 0; j < 5; ++j)
#pragma unroll
      for (int i = 0; i < NG; ++i)
        if (own[i])
#pragma unroll
          for (int e = 0; e < E; ++e)
            pp[(int64_t)j * D + (lane + CW * i) * E + e] = j < 4 ? X[j < 4 ? j : 0][i][e] : Gs[i][e];
  }
}

// Parameter gradients from the workgroups' sums: 16 columns by 64 slices of partial rows per
// workgroup (64-byte reads, many of them in flight), slices added in order.
constexpr int kSumC = 16, kSumR = 64;
template <typename T>
__global__ __launch_bounds__(kSumC* kSumR) void norm_conv_bwd_sum_kernel(
    const float* __restrict__ part, int nk, int D, const T* __restrict__ ln_w, const T* __restrict__ ln_b,
    const T* __restrict__ conv_w, float* __restrict__ d_ln_w, float* __restrict__ d_ln_b,
    float* __restrict__ d_conv_w, float* __restrict__ d_conv_b) {
  __shared__ float acc[kSumR][5][kSumC + 1];
  const int x = threadIdx.x % kSumC, j = threadIdx.x / kSumC;
  const int c = blockIdx.x * kSumC + x;
  float s[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
  if (c < D) {
#pragma unroll 4
    for (int k = j; k < nk; k += kSumR)
#pragma unroll
      for (int m = 0; m < 5; ++m) s[m] += part[((int64_t)k * 5 + m) * D + c];
  }
#pragma unroll
  for (int m = 0; m < 5; ++m) acc[j][m][x] = s[m];
  __syncthreads();
  // Slice sums of value j, in order.  A thread reads and overwrites its own column acc[.][j][x] only, so
  // nothing is waited for in between (and j = 4 and j = 5 share a wave: a barrier in here would be
  // passed twice by it).
  if (j < 5) {
    float t = 0.f;
    for (int r = 0; r < kSumR; ++r) t += acc[r][j][x];
    acc[0][j][x] = t;
  }
  __syncthreads();
  if (j == 0 && c < D) {
    float w[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) w[k] = to_f<T>(conv_w[(int64_t)c * 4 + k]);
    const float g = to_f<T>(ln_w[c]), b = to_f<T>(ln_b[c]), Gc = acc[0][4][x];
    float dg = 0.f;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      dg += w[k] * acc[0][k][x];
      d_conv_w[(int64_t)c * 4 + k] = g * acc[0][k][x] + b * Gc;
    }
    d_ln_w[c] = dg;
    d_ln_b[c] = Gc * ((w[0] + w[1]) + (w[2] + w[3]));
    d_conv_b[c] = Gc;
  }
}

// Waves per row, rows of a run and the grid of norm_conv_bwd_kernel for rows of D columns.
struct Plan {
  int wpr, run_rows, runs_per_seq, nruns, grid;
};
Plan plan_of(int64_t B, int64_t L, int64_t D) {
  Plan p;
  p.wpr = D <= 512 ? 1 : D <= 1024 ? 2 : 4;
  const int64_t target = kTargetWaves / p.wpr;
  p.run_rows = (int)std::max<int64_t>(kMinRun, (B * L + target - 1) / target);
  p.runs_per_seq = (int)((L + p.run_rows - 1) / p.run_rows);
  p.nruns = (int)(B * p.runs_per_seq);
  const int slices = kWpb / p.wpr;
  p.grid = (p.nruns + slices - 1) / slices;
  return p;
}

template <typename T>
int launch_bwd(const void* go, int64_t g_bs, int64_t g_rs, const void* x, int64_t x_bs, int64_t x_rs,
               const void* ln_w, const void* ln_b, const void* conv_w, void* dx, int64_t d_bs, int64_t d_rs,
               const void* res, int64_t r_bs, int64_t r_rs, float* d_ln_w, float* d_ln_b, float* d_conv_w, float* d_conv_b, void* ws, int64_t B, int64_t L,
               int64_t D, float eps, hipStream_t s) {
  constexpr int E = Vec<T>::N;
  const int G = (int)(D / E);
  const bool rows = B > 0 && L > 0;
  const Plan p = rows ? plan_of(B, L, D) : Plan{1, 0, 0, 0, 0};
  if (rows) {
    bool launched = false;
    const int ng = (G + p.wpr * kWave - 1) / (p.wpr * kWave);
#define HDCM_BWD(N, WPR)                                                                                               \
  if (!launched && p.wpr == WPR && ng <= N) {                                                                          \
    HDCM_LAUNCH((norm_conv_bwd_kernel<T, N, WPR>), dim3((unsigned)p.grid), dim3(kWpb * kWave), 0, s, (const T*)go,     \
                g_bs, g_rs, (const T*)x, x_bs, x_rs, (const T*)ln_w, (const T*)conv_w, (T*)dx, d_bs, d_rs,              \
                (const T*)res, r_bs, r_rs, (float*)ws,                                                                 \
                (int)L, (int)D, eps, p.run_rows, p.runs_per_seq, p.nruns);                                             \
    launched = true;                                                                                                   \
  }
    // bf16 rows have one 16-byte group per lane up to 2048 columns, fp32 rows one or two; wider
    // ones (up to 768 groups: bf16 6144, fp32 3072 columns) up to three
    HDCM_BWD(1, 1)
    if constexpr (sizeof(T) == 4) {
      HDCM_BWD(2, 1)
      HDCM_BWD(2, 2)
    } else {
      HDCM_BWD(1, 2)
      HDCM_BWD(1, 4)
    }
    HDCM_BWD(2, 4)
    HDCM_BWD(3, 4)
#undef HDCM_BWD
    if (!launched) return HDCM_EUNSUPPORTED;
    const int st = hdcm_launch_status();
    if (st) return st;
  }
  HDCM_LAUNCH((norm_conv_bwd_sum_kernel<T>), dim3((unsigned)((D + kSumC - 1) / kSumC)), dim3(kSumC * kSumR), 0, s,
              (const float*)ws, p.grid, (int)D, (const T*)ln_w, (const T*)ln_b, (const T*)conv_w, d_ln_w, d_ln_b,
              d_conv_w, d_conv_b);
  return hdcm_launch_status();
}

}  // namespace

extern "C" size_t hdcm_norm_conv_bwd_workspace_bytes(int64_t B, int64_t L, int64_t D) {
  if (B <= 0 || L <= 0 || D <= 0) return 0;
  // The size callers lay out (8 bytes a row and 7 D floats per 64 rows), kept so that a buffer of it stays
  // enough; the sums take 5 D floats per workgroup, more than that only at many short sequences.
  const size_t laid_out = (size_t)((B * L * sizeof(float2) + 255) / 256) * 256 + (size_t)B * ((L + 63) / 64) * 7 * D * sizeof(float);
  return std::max(laid_out, (size_t)plan_of(B, L, D).grid * 5 * D * sizeof(float));
}

extern "C" int hdcm_norm_conv_bwd_add(const void* grad_out, int64_t g_batch_stride, int64_t g_row_stride,
                                      const void* x, int64_t x_batch_stride, int64_t x_row_stride, const void* ln_w,
                                      const void* ln_b, const void* conv_w, const void* res, int64_t res_batch_stride,
                                      int64_t res_row_stride, void* dx, int64_t dx_batch_stride,
                                      int64_t dx_row_stride, float* d_ln_w, float* d_ln_b, float* d_conv_w,
                                      float* d_conv_b, void* ws, size_t ws_bytes, int64_t B, int64_t L, int64_t D,
                                      float eps, int dtype, void* stream) {
  HDCM_CHECK_ARG(dtype == HDCM_F32 || dtype == HDCM_BF16, HDCM_EUNSUPPORTED);
  HDCM_CHECK_ARG(ln_w && ln_b && conv_w && d_ln_w && d_ln_b && d_conv_w && d_conv_b &&
                     ((grad_out && x && dx) || B == 0 || L == 0),
                 HDCM_EINVAL);
  HDCM_CHECK_ARG(B >= 0 && L >= 0 && D > 0, HDCM_EINVAL);
  const int E = 16 / hdcm_elt_size(dtype);
  HDCM_CHECK_ARG(D % E == 0, HDCM_EALIGN);
  HDCM_CHECK_ARG(D / (16 / hdcm_elt_size(dtype)) <= 768, HDCM_EUNSUPPORTED);  // bf16 6144, fp32 3072 (the forward's)
  HDCM_CHECK_ARG(B <= 65535 && L < (int64_t)1 << 30 && (L + 63) / 64 <= 65535, HDCM_EUNSUPPORTED);
  HDCM_CHECK_ARG(hdcm_aligned16(ln_w) && hdcm_aligned16(ln_b) && hdcm_aligned16(conv_w), HDCM_EALIGN);
  if (B == 0 || L == 0) {  // no rows (strides unused): the parameter gradients are zero
    if (dtype == HDCM_F32)
      return launch_bwd<float>(nullptr, 0, 0, nullptr, 0, 0, ln_w, ln_b, conv_w, nullptr, 0, 0, nullptr, 0, 0, d_ln_w, d_ln_b, d_conv_w,
                               d_conv_b, nullptr, 0, 0, D, eps, (hipStream_t)stream);
    return launch_bwd<bf16_t>(nullptr, 0, 0, nullptr, 0, 0, ln_w, ln_b, conv_w, nullptr, 0, 0, nullptr, 0, 0, d_ln_w, d_ln_b, d_conv_w,
                              d_conv_b, nullptr, 0, 0, D, eps, (hipStream_t)stream);
  }
  HDCM_CHECK_ARG(g_row_stride >= D && x_row_stride >= D && dx_row_stride >= D, HDCM_EINVAL);
  HDCM_CHECK_ARG(g_row_stride % E == 0 && x_row_stride % E == 0 && dx_row_stride % E == 0 && g_batch_stride % E == 0 &&
                     x_batch_stride % E == 0 && dx_batch_stride % E == 0,
                 HDCM_EALIGN);
  HDCM_CHECK_ARG(hdcm_aligned16(grad_out) && hdcm_aligned16(x) && hdcm_aligned16(dx) && hdcm_aligned16(ln_w) &&
                     hdcm_aligned16(ln_b) && hdcm_aligned16(conv_w),
                 HDCM_EALIGN);
  HDCM_CHECK_ARG(!res || res_row_stride >= D, HDCM_EINVAL);
  HDCM_CHECK_ARG(!res || (res_row_stride % E == 0 && res_batch_stride % E == 0 && hdcm_aligned16(res)), HDCM_EALIGN);
  HDCM_CHECK_ARG(ws != nullptr && ws_bytes >= hdcm_norm_conv_bwd_workspace_bytes(B, L, D), HDCM_EWORKSPACE);
  HDCM_CHECK_ARG(((uintptr_t)ws & 255u) == 0, HDCM_EALIGN);
  hipStream_t s = (hipStream_t)stream;
  if (dtype == HDCM_F32)
    return launch_bwd<float>(grad_out, g_batch_stride, g_row_stride, x, x_batch_stride, x_row_stride, ln_w, ln_b,
                             conv_w, dx, dx_batch_stride, dx_row_stride, res, res_batch_stride, res_row_stride, d_ln_w, d_ln_b,
                             d_conv_w, d_conv_b, ws, B, L, D, eps, s);
  return launch_bwd<bf16_t>(grad_out, g_batch_stride, g_row_stride, x, x_batch_stride, x_row_stride, ln_w, ln_b,
                            conv_w, dx, dx_batch_stride, dx_row_stride, res, res_batch_stride, res_row_stride, d_ln_w, d_ln_b,
                            d_conv_w, d_conv_b, ws, B, L, D, eps, s);
}

extern "C" int hdcm_norm_conv_bwd(const void* grad_out, int64_t g_batch_stride, int64_t g_row_stride,
                                  const void* x, int64_t x_batch_stride, int64_t x_row_stride, const void* ln_w,
                                  const void* ln_b, const void* conv_w, void* dx, int64_t dx_batch_stride,
                                  int64_t dx_row_stride, float* d_ln_w, float* d_ln_b, float* d_conv_w,
                                  float* d_conv_b, void* ws, size_t ws_bytes, int64_t B, int64_t L, int64_t D,
                                  float eps, int dtype, void* stream) {
  return hdcm_norm_conv_bwd_add(grad_out, g_batch_stride, g_row_stride, x, x_batch_stride, x_row_stride, ln_w, ln_b,
                                conv_w, nullptr, 0, 0, dx, dx_batch_stride, dx_row_stride, d_ln_w, d_ln_b, d_conv_w,
                                d_conv_b, ws, ws_bytes, B, L, D, eps, dtype, stream);
}
