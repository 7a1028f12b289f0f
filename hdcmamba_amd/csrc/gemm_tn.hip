// Weight-gradient GEMM for gfx950: out[n, k] = sum_m Y[m, n] X[m, k] over bf16 rows (tokens) m, fp32
// accumulation, one rounding; with it the column sums sum_m Y[m, n] (the bias gradient).
//   dW = dY^T X,  db = sum_rows dY   (autograd of nn.Linear, hdcmamba/model.py:313,320)
//
// The contraction runs over the rows of both operands, so neither has it contiguous.  A workgroup of
// four waves takes a 256 (n) x 128 (k) tile and a range of rows, 32 rows per step through three LDS
// stages filled two steps ahead by direct-to-LDS loads as they lie in memory ([row][column]); the
// MFMA operands are read transposed by ds_read_b64_tr_b16, which hands a lane four consecutive rows
// of one column.  Such a read takes 32 bytes of 16 rows per wave; the 32-byte pair p of row r sits at
// p ^ (r & 7), so that eight rows fall on different banks.  X is the MFMA A operand and Y is B: a lane
// holds four consecutive k of one n, stored as 16 bytes.
//
// Split: the outputs are few (in_proj 3264 x 768: 78 tiles, out_proj 768 x 832: 21) and the rows many,
// so the rows are cut into S ranges; each leaves an fp32 partial tile, and sum_parts_kernel adds them
// in order and rounds.  S is the number with the least estimated time (split_of).  The column sums
// come from the Y fragments of the workgroups of the first k tile (v_dot2_f32_bf16 against ones).
// Bound: LDS.  The transposing reads deliver about half the bytes per clock of ds_read_b128, so a
// wave's tile of 128 x 64 (12 fragments for 32 MFMAs) against 64 x 64 (8 for 16) is worth a third.
// In_proj (with the column sums)
// against the library's product and sum kernels: 32768 x 3264 x 768 193 against 342 us, x 4480 x 1024 362
// against 433, 8192 x 3264 x 768 65 against 108; out_proj: 32768 x 768 x 832 68 against 196 us, 8192 rows 33
// against 48.  Without the XCD-aware order 258, 396 and 87 us at 32768 rows.
#include <algorithm>
#include <type_traits>

#include "hdcm_common.h"

using namespace hdcm;

namespace {

constexpr int kBN = 256, kBK = 128;        // tile
constexpr int kStep = 32;     // rows per step
constexpr int kStages = 3;    // LDS buffers: a step's loads are issued two steps ahead
constexpr int kThreads = 256;
constexpr int kYChunks = kBN / 8, kXChunks = kBK / 8;  // 16-byte chunks of an LDS row
constexpr int kYTile = kStep * kYChunks, kXTile = kStep * kXChunks;
constexpr int kBufferFlags = 0x00020000;   // buffer resource word 3: raw 32-bit dwords
constexpr int kMaxSplit = 32;
typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));

// The workgroup barrier without __syncthreads' wait for every outstanding load (which would drain the
// pipeline of LDS loads): the caller has waited for what it needs, and the compiler keeps memory
// operations on their side of it.
__device__ __forceinline__ void plain_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

__global__ __launch_bounds__(kThreads, 2) void gemm_tn_kernel(const bf16_t* __restrict__ Y, int64_t y_rs,
                                                              const bf16_t* __restrict__ X, int64_t x_rs,
                                                              bf16_t* __restrict__ out, int64_t o_rs,
                                                              float* __restrict__ part, float* __restrict__ csum,
                                                              int M, int N, int K, int n_ntiles, int ntiles, int split_rows) {
  __shared__ uint4 sm[kStages * (kYTile + kXTile)];  // [stage][Y tile, X tile]
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int w = __builtin_amdgcn_readfirstlane(tid / kWave);
  // Workgroup b runs on XCD b % 8 (round-robin dispatch); each XCD takes a contiguous run of (range,
  // tile) pairs, tiles fastest, so that the tiles reading a range's rows share one L2.
  const int T = gridDim.x, bx = blockIdx.x & 7;
  const int idx = bx * (T >> 3) + min(bx, T & 7) + (int)(blockIdx.x >> 3);
  const int sp = idx / ntiles, tile = idx - sp * ntiles;
  const int nt = tile % n_ntiles, kt = tile / n_ntiles;
  const int n0 = nt * kBN, k0 = kt * kBK;
  const int m0 = sp * split_rows, m1 = min(M, m0 + split_rows);
  const int ny = min(N - n0, kBN), nx = min(K - k0, kBK);

  // Loads (1 KB each): instruction i of wave w fills two rows of the Y tile (32 chunks each), from 2 (4 w
  // + i) on, and four of the X tile (16 chunks), from 4 (2 w + i) on; lane j lands in chunk c = j % 32 or
  // j % 16 of its row r, which holds the global pair c / 2 ^ (r & 7).  Chunks past the matrix's columns
  // take an offset past the buffer's end, rows past m1 lie past it: both read zeros.
  const int kOut = (int)0x80000000u;
  int yoff[4], xoff[2];
  const auto column = [](int c, int r) { return 8 * ((((c >> 1) ^ (r & 7)) << 1) | (c & 1)); };
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 2 * (4 * w + i) + (lane >> 5), c = column(lane & 31, r);
    yoff[i] = c < ny ? (int)(((int64_t)r * y_rs + c) * 2) : kOut;
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = 4 * (2 * w + i) + (lane >> 4), c = column(lane & 15, r);
    xoff[i] = c < nx ? (int)(((int64_t)r * x_rs + c) * 2) : kOut;
  }
  // bytes from row m of the tile's first column to the end of row m1 - 1's columns (0 past the range: a
  // fixed count of loads per step)
  auto left = [&](int m, int64_t rs, int cols) {
    const int rows = min(kStep, m1 - m);
    return rows > 0 ? (int)(((int64_t)(rows - 1) * rs + cols) * 2) : 0;
  };
  auto fill = [&](int stage, int m) {
    const __amdgpu_buffer_rsrc_t ysrc = __builtin_amdgcn_make_buffer_rsrc((void*)(Y + (int64_t)m * y_rs + n0), (short)0,
                                                                          left(m, y_rs, ny), kBufferFlags);
    const __amdgpu_buffer_rsrc_t xsrc = __builtin_amdgcn_make_buffer_rsrc((void*)(X + (int64_t)m * x_rs + k0), (short)0,
                                                                          left(m, x_rs, nx), kBufferFlags);
    uint4* d = sm + stage * (kYTile + kXTile);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ysrc, (lds_ptr_t)(d + 64 * (4 * w + i)), 16, yoff[i], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 2; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xsrc, (lds_ptr_t)(d + kYTile + 64 * (2 * w + i)), 16, xoff[i], 0, 0, 0);
  };

  const int wn = w & 1, wk = w >> 1;  // this wave's 128 n x 64 k
  const int l16 = lane & 15, g = lane >> 4;
  f32x4_t acc[4][8];  // [k tile][n tile]
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float cs[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  const bool sums = csum != nullptr && kt == 0 && wk == 0;
  const bf16x2_t ones = __builtin_bit_cast(bf16x2_t, 0x3f803f80u);

  // Fragment of columns c0 .. c0 + 15 (lane x = column), rows 4 g + s and 16 + 4 g + s: lane c of a 16-lane
  // group points at row 4 g + c / 4, columns c0 + 4 (c % 4).  Reads and their wait are one asm block: the
  // compiler cannot tell which of the outstanding LDS loads an LDS read depends on (it waited for
  // all of them, draining the pipeline), while the step's own wait and barrier already order them.
  uint32_t ya[8], xa[4];
  {
    const int r = 4 * g + (l16 >> 2);
    const uint32_t base = (uint32_t)(uintptr_t)(lds_ptr_t)sm + 8 * (l16 & 3);
#pragma unroll
    for (int j = 0; j < 8; ++j) ya[j] = base + r * kBN * 2 + 32 * ((wn * 8 + j) ^ (r & 7));
#pragma unroll
    for (int i = 0; i < 4; ++i) xa[i] = base + kYTile * 16 + r * kBK * 2 + 32 * ((wk * 4 + i) ^ (r & 7));
  }
  auto read4 = [&](auto off, auto hi, const uint32_t* a, Frag<bf16_t>* out) {  // four fragments
    constexpr int kOff = decltype(off)::value, kHi = decltype(hi)::value;
    bf16x4_t f[8];
    asm volatile(
        "ds_read_b64_tr_b16 %0, %8 offset:%12\n\tds_read_b64_tr_b16 %1, %8 offset:%13\n\t"
        "ds_read_b64_tr_b16 %2, %9 offset:%12\n\tds_read_b64_tr_b16 %3, %9 offset:%13\n\t"
        "ds_read_b64_tr_b16 %4, %10 offset:%12\n\tds_read_b64_tr_b16 %5, %10 offset:%13\n\t"
        "ds_read_b64_tr_b16 %6, %11 offset:%12\n\tds_read_b64_tr_b16 %7, %11 offset:%13\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(f[0]), "=&v"(f[1]), "=&v"(f[2]), "=&v"(f[3]), "=&v"(f[4]), "=&v"(f[5]), "=&v"(f[6]), "=&v"(f[7])
        : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "n"(kOff), "n"(kOff + kHi)
        : "memory");
#pragma unroll
    for (int i = 0; i < 4; ++i) out[i].v = __builtin_shufflevector(f[2 * i], f[2 * i + 1], 0, 1, 2, 3, 4, 5, 6, 7);
  };
  auto compute = [&](auto stage) {
    constexpr int kOff = decltype(stage)::value * (kYTile + kXTile) * 16;
    Frag<bf16_t> fx[4], fy[8];
    using Off = std::integral_constant<int, kOff>;
    read4(Off{}, std::integral_constant<int, 16 * kBK * 2>{}, xa, fx);
    read4(Off{}, std::integral_constant<int, 16 * kBN * 2>{}, ya, fy);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = mma(fx[i], fy[j], acc[i][j]);
    read4(Off{}, std::integral_constant<int, 16 * kBN * 2>{}, ya + 4, fy + 4);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 4; j < 8; ++j) acc[i][j] = mma(fx[i], fy[j], acc[i][j]);
    if (sums) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const uint4 u = __builtin_bit_cast(uint4, fy[j].v);
        const unsigned d[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
        for (int e = 0; e < 4; ++e)
          cs[j] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, d[e]), ones, cs[j], false);
      }
    }
  };

  const int steps = (m1 - m0 + kStep - 1) / kStep;
  fill(0, m0);
  fill(1, m0 + kStep);
  for (int t = 0, m = m0; t < steps; t += kStages, m += kStages * kStep) {
    // step u's stage holds it once all but the next step's loads (6 per wave and step) have landed
    // for every wave; the barrier also frees the stage of the step before, filled next
#define HDCM_STEP(U)                                           \
  __builtin_amdgcn_s_waitcnt(0x0F76); /* vmcnt(6) */           \
  plain_barrier();                                             \
  fill((U + 2) % kStages, m + (U + 2) * kStep);                \
  compute(std::integral_constant<int, U>{});                   \
  if (t + U + 1 >= steps) break;
    HDCM_STEP(0)
    HDCM_STEP(1)
    HDCM_STEP(2)
#undef HDCM_STEP
  }

  if (sums) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float t = quad_group_sum(cs[j]);
      const int n = n0 + wn * 128 + j * 16 + l16;
      if (g == 0 && n < N) csum[(int64_t)sp * N + n] = t;
    }
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int n = n0 + wn * 128 + j * 16 + l16;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int k = k0 + wk * 64 + i * 16 + 4 * g;
      if (n < N && k < K) {
        const f32x4_t a = acc[i][j];
        if (part != nullptr)
          *reinterpret_cast<f32x4_t*>(part + ((int64_t)sp * N + n) * K + k) = a;
        else
          *reinterpret_cast<uint2*>(out + (int64_t)n * o_rs + k) = make_uint2(pack_bf16x2(a[0], a[1]), pack_bf16x2(a[2], a[3]));
      }
    }
  }
}

// out = the S partial tiles added in order, rounded; the column sums likewise.  Four columns per thread.
__global__ __launch_bounds__(kThreads) void sum_parts_kernel(const float* __restrict__ part, const float* __restrict__ csum,
                                                             int S, int N, int K, bf16_t* __restrict__ out, int64_t o_rs,
                                                             bf16_t* __restrict__ cout) {
  const int64_t n4 = (int64_t)N * K / 4, id = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (part != nullptr && id < n4) {
    const float4* p = reinterpret_cast<const float4*>(part) + id;
    float4 a = p[0];
#pragma unroll 4
    for (int s = 1; s < S; ++s) {
      const float4 b = p[s * n4];
      a.x += b.x, a.y += b.y, a.z += b.z, a.w += b.w;
    }
    const int64_t e = id * 4, n = e / K, k = e - n * K;
    *reinterpret_cast<uint2*>(out + n * o_rs + k) = make_uint2(pack_bf16x2(a.x, a.y), pack_bf16x2(a.z, a.w));
  }
  if (cout != nullptr && id < N) {
    float t = 0.f;
    for (int s = 0; s < S; ++s) t += csum[(int64_t)s * N + id];
    cout[id] = f2bf(t);
  }
}

// Row ranges S: the least of the tiles' time (measured: per step of 32 rows 0.58 us for a tile alone on
// its CU, 0.92 us for the two that share one, 6 us per round) and the partial tiles' (written and read
// at about 5 TB/s, and a launch of 4 us), in hundredths of a microsecond.
int split_of(int64_t M, int64_t N, int64_t K) {
  const int64_t tiles = ((N + kBN - 1) / kBN) * ((K + kBK - 1) / kBK), steps = (M + kStep - 1) / kStep;
  int64_t best = INT64_MAX;
  int S = 1;
  for (int s = 1; s <= kMaxSplit && s <= std::max<int64_t>(1, steps / 2); ++s) {
    const int64_t c = (tiles * s + 255) / 256, st = (steps + s - 1) / s;  // steps of 32
    int64_t t = c / 2 * (92 * st + 600) + c % 2 * (58 * st + 600);
    if (s > 1) t += s * N * K * 8 / 50000 + 400;
    if (t < best) best = t, S = s;
  }
  return S;
}

bool fits32(int64_t rs) { return rs <= ((int64_t)1 << 30) / (2 * kStep); }

}  // namespace

// From 4096 rows on, 1024 where the column sums are wanted too: the library's product is faster below
// (2048 x 768 x 832 18 against 22 us), but not with its column-sum kernel (2048 x 2240 x 512 40 against 24).
// Between 4096 and 10240 rows the library keeps outputs of 8 to 20 million values (in_proj at d_model 1536 and
// 2048), whose split leaves this kernel two partial rounds (rows x N x K, library and this: 4096 x 6336 x 1536
// 105, 124; 8192 185, 195; 10240 227, 242; 4096 x 8576 x 2048 184, 197; 8192 340, 374); the lines lie where the two
// cross: 3000 x 6336 x 1536 92, 92; 12288 379, 285; 8192 x 5184 x 1280 144, 133; 8192 x 10624 x 2560 578, 533.
extern "C" int hdcm_gemm_tn_preferred(int64_t M, int64_t N, int64_t K, int col_sums, int dtype) {
  if (!(dtype == HDCM_BF16 && M >= (col_sums ? 1024 : 4096) && N % 8 == 0 && K % 8 == 0 && N > 0 && K > 0 &&
        M < (int64_t)1 << 30 && N < (int64_t)1 << 24 && K < (int64_t)1 << 24 && fits32(N) && fits32(K)))
    return 0;
  return !(M >= 4096 && M <= 10240 && N * K >= 8000000 && N * K <= 20000000);
}

extern "C" size_t hdcm_gemm_tn_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const int S = split_of(M, N, K);
  return (size_t)S * N * (S > 1 ? K + 1 : 1) * sizeof(float);
}

extern "C" int hdcm_gemm_tn(const void* y, int64_t y_row_stride, const void* x, int64_t x_row_stride, void* out,
                            int64_t out_row_stride, void* col_sums, void* ws, size_t ws_bytes, int64_t M, int64_t N,
                            int64_t K, int dtype, void* stream) {
  HDCM_CHECK_ARG(dtype == HDCM_BF16, HDCM_EUNSUPPORTED);
  HDCM_CHECK_ARG(M > 0 && N > 0 && K > 0 && y && x && out, HDCM_EINVAL);
  HDCM_CHECK_ARG(y_row_stride >= N && x_row_stride >= K && out_row_stride >= K, HDCM_EINVAL);
  HDCM_CHECK_ARG(N % 8 == 0 && K % 8 == 0 && y_row_stride % 8 == 0 && x_row_stride % 8 == 0 && out_row_stride % 4 == 0 &&
                     hdcm_aligned16(y) && hdcm_aligned16(x) && ((uintptr_t)out & 7u) == 0 && ((uintptr_t)col_sums & 1u) == 0,
                 HDCM_EALIGN);
  HDCM_CHECK_ARG(M < (int64_t)1 << 30 && N < (int64_t)1 << 24 && K < (int64_t)1 << 24 && fits32(y_row_stride) &&
                     fits32(x_row_stride),
                 HDCM_EUNSUPPORTED);
  HDCM_CHECK_ARG(ws != nullptr && ws_bytes >= hdcm_gemm_tn_workspace_bytes(M, N, K), HDCM_EWORKSPACE);
  HDCM_CHECK_ARG(hdcm_aligned16(ws), HDCM_EALIGN);
  const int64_t n_nt = (N + kBN - 1) / kBN, n_kt = (K + kBK - 1) / kBK;
  HDCM_CHECK_ARG(n_nt * n_kt < (int64_t)1 << 24, HDCM_EUNSUPPORTED);
  const int S = split_of(M, N, K);
  const int64_t steps = (M + kStep - 1) / kStep;
  const int split_rows = (int)((steps + S - 1) / S * kStep);
  const int used = (int)((M + split_rows - 1) / split_rows);  // ranges that hold rows
  float* part = used > 1 ? (float*)ws : nullptr;
  float* cs = (float*)ws + (used > 1 ? (size_t)S * N * K : 0);
  hipStream_t s = (hipStream_t)stream;
  HDCM_LAUNCH(gemm_tn_kernel, dim3((unsigned)(n_nt * n_kt * used)), dim3(kThreads), 0, s, (const bf16_t*)y,
              y_row_stride, (const bf16_t*)x, x_row_stride, (bf16_t*)out, out_row_stride, part, col_sums ? cs : nullptr,
              (int)M, (int)N, (int)K, (int)n_nt, (int)(n_nt * n_kt), split_rows);
  const int st = hdcm_launch_status();
  if (st || (!part && !col_sums)) return st;
  const int64_t n = std::max<int64_t>(part ? N * K / 4 : 0, N);
  HDCM_LAUNCH(sum_parts_kernel, dim3((unsigned)((n + kThreads - 1) / kThreads)), dim3(kThreads), 0, s, part, cs, used,
              (int)N, (int)K, (bf16_t*)out, out_row_stride, (bf16_t*)col_sums);
  return hdcm_launch_status();
}
