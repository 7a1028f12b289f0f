// Gradient of the slot memory + GroupNorm + gate (slot_kernels.h has the forward, its
// decomposition, tiles and LDS layout) in two passes over the sequence, for gfx950.
//
// Forward, per head: y = attend(phi(q), phi(k), v) with weights w(t, j), out = GN(y) sigmoid(gate).
// Given dout, with dy the gradient of y (GroupNorm and gate backward):
//   d phi(q)_t = sum_{j<=t} w(t,j) (dy_t . v_j) phi(k_j)          = attend(dy, v, phi(k))
//   d v_j      = sum_{t>=j} w(t,j) (phi(k_j) . phi(q_t)) dy_t     = attend(phi(k), phi(q), dy), reversed
//   d phi(k)_j = sum_{t>=j} w(t,j) (v_j . dy_t) phi(q_t)          = attend(v, dy, phi(q)), reversed
//   d q = d phi(q) phi'(q), d k = d phi(k) phi'(k), phi'(z) = 1 (z > 0) else exp(z).
// A sequence whose length is a multiple of the chunk reads the same backwards (rows taken from the
// last one, negative row strides), chunks included.  So both passes have one shape, for "query"
// rows a, "key" rows b, value rows v and a second query e:
//   y1_i = attend(phi(a), phi(b), v)_i,   y2_i = attend(e, v, phi(b))_i,
//   forward pass  (FWD): a = q, b = k, v = v: y1 = y, from which the GroupNorm and gate backward
//                        makes e = dy in registers; stores d gate, dy and d q = y2 phi'(q);
//   reverse pass:        a = k, b = q, v = dy, e = v: stores d v = y1 and d k = y2 phi'(k).
// y1 and y2 share the tile's operands and the carried state: S = sum phi(b)^T v serves y1 as
// phi(a) S and y2 as e S^T, so the forward pass runs on the states the forward kernels left and
// the reverse one on one state pre-pass over (phi(q), dy).  y never reaches memory, the
// recomputed feature maps never do, and q, k, v, gate and dout are read once per pass.
// Measured against the passes this replaces (y recomputed, GroupNorm backward, staged phi(q),
// phi(k) and v, three attention passes, four state pre-passes): mixer forward and backward at
// 32768 x 1024 bf16 720 -> 435 us, of it the two passes 122 + 91 us (4.4 TB/s).
//
// Layouts (see slot_kernels.h): y1^T tiles leave lane (l16 = row, kg) columns 16 vt + 4 kg .. +3;
// two adjacent tiles are exactly a B operand of K = 32 under the slot order
//   slot s -> 32 t + (s < 4 ? 4 kg + s : 16 + 4 kg + s - 4),
// so e = dy enters the second half's products from registers, with v and S read in that order.
// Bound: HBM (8 activations read or written per element in the forward pass, 6 in the reverse).
#pragma once

#include "slot_kernels.h"

namespace {

// A operand over rows of a row-major tile: lane x = lane % 16 receives column d0 + x of rows
// r0 + (the slot order above).
template <typename T>
__device__ __forceinline__ void frag_cols(Frag<T>& f, const T* tile, int pitch, int r0, int d0, int lane) {
  const int x = lane & 15, g = lane >> 4;
  if constexpr (sizeof(T) == 2) {
    const T* p = tile + (r0 + 4 * g + (x >> 2)) * pitch + d0 + 4 * (x & 3);
    const bf16x4_t lo = lds_tr16(p), hi = lds_tr16(p + 16 * pitch);
    f.v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  } else {
#pragma unroll
    for (int s = 0; s < 8; ++s) f.v[s] = tile[(r0 + (s < 4 ? 4 * g + s : 16 + 4 * g + s - 4)) * pitch + d0 + x];
  }
}

// The first half of a fragment kept, the second zeroed: the last K step of an odd count of
// 16-wide tiles.
__device__ __forceinline__ void frag_first_half(Frag<bf16_t>& f) {
#pragma unroll
  for (int s = 4; s < 8; ++s) f.v[s] = (__bf16)0.f;
}
__device__ __forceinline__ void frag_first_half(Frag<float>& f) {
#pragma unroll
  for (int s = 4; s < 8; ++s) f.v[s] = 0.f;
}

// A operand over the value columns of v: lane x receives row j0 + x, columns c0 + (the slot
// order).  bf16 tiles hold v row-major, fp32 ones transposed.
template <typename T, int HD, int TC>
__device__ __forceinline__ void frag_vrow(Frag<T>& f, const T* sv, int j0, int c0, bool both, int lane) {
  using LD = Lds<T, HD, TC>;
  const int x = lane & 15, g = lane >> 4;
  if constexpr (LD::TR) {
    const T* p = sv + (j0 + x) * LD::PV + c0 + 4 * g;
    frag_load4x2(f, p, both ? p + 16 : p);
  } else {
#pragma unroll
    for (int s = 0; s < 8; ++s)
      f.v[s] = sv[(c0 + (s < 4 ? 4 * g + s : (both ? 16 : 0) + 4 * g + s - 4)) * LD::PV + j0 + x];
  }
  if (!both) frag_first_half(f);
}

// phi of a fragment of raw values, rounded to the operand type.
__device__ __forceinline__ Frag<bf16_t> frag_phi(const Frag<bf16_t>& f) {
  float x[8];
  unpack_bf16x8(f.v, x);
#pragma unroll
  for (int s = 0; s < 8; ++s) x[s] = phi_f(x[s]);
  Frag<bf16_t> o;
  o.v = pack_bf16x8(x);
  return o;
}
__device__ __forceinline__ Frag<float> frag_phi(const Frag<float>& f) {
  Frag<float> o;
#pragma unroll
  for (int s = 0; s < 8; ++s) o.v[s] = phi_f(f.v[s]);
  return o;
}

// This lane's 4 NVT values of one row in the output layout (columns 16 vt + 4 kg .. +3 of every
// tile vt).  bf16 rows with an even tile count move in 16-byte runs of 8 consecutive columns,
// traded between the lane pairs (kg, kg ^ 1) by v_permlane16_swap (slot_kernels.h, kPairs).
template <typename T, int HD>
struct RowIo {
  static constexpr int NVT = HD / 16;
  static constexpr bool kPairs = sizeof(T) == 2 && NVT % 2 == 0;
  static constexpr int NG = kPairs ? NVT / 2 : NVT;
  static constexpr int kStep = kPairs ? 32 : 16;
  static __device__ __forceinline__ int col(int kg) { return kPairs ? 16 * (kg & 1) + 8 * (kg >> 1) : 4 * kg; }
  // p: the row's first column of this head plus col(kg)
  static __device__ __forceinline__ void load(uint4 (&raw)[NG], const T* p) {
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      if constexpr (kPairs || sizeof(T) == 4) {
        raw[g] = *reinterpret_cast<const uint4*>(p + g * kStep);
      } else {
        const uint2 v = *reinterpret_cast<const uint2*>(p + g * kStep);
        raw[g] = make_uint4(v.x, v.y, 0u, 0u);
      }
    }
  }
  static __device__ __forceinline__ void unpack(const uint4 (&raw)[NG], float (&v)[NVT][4]) {
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      if constexpr (kPairs) {
        const auto a = __builtin_amdgcn_permlane16_swap(raw[g].x, raw[g].z, false, false);
        const auto b = __builtin_amdgcn_permlane16_swap(raw[g].y, raw[g].w, false, false);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          v[2 * g + h][0] = __uint_as_float(a[h] << 16);
          v[2 * g + h][1] = __uint_as_float(a[h] & 0xffff0000u);
          v[2 * g + h][2] = __uint_as_float(b[h] << 16);
          v[2 * g + h][3] = __uint_as_float(b[h] & 0xffff0000u);
        }
      } else {
        load4<T>(reinterpret_cast<const T*>(&raw[g]), v[g]);
      }
    }
  }
  static __device__ __forceinline__ void store(T* p, const float (&v)[NVT][4], bool ok) {
    if constexpr (kPairs) {
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        uint32_t w[2][2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          w[h][0] = pack_bf16x2(v[2 * g + h][0], v[2 * g + h][1]);
          w[h][1] = pack_bf16x2(v[2 * g + h][2], v[2 * g + h][3]);
        }
        const auto a = __builtin_amdgcn_permlane16_swap(w[0][0], w[1][0], false, false);
        const auto b = __builtin_amdgcn_permlane16_swap(w[0][1], w[1][1], false, false);
        if (ok) *reinterpret_cast<uint4*>(p + g * kStep) = make_uint4(a[0], b[0], a[1], b[1]);
      }
    } else if (ok) {
#pragma unroll
      for (int g = 0; g < NG; ++g) store4<T>(p + g * kStep, v[g]);
    }
  }
};

// Operands of a pass; pointers at the sequence batch's first row taken (the last one in the
// reverse pass, with negative row strides), first column of head 0.
template <typename T>
struct GradArgs {
  const T *a, *b, *v, *e;  // e: the gate (FWD) or v (reverse)
  const T* dout;           // FWD
  int64_t prs;             // row stride of a, b, e (projs)
  int64_t vrs, dors;
  T *o1, *o2, *dy;         // d gate or d v; d q or d k; dy (FWD)
  int64_t o_rs, dy_rs;
  const T *gamma, *gn_w, *gn_b;
  const float *Ain, *Win;  // segment-start states A and (null: zero) W
  float* part;             // FWD: [B * nseg][2][H * HD] partial sums of d gn_w, d gn_b
  float gn_eps;
  int L, C, cshift, conf, seg_rows, nseg;
};

template <typename T, int HD, int TC, bool HAS_W, bool FWD>
__global__ __launch_bounds__(kThreads, HD > 64 ? 1 : 2) void slot_grad_kernel(const GradArgs<T> A) {
  using LD = Lds<T, HD, TC>;
  using RL = RowLoader<T, HD, TC>;
  using IO = RowIo<T, HD>;
  __shared__ __attribute__((aligned(16))) T sm[LD::total];
  __shared__ float sgw[HD], sgb[HD];
  static_assert(LD::total * sizeof(T) + 2 * HD * sizeof(float) <= 160 * 1024, "LDS budget");
  static_assert(kWaves * 2 * HD * sizeof(float) <= LD::total * sizeof(T), "column sums reuse the tiles");
  constexpr int NVT = HD / 16, NKS = LD::HDK / 32, NJS = TC / 32, NIT = TC / 16;
  constexpr int OWN = (NVT + kWaves - 1) / kWaves;

  const int tid = threadIdx.x, lane = tid & (kWave - 1), w = tid / kWave;
  const int l16 = lane & 15, kg = lane >> 4;
  const int h = blockIdx.x, seg = blockIdx.y, bb = blockIdx.z, H = gridDim.x;
  const T gamma_raw = A.gamma[h];
  T gnw_raw = T(), gnb_raw = T();
  if constexpr (FWD) {
    gnw_raw = A.gn_w[h * HD + tid % HD];
    gnb_raw = A.gn_b[h * HD + tid % HD];
  }
  const bool one_chunk = A.cshift >= 31;
  const int C = A.C;
  const int p_begin = seg * A.seg_rows, p_end = min(A.L, p_begin + A.seg_rows);
  auto tile_len = [&](int p) {
    const int t = min(TC, p_end - p);
    return A.conf ? min(t, C - p % C) : t;
  };
  // row r of the batch: base + (bb L + r) * stride; in the reverse pass the batches run backwards too
  const int64_t row0 = (int64_t)bb * A.L;
  const int64_t col0 = (int64_t)h * HD;

  f32x4_t stA[OWN][NVT];
  f32x4_t stW[HAS_W ? OWN : 1][HAS_W ? NVT : 1];
  const int64_t st0 = (((int64_t)bb * H + h) * A.nseg + seg) * HD * HD;
#pragma unroll
  for (int ov = 0; ov < OWN; ++ov) {
    const int vt = w + kWaves * ov;
#pragma unroll
    for (int mt = 0; mt < NVT; ++mt) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t e = st0 + (mt * 16 + kg * 4 + r) * HD + vt * 16 + l16;
        stA[ov][mt][r] = vt < NVT ? A.Ain[e] : 0.f;
        if constexpr (HAS_W) stW[ov][mt][r] = A.Win != nullptr && vt < NVT ? A.Win[e] : 0.f;
      }
    }
  }

  uint4 ra[RL::N], rbv[2 * RL::N];  // a; b then v
  auto load_tile = [&](int p) {
    const int tl = tile_len(p);
    RL::load(ra, A.a + col0 + (row0 + p) * A.prs, A.prs, tl, tid);
    RL::load(rbv, A.b + col0 + (row0 + p) * A.prs, A.prs, tl, tid);
    RL::load(rbv + RL::N, A.v + col0 + (row0 + p) * A.vrs, A.vrs, tl, tid);
  };
  load_tile(p_begin);
  // e (and dout) in the output layout, one tile ahead
  uint4 re[IO::NG], rd[FWD ? IO::NG : 1];
  const int giq = (w < NIT ? w : 0) * 16 + l16;
  auto load_rows = [&](int p) {
    const int64_t r = row0 + p + (giq < tile_len(p) ? giq : 0);
    IO::load(re, A.e + col0 + r * A.prs + IO::col(kg));
    if constexpr (FWD) IO::load(rd, A.dout + col0 + r * A.dors + IO::col(kg));
  };
  if (w < NIT) load_rows(p_begin);

  const float lg2 = log2f(to_f<T>(gamma_raw));
  const float ginv[4] = {1.0f, fexp2(-lg2), fexp2(-2.0f * lg2), fexp2(-3.0f * lg2)};
  if (FWD && tid < HD) {
    sgw[tid] = to_f<T>(gnw_raw);
    sgb[tid] = to_f<T>(gnb_raw);
  }
  zero_contraction_pad<T, HD, TC>(sm, tid);
  float sw[FWD ? NVT : 1][4], sb[FWD ? NVT : 1][4];  // this lane's columns of d gn_w, d gn_b
  if constexpr (FWD) {
#pragma unroll
    for (int vt = 0; vt < NVT; ++vt)
#pragma unroll
      for (int r = 0; r < 4; ++r) sw[vt][r] = sb[vt][r] = 0.f;
  }

  for (int p = p_begin, tlen; p < p_end; p += tlen) {
    tlen = tile_len(p);
    __syncthreads();
    // a as stored (phi is taken on its fragments: each row is used by one wave only); b and v as
    // in the forward
    RL::stage(ra, sm + LD::oQ, LD::PQ, tlen, tid);
    stage_tile<T, HD, TC, 1, 2, false, true>(rbv, sm, tlen, lg2, tid);
    {
      float cA = 1.0f, cW = 0.0f;
      if constexpr (HAS_W) {
        cA = fexp2((float)(p % C) * lg2);
        cW = fexp2(lg2);
      }
#pragma unroll
      for (int ov = 0; ov < OWN; ++ov) {
        const int vt = w + kWaves * ov;
        if (vt >= NVT) continue;
#pragma unroll
        for (int mt = 0; mt < NVT; ++mt) {
          float v[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            v[r] = cA * stA[ov][mt][r];
            if constexpr (HAS_W) v[r] += cW * stW[ov][mt][r];
          }
          store4<T>(sm + LD::oS + (vt * 16 + l16) * LD::PQ + mt * 16 + kg * 4, v);
        }
      }
    }
    const int pn = p + tlen < p_end ? p + tlen : p;  // the last tile again: a fixed load count
    load_tile(pn);
    __syncthreads();

    if (w < NIT) {
      const int iq = w * 16 + l16;
      const float qd = fexp2((float)iq * lg2);
      // the tile's weights for this lane's key rows of step t (0 for masked pairs)
      auto weights = [&](int t, float (&c)[8]) {
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
          const int jt = 2 * t + hh, j0 = jt * 16 + kg * 4;
          if (one_chunk) {
            const float d0 = fexp2((float)(iq - j0) * lg2);
#pragma unroll
            for (int r = 0; r < 4; ++r) c[hh * 4 + r] = (jt <= w && j0 + r <= iq) ? d0 * ginv[r] : 0.f;
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int j = j0 + r;
              const int ex = iq - j - (((iq >> A.cshift) != (j >> A.cshift)) ? 1 : 0);
              c[hh * 4 + r] = (jt <= w && j <= iq) ? fexp2((float)ex * lg2) : 0.f;
            }
          }
        }
      };
      // decayed scores as the next product's B operand (masked pairs 0, whatever the product holds)
      auto decayed = [&](const f32x4_t (&s)[2], int t) {
        float c[8], pv[8];
        weights(t, c);
#pragma unroll
        for (int k = 0; k < 8; ++k) pv[k] = c[k] != 0.f ? s[k >> 2][k & 3] * c[k] : 0.f;
        Frag<T> f;
        frag_from_f32(f, pv);
        return f;
      };

      // ---- y1 = qd phi(a) S + P1 v
      f32x4_t y1[NVT];
#pragma unroll
      for (int vt = 0; vt < NVT; ++vt) y1[vt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      {
        Frag<T> fq[NKS];
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
          Frag<T> f;
          frag_rows8<T, HD, TC>(f, sm + LD::oQ, iq, ks * 32 + kg * 8);
          fq[ks] = frag_phi(f);
        }
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
          for (int vt = 0; vt < NVT; ++vt) {
            Frag<T> a;
            frag_rows8<T, HD, TC>(a, sm + LD::oS, vt * 16 + l16, ks * 32 + kg * 8);
            y1[vt] = mma(a, fq[ks], y1[vt]);
          }
#pragma unroll
        for (int vt = 0; vt < NVT; ++vt) y1[vt] *= qd;
#pragma unroll
        for (int t = 0; t < NJS; ++t) {
          if (2 * t > w) continue;
          f32x4_t s[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
          for (int hh = 0; hh < 2; ++hh) {
            if (2 * t + hh > w) continue;
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) {
              Frag<T> a;
              frag_rows8<T, HD, TC>(a, sm + LD::oK, (2 * t + hh) * 16 + l16, ks * 32 + kg * 8);
              s[hh] = mma(a, fq[ks], s[hh]);
            }
          }
          const Frag<T> pf = decayed(s, t);
#pragma unroll
          for (int vt = 0; vt < NVT; ++vt) {
            Frag<T> a;
            frag_tok<T, HD, TC>(a, sm + LD::oV, vt * 16, 32 * t, lane);
            y1[vt] = mma(a, pf, y1[vt]);
          }
        }
      }

      // ---- e: dy from the GroupNorm and gate backward (FWD), or the loaded rows
      const bool in_tile = iq < tlen;
      const int64_t orow = row0 + p + iq;
      float ev[NVT][4];
      IO::unpack(re, ev);
      if constexpr (FWD) {
        float dv[NVT][4];
        IO::unpack(rd, dv);
        float sum = 0.f;
#pragma unroll
        for (int vt = 0; vt < NVT; ++vt)
#pragma unroll
          for (int r = 0; r < 4; ++r) sum += y1[vt][r];
        const float mean = quad_group_sum(sum) * (1.0f / HD);
        float sq = 0.f;
#pragma unroll
        for (int vt = 0; vt < NVT; ++vt)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            y1[vt][r] -= mean;
            sq += y1[vt][r] * y1[vt][r];
          }
        const float rinv = rsqrtf(quad_group_sum(sq) * (1.0f / HD) + A.gn_eps);
        float sa = 0.f, sx = 0.f;
#pragma unroll
        for (int vt = 0; vt < NVT; ++vt) {
          const int c0 = vt * 16 + kg * 4;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float xh = y1[vt][r] * rinv;
            const float sg = frcp(1.0f + fexp(-ev[vt][r]));
            const float wv = sgw[c0 + r];
            const float d = in_tile ? dv[vt][r] : 0.f;
            const float dyn = d * sg;
            ev[vt][r] = d * (xh * wv + sgb[c0 + r]) * sg * (1.0f - sg);  // d gate
            sw[vt][r] += dyn * xh;
            sb[vt][r] += dyn;
            const float dxh = dyn * wv;
            sa += dxh;
            sx += dxh * xh;
            y1[vt][r] = xh;
            dv[vt][r] = dxh;
          }
        }
        IO::store(A.o1 + orow * A.o_rs + col0 + IO::col(kg), ev, in_tile);
        const float ma = quad_group_sum(sa) * (1.0f / HD), mx = quad_group_sum(sx) * (1.0f / HD);
#pragma unroll
        for (int vt = 0; vt < NVT; ++vt)
#pragma unroll
          for (int r = 0; r < 4; ++r) ev[vt][r] = rinv * (dv[vt][r] - ma - y1[vt][r] * mx);
        IO::store(A.dy + orow * A.dy_rs + col0 + IO::col(kg), ev, in_tile);
      } else {
        float o[NVT][4];
#pragma unroll
        for (int vt = 0; vt < NVT; ++vt)
#pragma unroll
          for (int r = 0; r < 4; ++r) o[vt][r] = y1[vt][r];
        IO::store(A.o1 + orow * A.o_rs + col0 + IO::col(kg), o, in_tile);
      }
      load_rows(pn);

      // ---- y2 = qd e S^T + P2 phi(b), P2 the decayed e . v
      Frag<T> fe[NKS];
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) {
        float x[8];
#pragma unroll
        for (int s = 0; s < 8; ++s) {
          const int vt = 2 * ks + (s >> 2);
          x[s] = vt < NVT ? ev[vt < NVT ? vt : 0][s & 3] : 0.f;
        }
        frag_from_f32(fe[ks], x);
      }
      f32x4_t y2[NVT];
#pragma unroll
      for (int mt = 0; mt < NVT; ++mt) y2[mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
        for (int mt = 0; mt < NVT; ++mt) {
          Frag<T> a;
          if (2 * ks + 1 < NVT) {
            frag_cols<T>(a, sm + LD::oS, LD::PQ, 32 * ks, mt * 16, lane);
          } else {  // the last 16 value rows of S^T alone: the other half re-reads them
            frag_cols<T>(a, sm + LD::oS, LD::PQ, 32 * ks - 16, mt * 16, lane);
            Frag<T> b;
#pragma unroll
            for (int s = 0; s < 4; ++s) b.v[s] = a.v[s + 4], b.v[s + 4] = a.v[s + 4];
            frag_first_half(b);
            a = b;
          }
          y2[mt] = mma(a, fe[ks], y2[mt]);
        }
#pragma unroll
      for (int mt = 0; mt < NVT; ++mt) y2[mt] *= qd;
#pragma unroll
      for (int t = 0; t < NJS; ++t) {
        if (2 * t > w) continue;
        f32x4_t s[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
          if (2 * t + hh > w) continue;
#pragma unroll
          for (int ks = 0; ks < NKS; ++ks) {
            Frag<T> a;
            frag_vrow<T, HD, TC>(a, sm + LD::oV, (2 * t + hh) * 16, 32 * ks, 2 * ks + 1 < NVT, lane);
            s[hh] = mma(a, fe[ks], s[hh]);
          }
        }
        const Frag<T> pf = decayed(s, t);
#pragma unroll
        for (int mt = 0; mt < NVT; ++mt) {
          Frag<T> a;
          frag_cols<T>(a, sm + LD::oK, LD::PQ, 32 * t, mt * 16, lane);
          y2[mt] = mma(a, pf, y2[mt]);
        }
      }
      // times phi'(a), a as stored
      float o2[NVT][4];
#pragma unroll
      for (int mt = 0; mt < NVT; ++mt) {
        float z[4];
        load4<T>(sm + LD::oQ + iq * LD::PQ + mt * 16 + kg * 4, z);
#pragma unroll
        for (int r = 0; r < 4; ++r) o2[mt][r] = y2[mt][r] * (z[r] > 0.f ? 1.0f : fexp(z[r]));
      }
      IO::store(A.o2 + orow * A.o_rs + col0 + IO::col(kg), o2, in_tile);
    }

    // ---- state update, as in the forward
    {
      const float gt = fexp2((float)tlen * lg2);
#pragma unroll
      for (int ov = 0; ov < OWN; ++ov) {
        const int vt = w + kWaves * ov;
        if (vt >= NVT) continue;
        Frag<T> bv[NJS];
#pragma unroll
        for (int ks = 0; ks < NJS; ++ks) frag_tok<T, HD, TC>(bv[ks], sm + LD::oV, vt * 16, 32 * ks, lane);
#pragma unroll
        for (int mt = 0; mt < NVT; ++mt) {
          f32x4_t acc;
          if constexpr (HAS_W) acc = stW[ov][mt] * gt;
          else acc = stA[ov][mt] * gt;
#pragma unroll
          for (int ks = 0; ks < NJS; ++ks) {
            Frag<T> a;
            frag_tok<T, HD, TC>(a, sm + LD::oKd, mt * 16, 32 * ks, lane);
            acc = mma(a, bv[ks], acc);
          }
          if constexpr (HAS_W) stW[ov][mt] = acc;
          else stA[ov][mt] = acc;
        }
      }
      if constexpr (HAS_W) {
        if (((p + tlen) % C) == 0) {
          const float gC = fexp2((float)C * lg2);
#pragma unroll
          for (int ov = 0; ov < OWN; ++ov)
#pragma unroll
            for (int mt = 0; mt < NVT; ++mt) {
              stA[ov][mt] = stA[ov][mt] * gC + stW[ov][mt];
              stW[ov][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
            }
        }
      }
    }
  }

  if constexpr (FWD) {
    // column sums over the wave's 16 rows, then over the waves in LDS in wave order
    __syncthreads();  // every wave is done with the tiles
    float* red = reinterpret_cast<float*>(sm);  // [wave][2][HD]
#pragma unroll
    for (int vt = 0; vt < NVT; ++vt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float a = group_sum<16>(sw[vt][r]), b = group_sum<16>(sb[vt][r]);
        if (l16 == 0) {
          red[(w * 2) * HD + vt * 16 + kg * 4 + r] = a;
          red[(w * 2 + 1) * HD + vt * 16 + kg * 4 + r] = b;
        }
      }
    __syncthreads();
    if (tid < 2 * HD) {
      float t = 0.f;
#pragma unroll
      for (int k = 0; k < kWaves; ++k) t += red[k * 2 * HD + tid];
      const int j = tid / HD, c = tid % HD;
      A.part[((((int64_t)bb * A.nseg + seg) * 2 + j) * H + h) * HD + c] = t;
    }
  }
}

}  // namespace

namespace hdcm_slot {
// Arguments of hdcm_slot_grad after its checks (pointers typed in the launch).
struct GradCall {
  const void *projs, *gamma, *gn_w, *gn_b, *ws_fwd, *dout;
  int64_t prs, q_col, dors, dprs;
  void* dprojs;
  float gn_eps;
  float *dgn_w, *dgn_b;
  void *dy, *ws_rev;
  float* part;
  int64_t B, L, dm, H, C;
};
int grad_launch_bf16(const GradCall& g, const SlotPlan& pl, hipStream_t s);
int grad_launch_f32(const GradCall& g, const SlotPlan& pl, hipStream_t s);
}  // namespace hdcm_slot

namespace {

template <typename T, int HD>
int launch_grad(const hdcm_slot::GradCall& g, const SlotPlan& pl, hipStream_t s) {
  constexpr int TC = TileOf<T>::value;
  const dim3 grid((unsigned)g.H, pl.nseg, (unsigned)g.B);
  const int64_t rows = g.B * g.L, dm = g.dm;
  const T* q = (const T*)g.projs + g.q_col;
  T* dq = (T*)g.dprojs + g.q_col;
  GradArgs<T> A;
  A.a = q, A.b = q + dm, A.v = q + 2 * dm, A.e = q + 3 * dm;
  A.dout = (const T*)g.dout, A.dors = g.dors;
  A.prs = A.vrs = g.prs;
  A.o1 = dq + 3 * dm, A.o2 = dq, A.o_rs = g.dprs;
  A.dy = (T*)g.dy, A.dy_rs = dm;
  A.gamma = (const T*)g.gamma, A.gn_w = (const T*)g.gn_w, A.gn_b = (const T*)g.gn_b, A.gn_eps = g.gn_eps;
  A.Ain = slot_ws_a(g.ws_fwd, g.B, g.H, pl), A.Win = slot_ws_w(g.ws_fwd, g.B, g.H, pl);
  A.part = g.part;
  A.L = (int)g.L, A.C = (int)g.C, A.cshift = pl.cshift, A.conf = pl.conf, A.seg_rows = pl.seg_rows, A.nseg = pl.nseg;
  if (pl.has_w) HDCM_LAUNCH((slot_grad_kernel<T, HD, TC, true, true>), grid, dim3(kThreads), 0, s, A);
  else HDCM_LAUNCH((slot_grad_kernel<T, HD, TC, false, true>), grid, dim3(kThreads), 0, s, A);
  int st = hdcm_launch_status();
  if (st) return st;
  st = hdcm_colsum(g.part, 2 * dm, (int)(g.B * pl.nseg), 2 * (int)dm, 2 * (int)dm, 0, g.dgn_w, (int)dm, g.dgn_b, s);
  if (st) return st;

  // reverse: every row from the last one
  const T* dy_end = (const T*)g.dy + (rows - 1) * dm;
  const T* q_end = q + (rows - 1) * g.prs;
  T* dq_end = dq + (rows - 1) * g.dprs;
  float* U = (float*)g.ws_rev;
  if (pl.nseg > 1) {
    HDCM_LAUNCH((slot_state_kernel<T, HD, TC, true, true>), dim3((unsigned)g.H, pl.nseg - 1, (unsigned)g.B),
                dim3(kThreads), 0, s, q_end, -g.prs, 0, 0, (int)g.L, (const T*)g.gamma, pl.seg_rows, pl.nseg, U,
                dy_end, -dm);
    st = hdcm_launch_status();
    if (st) return st;
  }
  st = launch_scan<T>(nullptr, U, g.gamma, g.B, g.H, pl, s);
  if (st) return st;
  A.a = q_end + dm, A.b = q_end, A.v = dy_end, A.e = q_end + 2 * dm;
  A.prs = -g.prs, A.vrs = -dm;
  A.o1 = dq_end + 2 * dm, A.o2 = dq_end + dm, A.o_rs = -g.dprs;
  A.Ain = slot_ws_a(U, g.B, g.H, pl), A.Win = slot_ws_w(U, g.B, g.H, pl);
  if (pl.has_w) HDCM_LAUNCH((slot_grad_kernel<T, HD, TC, true, false>), grid, dim3(kThreads), 0, s, A);
  else HDCM_LAUNCH((slot_grad_kernel<T, HD, TC, false, false>), grid, dim3(kThreads), 0, s, A);
  return hdcm_launch_status();
}

}  // namespace
