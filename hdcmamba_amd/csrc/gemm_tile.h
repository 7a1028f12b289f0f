// Tiles of the GEMMs that stage both operands through LDS in rows of 128 bytes (gemm.hip, gemm_f32.hip).
#pragma once

#include "hdcm_common.h"

namespace hdcm {

constexpr int kGroup = 4;                 // o-tiles per band of the workgroup order
constexpr int kBufferFlags = 0x00020000;  // buffer resource word 3: raw 32-bit dwords
typedef __attribute__((address_space(3))) void* lds_ptr_t;

// Tile (ot, tt) of this workgroup.  Workgroup b runs on XCD b % 8; XCD x takes a contiguous run of tile
// indices, walked in bands of kGroup o-tiles (o fastest inside a band), so the workgroups resident
// on one XCD share a few panels of both operands in its L2.
__device__ __forceinline__ void tile_of(int n_otiles, int& ot, int& tt) {
  const int T = gridDim.x, b = blockIdx.x, x = b & 7, sl = b >> 3;
  int pre = 0;  // tiles taken by XCDs 0..x-1
  for (int y = 0; y < x; ++y) pre += (T - y + 7) >> 3;
  const int i = pre + sl;
  const int n_tt = T / n_otiles;
  const int band = i / (kGroup * n_tt), r = i - band * kGroup * n_tt;
  const int wb = min(kGroup, n_otiles - band * kGroup);
  tt = r / wb;
  ot = band * kGroup + (r - tt * wb);
}

// A workgroup is NWO x NWT waves, a wave NI x NJ MFMA tiles of 16 x 16.
template <int NWO, int NWT, int NI, int NJ>
struct Tile {
  static constexpr int nwo = NWO, nwt = NWT, ni = NI, nj = NJ;
  static constexpr int BO = NWO * NI * 16, BT = NWT * NJ * 16;
  static constexpr int waves = NWO * NWT, threads = waves * kWave;
  static constexpr int WL = BO / waves / 8, XL = BT / waves / 8;  // load instructions per wave and K step
  static_assert(BO % (waves * 8) == 0 && BT % (waves * 8) == 0, "whole 8-row loads");
};

template <class TL>
int64_t tiles_of(int64_t M, int64_t N) {
  return ((N + TL::BO - 1) / TL::BO) * ((M + TL::BT - 1) / TL::BT);
}

}  // namespace hdcm
