// lanes.hpp - reductions over the 64 lanes of a wavefront.
//
// The butterfly of lane distances 32, 16, 8, 4, 2, 1: lane i combines its value
// with lane (i ^ d)'s, so every lane ends with the same sum, formed in the same
// tree whatever moves the values.  Distances 32 and 16 are the two halves
// swapped between two registers, 8 to 1 are data-parallel-primitive moves: a
// step costs a handful of vector instructions (about 30 cycles with the
// addition).  The general shuffle goes through the LDS unit, two permutes of
// over 100 cycles for each FP64 step; a reduction's second pass, which does
// little else, took 2.4 us more with it (six sums, one wavefront each).
#pragma once
#include <hip/hip_runtime.h>

namespace pihm {

struct LanePair {
  double a, b;   // lane i's and lane (i ^ D)'s value, in either order
};

template <int D>
__device__ __forceinline__ LanePair lane_pair(double v) {
  static_assert(D == 32 || D == 16 || D == 8 || D == 4 || D == 2 || D == 1, "a butterfly distance");
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = (unsigned)u, hi = (unsigned)(u >> 32);
  unsigned al = lo, ah = hi, bl, bh;
  if constexpr (D == 32) {
    const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
    const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
    al = l[0]; bl = l[1]; ah = h[0]; bh = h[1];
  } else if constexpr (D == 16) {
    const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
    const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
    al = l[0]; bl = l[1]; ah = h[0]; bh = h[1];
  } else {
    constexpr int kRor8 = 0x128, kHalfMirror = 0x141, kQuad3210 = 0x1B, kQuad1032 = 0x4E, kQuad2301 = 0xB1;
    if constexpr (D == 4) {   // i -> i ^ 7, then ^ 3
      bl = __builtin_amdgcn_mov_dpp(lo, kHalfMirror, 0xf, 0xf, true);
      bh = __builtin_amdgcn_mov_dpp(hi, kHalfMirror, 0xf, 0xf, true);
      bl = __builtin_amdgcn_mov_dpp(bl, kQuad3210, 0xf, 0xf, true);
      bh = __builtin_amdgcn_mov_dpp(bh, kQuad3210, 0xf, 0xf, true);
    } else {
      constexpr int c = (D == 8) ? kRor8 : (D == 2) ? kQuad1032 : kQuad2301;
      bl = __builtin_amdgcn_mov_dpp(lo, c, 0xf, 0xf, true);
      bh = __builtin_amdgcn_mov_dpp(hi, c, 0xf, 0xf, true);
    }
  }
  return LanePair{__builtin_bit_cast(double, ((unsigned long long)ah << 32) | al),
                  __builtin_bit_cast(double, ((unsigned long long)bh << 32) | bl)};
}

// Combines v over the wavefront with op(a, b), which must be commutative.
template <class Op>
__device__ __forceinline__ double wave_all(double v, Op op) {
  LanePair p = lane_pair<32>(v);
  v = op(p.a, p.b);
  p = lane_pair<16>(v);
  v = op(p.a, p.b);
  p = lane_pair<8>(v);
  v = op(p.a, p.b);
  p = lane_pair<4>(v);
  v = op(p.a, p.b);
  p = lane_pair<2>(v);
  v = op(p.a, p.b);
  p = lane_pair<1>(v);
  return op(p.a, p.b);
}
__device__ __forceinline__ double wave_sum(double v) {
  return wave_all(v, [](double a, double b) { return a + b; });
}
__device__ __forceinline__ double wave_min(double v) {
  return wave_all(v, [](double a, double b) { return fmin(a, b); });
}
__device__ __forceinline__ double wave_max(double v) {
  return wave_all(v, [](double a, double b) { return fmax(a, b); });
}

}  // namespace pihm
