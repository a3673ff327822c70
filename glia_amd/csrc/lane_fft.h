// lane_fft.h -- line transforms that exchange data between lanes with register swaps (gfx950), FP32.
//
// A line of length L = R * NT lives in NT lanes of one wave: lane t (t < NT) holds x[NT j + t] in
// v[j], j < R.  A transform is a radix-R DFT in registers, the twiddle W_L^{t k1}, a transpose of the
// lane index t against the low bits of k1, and a radix-NT DFT in registers.  The transpose is one
// v_permlane32_swap (NT = 2: t is lane bit 5) or also v_permlane16_swap (NT = 4: t is lane bits 5 and
// 4) per pair of registers, so a line transform needs neither LDS exchange nor barrier.  The output
// keeps the input's layout, v[j] = X[NT j + t], so transforms chain directly.
#pragma once
#include <hip/hip_runtime.h>

#include "fft2s.h"

namespace glia {
namespace dev {

typedef unsigned u2v __attribute__((ext_vector_type(2)));

// a = [a.lo, b.lo], b = [a.hi, b.hi] over the halves of the wave: lane bit 5 against (a, b)
__device__ __forceinline__ void lane_swap32(float& a, float& b) {
  const u2v r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(r.x);
  b = __uint_as_float(r.y);
}
// the same for lane bit 4 (rows of 16 lanes)
__device__ __forceinline__ void lane_swap16(float& a, float& b) {
  const u2v r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(r.x);
  b = __uint_as_float(r.y);
}
__device__ __forceinline__ void lane_swap32(float2& a, float2& b) {
  lane_swap32(a.x, b.x);
  lane_swap32(a.y, b.y);
}
__device__ __forceinline__ void lane_swap16(float2& a, float2& b) {
  lane_swap16(a.x, b.x);
  lane_swap16(a.y, b.y);
}

// tw[NT k + t] = exp(-2 pi i t k / L), k < R: ordered so that a lane's twiddles sit at fixed distances
template <int R, int NT, int S>
__device__ __forceinline__ void lane_fft(float2 (&v)[R], int t, const float2* tw) {
  static_assert(NT == 2 || NT == 4, "two or four lanes per line");
  static_assert(R % NT == 0, "the radix is a multiple of the lane count");
  Dft<R, S>::run(v);
  float2 o[R];
#pragma unroll
  for (int a = 0; a < R / NT; a++) {
    // long lines: a few groups at a time, so that the twiddles of later groups are not loaded early
    if (R >= 40 && a % (8 / NT) == 0) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = NT * a; k < NT * a + NT; k++) {
      if (k == 0) continue;
      const float2 w = tw[NT * k + t];
      v[k] = (S < 0) ? cmul(v[k], w) : cmulc(v[k], w);
    }
    if constexpr (NT == 2) {
      float2 p = v[2 * a], q = v[2 * a + 1];
      lane_swap32(p, q);
      o[a] = cadd(p, q);
      o[a + R / 2] = csub(p, q);
    } else {
      float2 u[4] = {v[4 * a], v[4 * a + 1], v[4 * a + 2], v[4 * a + 3]};
      lane_swap32(u[0], u[2]);
      lane_swap32(u[1], u[3]);
      lane_swap16(u[0], u[1]);
      lane_swap16(u[2], u[3]);
      Dft<4, S>::run(u);
#pragma unroll
      for (int k2 = 0; k2 < 4; k2++) o[a + (R / 4) * k2] = u[k2];
    }
  }
#pragma unroll
  for (int j = 0; j < R; j++) v[j] = o[j];
}

}  // namespace dev
}  // namespace glia
