// rd_gpu.h -- device helpers shared by the kernel files: typed global pointers with a cache policy,
// wave numbers, the preconditioner factor and block reductions.
#pragma once
#include <hip/hip_runtime.h>

#include "fft2s.h"
#include "rd_device.h"

namespace glia {
using namespace dev;

// ---------------------------------------------------------------------------------------------
// helpers
// ---------------------------------------------------------------------------------------------
// pointers into device global memory (address space 1): loads and stores through them compile to
// global_* instructions with a uniform base and 32-bit lane offsets instead of flat accesses
#define GLIA_GLOBAL __attribute__((address_space(1)))
typedef float v2f __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
// Cache policy of a kernel's global accesses, a template argument of its pointers: bit 0 makes
// the loads, bit 1 the stores non-temporal (the nt bit: the line streams through the caches instead
// of being kept for reuse).  Each pass sets its own (GLIA_NT_* below).
template <int H>
struct GRefT {
  GLIA_GLOBAL v2f* p;
  __device__ __forceinline__ operator float2() const {
    v2f a;
    if constexpr ((H & 1) != 0) {
      a = __builtin_nontemporal_load(p);
    } else {
      a = *p;
    }
    return make_float2(a.x, a.y);
  }
  __device__ __forceinline__ GRefT& operator=(float2 v) {
    v2f a;
    a.x = v.x;
    a.y = v.y;
    if constexpr ((H & 2) != 0) {
      __builtin_nontemporal_store(a, p);
    } else {
      *p = a;
    }
    return *this;
  }
};
template <int H>
struct GPtrT {
  GLIA_GLOBAL v2f* p;
  __device__ __forceinline__ GRefT<H> operator[](unsigned i) const { return GRefT<H>{p + i}; }
  __device__ __forceinline__ GPtrT operator+(int64_t o) const { return GPtrT{p + o}; }
  __device__ __forceinline__ explicit operator bool() const { return p != nullptr; }
};
using GPtr = GPtrT<0>;
// 16-byte accesses of the elementwise passes under the same policy bits
template <int H>
__device__ __forceinline__ v4f ld4(GLIA_GLOBAL v4f* p) {
  if constexpr ((H & 1) != 0) {
    return __builtin_nontemporal_load(p);
  } else {
    return *p;
  }
}
template <int H>
__device__ __forceinline__ void st4(GLIA_GLOBAL v4f* p, v4f v) {
  if constexpr ((H & 2) != 0) {
    __builtin_nontemporal_store(v, p);
  } else {
    *p = v;
  }
}
template <int H = 0>
__device__ __forceinline__ GPtrT<H> gptr(const void* q) { return GPtrT<H>{(GLIA_GLOBAL v2f*)q}; }

// complex slot s of a member: work slots below CS_NUM, state-pool entries (history/checkpoints) above
template <int H = 0>
__device__ __forceinline__ GPtrT<H> cptr(const MemberDev& M, int s) {
  return gptr<H>((s < CS_NUM) ? M.c[s] : M.hist[s - CS_NUM]);
}
// the same slot as a plain pointer (elementwise kernels)
__device__ __forceinline__ float2* craw(const MemberDev& M, int s) { return (s < CS_NUM) ? M.c[s] : M.hist[s - CS_NUM]; }
// a real field viewed as float2 pairs (x[2n], x[2n+1])
template <int H = 0>
__device__ __forceinline__ GPtrT<H> rptr2(const MemberDev& M, int r) { return gptr<H>(M.r[r]); }

// wave number with the Nyquist mode zeroed (reference src/cuda/SpectralOperators.cu:63-72)
__device__ __forceinline__ float wnum(int k, int n) {
  const int h = n >> 1;
  return (k < h) ? (float)k : ((k == h) ? 0.f : (float)(k - n));
}

// spectral preconditioner factor times N^3 (reference src/cuda/DiffCoef.cu:11-63):
// FFT(B r) = r_hat / (1 + 0.25 dt kbar |w|^2), or r_hat when the denominator is 0
__device__ __forceinline__ float precf(float pc, float wx, float wy, float wz) {
  const float v = 1.0f + pc * (wx * wx + wy * wy + wz * wz);
  return (v == 0.0f) ? 1.0f : 1.0f / v;
}

// block-wide FP64 reduction of NQ values; thread 0 writes out[0..NQ)
template <int NQ>
__device__ __forceinline__ void block_reduce_store(double (&v)[NQ], double* out) {
  __shared__ double red[NQ][16];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int nw = (blockDim.x + 63) >> 6;
#pragma unroll
  for (int q = 0; q < NQ; q++) {
    double x = v[q];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) x += __shfl_down(x, off, 64);
    if (lane == 0) red[q][wid] = x;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int q = 0; q < NQ; q++) {
      double s = 0;
      for (int w = 0; w < nw; w++) s += red[q][w];
      out[q] = s;
    }
  }
}

// block-wide sum of one value, result broadcast to every thread
__device__ __forceinline__ double block_sum_all(double x) {
  __shared__ double red[16];
  __shared__ double res;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int nw = (blockDim.x + 63) >> 6;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) x += __shfl_down(x, off, 64);
  if (lane == 0) red[wid] = x;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0;
    for (int w = 0; w < nw; w++) s += red[w];
    res = s;
  }
  __syncthreads();
  const double r = res;
  __syncthreads();
  return r;
}

// sum of column q of part[nb][nq], identical on every thread (fixed order: deterministic)
__device__ __forceinline__ double sum_partials(const double* part, int nb, int nq, int q) {
  double s = 0;
  for (int b = threadIdx.x; b < nb; b += blockDim.x) s += part[(int64_t)b * nq + q];
  return block_sum_all(s);
}

// start of every CN solve: parameters and a clean iteration state
__device__ __forceinline__ void pcg_begin_state(PcgState* s, double tau) {
  s->tau = tau;
  s->beta = s->betaold = s->dpi = s->dpiold = s->alpha = s->bcoef = 0;
  s->dp = s->rnorm0 = s->ttol = 0;
  s->i = 0;
  s->its = 0;
  s->reason = 0;
  s->done = 0;
  if (!s->active) {  // DiffusionSolver::solve returns at once when k_scale == 0
    s->done = 1;
    s->solves += 1;
  }
}

// The x-planes on which the matvec's middle is not zero (MemberDev::planes), for the X passes around it:
// the inverse pass need not write, nor the forward pass read, the other planes' rows.  A quarter of a
// scan's planes hold no brain.  Without use every plane counts.
// The words are named one by one: an array of them stayed in scratch memory (16-40 bytes a lane, 11
// spilled registers in the 256-point inverse pass), which cost more traffic than the skipped rows saved:
// inverse and forward X pass 122 and 121 -> 106 and 112 us at 8 x 160^3, 234 and 259 -> 203 and 220 at 4 x 256^3
// (115 and 127, 237 and 257 with every row written and read).
struct PlaneBits {
  uint64_t q0, q1, q2, q3;
  __device__ __forceinline__ PlaneBits(const MemberDev& M, int use) {
    const auto word = [&](int i) -> uint64_t {
      return use ? (uint64_t)M.planes[2 * i + 1] << 32 | M.planes[2 * i] : ~0ull;
    };
    q0 = word(0), q1 = word(1), q2 = word(2), q3 = word(3);
  }
  __device__ __forceinline__ unsigned word32(int i) const {
    const uint64_t q = i < 2 ? q0 : i < 4 ? q1 : i < 6 ? q2 : i < 8 ? q3 : ~0ull;
    return (unsigned)(i & 1 ? q >> 32 : q);
  }
  // plane c + v with c known at compile time and v < NT <= 32
  template <int NT>
  __device__ __forceinline__ bool on(int c, int v) const {
    const int sh = c & 31;
    if (sh + NT <= 32) return (word32(c >> 5) >> (sh + v)) & 1;
    return ((((uint64_t)word32((c >> 5) + 1) << 32) | word32(c >> 5)) >> (sh + v)) & 1;
  }
};

// the vector update of an elasticity CG iteration, from its state and, for the x and r update, the
// summed <p, A p>: p = z + t p with t = beta / betaold (upd false: p = z, the first iteration and a
// zero beta), or x += t p, r -= t w with t = beta / <p, A p> (upd false: none, where the CG stops on
// <p, A p>: 0, not finite, or of the sign opposite to the last one's after the first iteration)
struct CgStep {
  float t;
  bool upd;
};
template <bool XR>
__device__ __forceinline__ CgStep cg_step(const PcgState* S, const double* sc) {
  CgStep c{0.0f, false};
  if (XR) {
    const double q = sc[0];
    c.upd = !(isnan(q) || isinf(q) || q == 0.0 || (S->i != 0 && q * S->dpi <= 0.0));
    if (c.upd) c.t = (float)(S->beta / q);
  } else {
    const double b = S->i ? S->beta / S->betaold : 0.0;
    c.upd = b != 0.0;
    c.t = (float)b;
  }
  return c;
}

}  // namespace glia
