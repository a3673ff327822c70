// plane_fft.h -- building blocks of the kernels that take whole x-planes through the Y and Z transforms
// (plane_kernels.hip, plane_point.hip).
//
// Between the inverse and the forward X pass, every operator of this solver acts on the x-planes
// independently: inverse transforms along y and z, a pointwise product with a real field, forward
// transforms along z and y.  As separate passes (rd_kernels.hip) each of these reads and writes
// whole fields; here one block takes one plane of one field through all of them and touches memory
// for the input plane, the real field and the output plane only.  The line transforms run in
// registers with lane swaps (lane_fft.h); LDS only turns the plane between the two layouts:
//   Y layout: 16 columns (kz) x 4 lanes per wave, lane (c, t) holds rows y = 4 j + t of column c,
//             so global rows are read and written in 128-byte runs
//   Z layout: 32 lines (y) x 2 lanes per wave, lane (l, t) holds entries 2 j + t of line l; the
//             real-to-half-complex step pairs entries k and M - k of one lane
// A wave owns its 32 lines between the two turns, so real fields are staged through the same LDS
// rows without block barriers.
#pragma once
#include <hip/hip_runtime.h>

#include "lane_fft.h"
#include "rd_gpu.h"
#include "rd_launch.h"

namespace glia {
using namespace dev;

// sizes of one plane: N1 lines of N2 reals (M = N2/2 packed complex entries)
template <int N1, int N2>
struct PL {
  static constexpr int M = N2 / 2;
  static constexpr int RY = N1 / 4, RZ = M / 2, H = RZ / 2;  // values per lane in the two layouts
  static constexpr int WY = M / 16, WZ = (N1 + 31) / 32;     // waves that hold them
  static constexpr int W = WY > WZ ? WY : WZ, T = 64 * W;  // waves and threads of one plane
  // row pitch of the plane in LDS, odd so that 32 lanes on 32 lines hit distinct banks; 17 mod 64 at
  // M = 128 keeps the 4 x 16 column accesses of the Y layout apart too
  static constexpr int P = M == 128 ? 145 : M + 1;
  // planes that would leave room for one block only are turned in two halves (real, then imaginary)
  static constexpr bool SPLIT = N1 * P * 8 > 76 * 1024;
  static constexpr int LDS = 32 * WZ * P * (SPLIT ? 1 : 2);  // floats
  static constexpr int LINES = N1;
  // Planes of 5 to 7 waves go two to a block.  As blocks of their own only one would run on a CU: a
  // block's waves are dealt to the SIMDs from the first one on, so a second block of 5 waves would put
  // four on that SIMD, which their registers do not allow; ten waves of one block put three there (8 x
  // 160^3: 285 -> 252 us).  With more than 40 values a lane three waves a SIMD spill, and one plane a
  // block is the better one (192 x 128: 3.25 -> 2.83 ms a solve; 192 x 192 alike).
  static constexpr int CH = W > 4 && W < 8 && RY <= 40 && RZ <= 40 ? 2 : 1;
  static constexpr int TB = CH * T, MINW = CH == 2 ? 3 : 2;
};

__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// a select by value (a conditional of two array elements would select between their addresses)
__device__ __forceinline__ float2 pick(int c, float2 a, float2 b) { return make_float2(c ? a.x : b.x, c ? a.y : b.y); }

// a lane's place in the two layouts.  renew() hides where the values came from, so that addresses and
// wave numbers of a later stage are computed there instead of being kept in registers from an
// earlier one (at 256 points that is the difference between no spills and a third of a plane)
struct PlaneLane {
  int yc, yt, zl, zt;
  bool y_on;
  __device__ __forceinline__ void renew() { asm volatile("" : "+v"(yc), "+v"(yt), "+v"(zl), "+v"(zt)); }
};
template <class K>
__device__ __forceinline__ PlaneLane plane_lane() {
  const int lane = (int)threadIdx.x & 63, wave = ((int)threadIdx.x >> 6) % K::W;
  PlaneLane L;
  L.yc = wave * 16 + (lane & 15);
  L.yt = lane >> 4;
  L.zl = wave * 32 + (lane & 31);
  L.zt = lane >> 5;
  L.y_on = K::W == K::WY || wave < K::WY;
  return L;
}

// Z layout from LDS: f[p-1] = X[2p - t] and g[p-1] = X[M - 2p + t], p = 1 .. H; the last pair of an
// even lane is (X[0], X[M/2]) instead.  C selects the component of a split plane.
template <class K, int C>
__device__ __forceinline__ void z_read(const float* lds, const PlaneLane& L, float2 (&f)[K::H], float2 (&g)[K::H]) {
  auto get = [&](int k, float2& d) {
    if constexpr (!K::SPLIT) {
      d = reinterpret_cast<const float2*>(lds)[L.zl * K::P + k];
    } else if constexpr (C == 0) {
      d.x = lds[L.zl * K::P + k];
    } else {
      d.y = lds[L.zl * K::P + k];
    }
  };
#pragma unroll
  for (int p = 1; p <= K::H; p++) {
    if (p < K::H)
      get(2 * p - L.zt, f[p - 1]);
    else
      get(L.zt ? K::RZ - 1 : 0, f[p - 1]);
    get(K::M - 2 * p + L.zt, g[p - 1]);
  }
}
template <class K, int C>
__device__ __forceinline__ void z_write(float* lds, const PlaneLane& L, const float2 (&f)[K::H], const float2 (&g)[K::H]) {
  auto put = [&](int k, float2 d) {
    if constexpr (!K::SPLIT)
      reinterpret_cast<float2*>(lds)[L.zl * K::P + k] = d;
    else
      lds[L.zl * K::P + k] = C == 0 ? d.x : d.y;
  };
#pragma unroll
  for (int p = 1; p <= K::H; p++) {
    if (p < K::H)
      put(2 * p - L.zt, f[p - 1]);
    else
      put(L.zt ? K::RZ - 1 : 0, f[p - 1]);
    put(K::M - 2 * p + L.zt, g[p - 1]);
  }
}
// a pointer that is the same in every lane, kept in scalar registers
template <int HP>
__device__ __forceinline__ GPtrT<HP> uniform(GPtrT<HP> g) {
  const uint64_t a = (uint64_t)g.p;
  const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)a);
  const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(a >> 32));
  return gptr<HP>((const void*)(((uint64_t)hi << 32) | lo));
}

// rows of 32-line groups outside the mask are zero: nothing is written for them, and they read as zero
template <class K, int C>
__device__ __forceinline__ void y_write(float* lds, const PlaneLane& L, unsigned mask, const float2 (&v)[K::RY]) {
#pragma unroll
  for (int g = 0; g < K::WZ; g++) {
    if (!(mask >> g & 1)) continue;
#pragma unroll
    for (int j = 8 * g; j < (8 * g + 8 < K::RY ? 8 * g + 8 : K::RY); j++) {
      const int i = L.yt * K::P + L.yc + 4 * j * K::P;
      if constexpr (!K::SPLIT)
        reinterpret_cast<float2*>(lds)[i] = v[j];
      else
        lds[i] = C == 0 ? v[j].x : v[j].y;
    }
  }
}
template <class K, int C>
__device__ __forceinline__ void y_read(const float* lds, const PlaneLane& L, unsigned mask, float2 (&v)[K::RY]) {
#pragma unroll
  for (int g = 0; g < K::WZ; g++) {
    const bool on = mask >> g & 1;
#pragma unroll
    for (int j = 8 * g; j < (8 * g + 8 < K::RY ? 8 * g + 8 : K::RY); j++) {
      const int i = L.yt * K::P + L.yc + 4 * j * K::P;
      if constexpr (!K::SPLIT)
        v[j] = on ? reinterpret_cast<const float2*>(lds)[i] : make_float2(0.0f, 0.0f);
      else if constexpr (C == 0)
        v[j].x = on ? lds[i] : 0.0f;
      else
        v[j].y = on ? lds[i] : 0.0f;
    }
  }
}

// turn the plane from the Y to the Z layout; no lane may still be reading the plane's LDS
template <class K>
__device__ __forceinline__ void turn_to_z(float* lds, const PlaneLane& L, unsigned mask, bool z_on, const float2 (&v)[K::RY], float2 (&f)[K::H],
                                          float2 (&g)[K::H]) {
  if (L.y_on) y_write<K, 0>(lds, L, mask, v);
  __syncthreads();
  if (z_on) z_read<K, 0>(lds, L, f, g);
  if constexpr (K::SPLIT) {
    __syncthreads();
    if (L.y_on) y_write<K, 1>(lds, L, mask, v);
    __syncthreads();
    if (z_on) z_read<K, 1>(lds, L, f, g);
  }
}
// and back; the wave's own lines must be free
template <class K>
__device__ __forceinline__ void turn_to_y(float* lds, const PlaneLane& L, unsigned mask, bool z_on, const float2 (&f)[K::H], const float2 (&g)[K::H],
                                          float2 (&v)[K::RY]) {
  if (z_on) z_write<K, 0>(lds, L, f, g);
  __syncthreads();
  if (L.y_on) y_read<K, 0>(lds, L, mask, v);
  if constexpr (K::SPLIT) {
    __syncthreads();
    if (z_on) z_write<K, 1>(lds, L, f, g);
    __syncthreads();
    if (L.y_on) y_read<K, 1>(lds, L, mask, v);
  }
}

// packed spectrum pairs -> z[n] = x[2n] + i x[2n+1] (unnormalized C2R), entries n = 2 j + t in z[j].
// With e = X[k] + conj X[M-k], d = X[k] - conj X[M-k], T = d e^{2 pi i k / n2}: Z'[k] = e + i T and
// Z'[M-k] = conj(e - i T).  tw2[k] = exp(-2 pi i k / n2).
template <class K>
__device__ __forceinline__ void z_inverse(float2 (&f)[K::H], float2 (&g)[K::H], float2 (&z)[K::RZ], int t,
                                          const float2* twm, const float2* tw2) {
  constexpr int H = K::H, R = K::RZ;
#pragma unroll
  for (int p = 1; p <= H; p++) {
    if (R >= 40 && p % 4 == 1) __builtin_amdgcn_sched_barrier(0);
    const float2 a = f[p - 1], b = g[p - 1];
    const float2 bc = cconj(b);
    const float2 e = cadd(a, bc), T = cmulc(csub(a, bc), tw2[2 * p - t]);
    float2 u = make_float2(e.x - T.y, e.y + T.x), w = make_float2(e.x + T.y, T.x - e.y);
    if (p == H) {  // even lanes: k = 0 (Re X[0] and Re X[M] packed) and k = M/2, its own mirror
      u = pick(t, u, make_float2(a.x + a.y, a.x - a.y));
      w = pick(t, w, make_float2(2.0f * b.x, -2.0f * b.y));
    }
    f[p - 1] = u;
    g[p - 1] = w;
  }
  // entry order: even lanes k = 2 j, odd lanes k = 2 j + 1
  z[0] = pick(t, f[0], f[H - 1]);
#pragma unroll
  for (int j = 1; j < H; j++) z[j] = pick(t, f[j], f[j - 1]);
#pragma unroll
  for (int p = 1; p <= H; p++) z[R - p] = g[p - 1];
  lane_fft<R, 2, +1>(z, t, twm);
}

// z[n] -> packed spectrum pairs of R2C, times 2 (the pointwise stage carries the factor 1/2)
template <class K>
__device__ __forceinline__ void z_forward(float2 (&z)[K::RZ], float2 (&f)[K::H], float2 (&g)[K::H], int t,
                                          const float2* twm, const float2* tw2) {
  constexpr int H = K::H, R = K::RZ;
  lane_fft<R, 2, -1>(z, t, twm);
#pragma unroll
  for (int p = 1; p <= H; p++) {
    if (R >= 40 && p % 4 == 1) __builtin_amdgcn_sched_barrier(0);
    const float2 a = pick(t, z[p - 1], z[p < H ? p : 0]);
    const float2 b = z[R - p];
    const float2 bc = cconj(b);
    // e + (-i d) w and the conjugate of e - (-i d) w
    const float2 e = cadd(a, bc), o = cmul(mul_mi(csub(a, bc)), tw2[2 * p - t]);
    float2 u = cadd(e, o), w = cconj(csub(e, o));
    if (p == H) {
      u = pick(t, u, make_float2(2.0f * (a.x + a.y), 2.0f * (a.x - a.y)));
      w = pick(t, w, make_float2(2.0f * b.x, -2.0f * b.y));
    }
    f[p - 1] = u;
    g[p - 1] = w;
  }
}

// wave number of row 4 j + t (wnum without branches: j is known at compile time)
template <int N1>
__device__ __forceinline__ float y_wave(int j, int t) {
  constexpr int h = N1 / 8;  // j of the Nyquist row
  const float w = (float)t + (float)(4 * j - (j >= h ? N1 : 0));
  return j == h ? (t ? w : 0.0f) : w;
}

// the block's twiddle tables in LDS (after its data loads are issued): lane_fft's for n1 and n2/2, and
// exp(-2 pi i k / n2)
template <class K, int N1>
__device__ __forceinline__ void stage_plane_twiddles(float2* ty, float2* tm, float2* t2, const float2* __restrict__ tw1,
                                                     const float2* __restrict__ twm, const float2* __restrict__ tw2) {
  for (int i = threadIdx.x; i < N1; i += K::TB) ty[i] = tw1[(i & 3) * (i >> 2)];
  for (int i = threadIdx.x; i < K::M; i += K::TB) {
    tm[i] = twm[(i & 1) * (i >> 1)];
    t2[i] = tw2[i];
  }
  __syncthreads();
}

// A real field on the plane, read in the Z layout: the wave's 32 lines are loaded in order, put into
// its own LDS rows and read back as pairs.  A split plane's rows hold half a line at a time.
// real_fetch issues the loads of one part, real_use hands the pairs of that part to fn(j, pair).
template <class K>
struct RealPart {
  static constexpr int PARTS = K::SPLIT ? 4 : 1;
  static constexpr int PM = K::M / PARTS;        // pairs per line and part
  static constexpr int CNT = 32 * PM / 64;       // pairs per lane and part
};
// The lane number for a part's addresses.  On 256 lines of 160 reals the quotients by a part's 20 pairs a
// line, kept from one part to the next beside 64 values a lane, spilled 170 registers: it is renewed there and
// they are made again, 77 spills (CN solves of 4 x 160 x 256 x 160 with a scan's zeros 9.85 -> 9.32 ms, with a
// coefficient zero nowhere 6.46 -> 6.03).  With fewer values a lane it costs 2%, at 24 pairs a line it is even.
template <class K>
__device__ __forceinline__ int part_lane() {
  using RP = RealPart<K>;
  int lane = (int)threadIdx.x & 63;
  if constexpr (RP::PARTS > 1 && RP::PM % 8 != 0 && K::RY == 64) asm volatile("" : "+v"(lane));
  return lane;
}
template <class K, int PART, int HP>
__device__ __forceinline__ void real_fetch(float2 (&q)[RealPart<K>::CNT], GPtrT<HP> field, const PlaneLane& L) {
  using RP = RealPart<K>;
  const int lane = part_lane<K>();
  const int wave = __builtin_amdgcn_readfirstlane(L.zl >> 5);
  const auto f0 = field + (wave * 32 * K::M + PART * RP::PM);
#pragma unroll
  for (int i = 0; i < RP::CNT; i++) {
    const unsigned e = (unsigned)(i * 64 + lane), row = e / RP::PM;
    if (K::LINES % 32 != 0 && wave * 32 + (int)row >= K::LINES) {
      q[i] = make_float2(0.0f, 0.0f);
    } else if constexpr (RP::PARTS == 1) {  // the wave's lines are one run
      q[i] = (f0 + i * 64)[(unsigned)lane];
    } else {
      q[i] = f0[row * K::M + e % RP::PM];
    }
  }
}
template <class K, int PART, class Fn>
__device__ __forceinline__ void real_use(float* lds, const float2 (&q)[RealPart<K>::CNT], const PlaneLane& L, Fn fn) {
  using RP = RealPart<K>;
  const int lane = part_lane<K>();
  const int l0 = L.zl & ~31;
  wave_fence();  // the wave's earlier reads of its rows come first
#pragma unroll
  for (int i = 0; i < RP::CNT; i++) {
    const int e = i * 64 + lane, row = l0 + e / RP::PM, n = e % RP::PM;
    if constexpr (!K::SPLIT) {
      reinterpret_cast<float2*>(lds)[row * K::P + n] = q[i];
    } else {
      lds[row * K::P + 2 * n] = q[i].x;
      lds[row * K::P + 2 * n + 1] = q[i].y;
    }
  }
  wave_fence();
  constexpr int J = K::RZ / RP::PARTS;
#pragma unroll
  for (int j = 0; j < J; j++) {
    const int n = 2 * j + L.zt;
    float2 r;
    if constexpr (!K::SPLIT) {
      r = reinterpret_cast<const float2*>(lds)[L.zl * K::P + n];
    } else {
      r.x = lds[L.zl * K::P + 2 * n];
      r.y = lds[L.zl * K::P + 2 * n + 1];
    }
    fn(PART * J + j, r);
  }
}

// the whole field on a split plane, part by part: the next part's loads are in flight while one part
// is staged and used (8 x 256^3 matvec middle: 1086 us with one part in flight, 892 us with two)
template <class K, int HP, class Fn>
__device__ __forceinline__ void real_stream(float* lds, GPtrT<HP> field, PlaneLane& L, Fn fn) {
  using RP = RealPart<K>;
  static_assert(RP::PARTS == 4, "four parts");
  float2 a[RP::CNT], b[RP::CNT];
  __builtin_amdgcn_sched_barrier(0);
  L.renew();
  real_fetch<K, 0>(a, field, L);
  real_fetch<K, 1>(b, field, L);
  real_use<K, 0>(lds, a, L, fn);
  __builtin_amdgcn_sched_barrier(0);
  real_fetch<K, 2>(a, field, L);
  real_use<K, 1>(lds, b, L, fn);
  __builtin_amdgcn_sched_barrier(0);
  real_fetch<K, 3>(b, field, L);
  real_use<K, 2>(lds, a, L, fn);
  __builtin_amdgcn_sched_barrier(0);
  real_use<K, 3>(lds, b, L, fn);
  __builtin_amdgcn_sched_barrier(0);
}

// The plane sizes built: sides within a factor of two.  Beyond that most of a block's waves would sit
// idle in one of the layouts (at 256 x 64, two of eight waves hold the columns).
#define GLIA_PLANES(X)                                                                        \
  X(32, 32) X(32, 64) X(48, 32) X(48, 64) X(48, 96) X(64, 32) X(64, 64) X(64, 96) X(64, 128)  \
  X(80, 64) X(80, 96) X(80, 128) X(80, 160) X(96, 64) X(96, 96) X(96, 128) X(96, 160) X(96, 192) \
  X(128, 64) X(128, 96) X(128, 128) X(128, 160) X(128, 192) X(128, 256)                       \
  X(160, 96) X(160, 128) X(160, 160) X(160, 192) X(160, 256)                                  \
  X(192, 96) X(192, 128) X(192, 160) X(192, 192) X(192, 256)                                  \
  X(256, 128) X(256, 160) X(256, 192) X(256, 256)

template <template <int, int> class F, typename... Args>
static int dispatch_plane(const Dims& d, Args&&... args) {
#define GLIA_PLANE_CASE(A, B) \
  if (d.n1 == A && d.n2 == B) return F<A, B>::run(args...);
  GLIA_PLANES(GLIA_PLANE_CASE)
#undef GLIA_PLANE_CASE
  return -1;
}

}  // namespace glia
