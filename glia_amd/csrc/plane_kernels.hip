// plane_kernels.hip -- the diffusion operator's Y and Z passes fused over x-planes (plane_fft.h).
//
// What bounds it: at 128 points the vector units (about 4200 instructions a lane and component, 65% of
// the issue slots; two blocks a CU).  From 160 points a CU holds ten or fewer waves (registers), too
// few to cover a block's loads and stores with arithmetic.  Measured against the three passes it
// replaces, matvec middle of one CG iteration with every member active: 16 x 128^3 450 -> 193 us,
// 8 x 160^3 424 -> 252, 8 x 192^3 726 -> 442, 8 x 256^3 1761 -> 882 (17 fields of traffic became 6).
// Whole CN solves of one and five members on 32, 96 and 256 x n1 x n2 grids, a scan's ellipsoid in the box: 1.16
// times as fast in the mean, 0.99 (one member, 32 x 256 x 192) to 1.35 (5 x 256 x 128 x 128).  With a coefficient
// that is zero nowhere 1.06 in the mean, 0.84 (5 x 256 x 160 x 96) to 1.23: pairs of sides where one layout leaves
// waves idle lose there.  The sides alone decide: the host does not know k, and members of an ensemble with
// different zeros must give the bits they give alone.
#include "plane_fft.h"

namespace glia {
using namespace dev;

// Which 32-line groups of each x-plane hold a nonzero of the real slot k_slot (bit g: lines 32 g ..),
// for the matvec's plane pass: where k is zero the product is zero, so a plane or group without a
// nonzero needs no transform.  k vanishes outside the brain, half or more of a scan's box.  Computed
// anew for every solve (the field may have changed), in the launch that starts it.
__global__ void __launch_bounds__(256) k_plane_mask(const MemberDev* __restrict__ mem, Dims d, int k_slot, int begin,
                                                    double tau) {
  const MemberDev& M = mem[blockIdx.y];
  if (begin && blockIdx.x == 0 && threadIdx.x == 0) pcg_begin_state(M.st, tau);
  const unsigned n4 = (unsigned)(32 * d.n2 / 4), all = (unsigned)(d.n1 * d.n2 / 4);  // 16-byte words: group, plane
  const v4f* f = reinterpret_cast<const v4f*>(M.r[k_slot] + (int64_t)blockIdx.x * d.n1 * d.n2);
  unsigned mask = 0;
  for (int g = 0; 32 * g < d.n1; g++) {
    int any = 0;
    const unsigned end = (g + 1) * n4 < all ? (g + 1) * n4 : all;
    for (unsigned i = g * n4 + threadIdx.x; i < end; i += 256) {
      const v4f x = f[i];
      any |= !(x.x == 0.0f && x.y == 0.0f && x.z == 0.0f && x.w == 0.0f);
    }
    if (__syncthreads_or(any)) mask |= 1u << g;
  }
  if (threadIdx.x == 0) M.kmask[blockIdx.x] = mask;
}

// the planes with a nonzero as one bit each, for the X passes around the plane pass
__global__ void __launch_bounds__(64) k_plane_bits(const MemberDev* __restrict__ mem, Dims d) {
  const MemberDev& M = mem[blockIdx.x];
  for (int i = 0; i < 4; i++) {
    const int x = 64 * i + (int)threadIdx.x;
    const unsigned long long b = __ballot(x < d.n0 && M.kmask[x] != 0);
    if (threadIdx.x == 0) {
      M.planes[2 * i] = (unsigned)b;
      M.planes[2 * i + 1] = (unsigned)(b >> 32);
    }
  }
}

// Middle of the matvec on one plane and component: h = k * grad_d p on the grid, transformed back
// along z and y.  From U and V (inverse X pass of p and of i w_x p):
//   component x: out = F_yz(k F_yz^-1 V)                 y: out = i w_y F_yz(k F_yz^-1 (i w_y U))
//   component z: out = i w_z F_yz(k F_yz^-1 (i w_z U))
// One block per plane and component, the three components of a plane on one XCD (blocks go to the 8
// XCDs round-robin), which share the k and U planes in its L2.
template <int N1, int N2>
__global__ void __launch_bounds__((PL<N1, N2>::TB), (PL<N1, N2>::MINW))
k_plane_diff(const MemberDev* __restrict__ mem, Dims d, const float2* __restrict__ tw1, const float2* __restrict__ twm,
             const float2* __restrict__ tw2, int s_u, int s_v, int s_x, int s_y, int s_z, int k_slot,
             int use_planes) {
  using K = PL<N1, N2>;
  using RP = RealPart<K>;
  const MemberDev& Mb = mem[blockIdx.y];
  if (Mb.st->done) return;
  __shared__ float lds_[K::CH][K::LDS];
  __shared__ float2 ty[N1], tm[K::M], t2[K::M];
  // eight plane groups (one per XCD) times three components, CH planes a group
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), ch = wave / K::W;
  const int q = (int)blockIdx.x >> 3;
  const int comp = q % 3, plane = ((q / 3) * 8 + ((int)blockIdx.x & 7)) * K::CH + ch;
  float* lds = lds_[ch];
  const unsigned mask = (unsigned)__builtin_amdgcn_readfirstlane((int)Mb.kmask[plane]);
  const bool z_on = mask >> (wave - ch * K::W) & 1;
  const int64_t base = (int64_t)plane * N1 * K::M;
  const auto in = uniform(cptr<0>(Mb, comp == 0 ? s_v : s_u) + base);
  const auto out = uniform(cptr<0>(Mb, comp == 0 ? s_x : (comp == 1 ? s_y : s_z)) + base);
  const auto kf = uniform(rptr2<0>(Mb, k_slot) + base);
  PlaneLane L = plane_lane<K>();
  // nothing to transform (the block's other plane, if any, included: with one plane to do, the other's
  // rows read as zero below and give zeros)
  if (mask == 0 && (K::CH == 1 || Mb.kmask[plane ^ 1] == 0)) {
    if (L.y_on && !use_planes) {  // otherwise the X pass does not read these rows
#pragma unroll 4
      for (int j = 0; j < K::RY; j++) (out + 4 * j * K::M)[(unsigned)(L.yt * K::M + L.yc)] = make_float2(0.0f, 0.0f);
    }
    return;
  }
  float2 v[K::RY];
  float2 kq[RP::CNT];
  if (L.y_on) {
#pragma unroll
    for (int j = 0; j < K::RY; j++) v[j] = (in + 4 * j * K::M)[(unsigned)(L.yt * K::M + L.yc)];
  }
  if (!K::SPLIT && z_on) real_fetch<K, 0>(kq, kf, L);
  stage_plane_twiddles<K, N1>(ty, tm, t2, tw1, twm, tw2);
  if (L.y_on) {
    if (comp == 1) {
#pragma unroll
      for (int j = 0; j < K::RY; j++) v[j] = mul_i(cscale(v[j], y_wave<N1>(j, L.yt)));
    } else if (comp == 2) {
#pragma unroll
      for (int j = 0; j < K::RY; j++) v[j] = mul_i(cscale(v[j], (float)L.yc));
    }
    lane_fft<K::RY, 4, +1>(v, L.yt, ty);
  }
  float2 f[K::H], g[K::H];
  L.renew();
  turn_to_z<K>(lds, L, mask, z_on, v, f, g);
  L.renew();
  if (z_on) {
    float2 z[K::RZ];
    z_inverse<K>(f, g, z, L.zt, tm, t2);
    const float s = (float)(0.5 * d.inv_ng);
    auto mul = [&](int j, float2 k) { z[j] = make_float2(z[j].x * (k.x * s), z[j].y * (k.y * s)); };
    if constexpr (K::SPLIT) {
      real_stream<K>(lds, kf, L, mul);
    } else {
      real_use<K, 0>(lds, kq, L, mul);
    }
    L.renew();
    z_forward<K>(z, f, g, L.zt, tm, t2);
    wave_fence();
  }
  L.renew();
  turn_to_y<K>(lds, L, mask, z_on, f, g, v);
  L.renew();
  if (L.y_on) {
    lane_fft<K::RY, 4, -1>(v, L.yt, ty);
    const unsigned o0 = (unsigned)(L.yt * K::M + L.yc);
    if (comp == 0) {
#pragma unroll
      for (int j = 0; j < K::RY; j++) (out + 4 * j * K::M)[o0] = v[j];
    } else if (comp == 1) {
#pragma unroll
      for (int j = 0; j < K::RY; j++) (out + 4 * j * K::M)[o0] = mul_i(cscale(v[j], y_wave<N1>(j, L.yt)));
    } else {
#pragma unroll
      for (int j = 0; j < K::RY; j++) (out + 4 * j * K::M)[o0] = mul_i(cscale(v[j], (float)L.yc));
    }
  }
}

// ---------------------------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------------------------
bool plane_supported(const Dims& d) {
  if (d.n0 % 16 != 0) return false;
#define GLIA_PLANE_CASE(A, B) \
  if (d.n1 == A && d.n2 == B) return true;
  GLIA_PLANES(GLIA_PLANE_CASE)
#undef GLIA_PLANE_CASE
  return false;
}

template <int N1, int N2>
struct RunPlaneDiff {
  static int run(const LaunchCtx& c, int s_u, int s_v, int s_x, int s_y, int s_z, int k_slot) {
    k_plane_diff<N1, N2><<<dim3(3 * c.d.n0 / PL<N1, N2>::CH, c.nm), PL<N1, N2>::TB, 0, c.stream>>>(c.mem, c.d, c.tw1, c.twm, c.tw2, s_u, s_v,
                                                                              s_x, s_y, s_z, k_slot, c.use_planes);
    return (int)hipGetLastError();
  }
};
int launch_plane_diff(const LaunchCtx& c, int s_u, int s_v, int s_x, int s_y, int s_z, int k_slot) {
  return dispatch_plane<RunPlaneDiff>(c.d, c, s_u, s_v, s_x, s_y, s_z, k_slot);
}
int launch_plane_mask(const LaunchCtx& c, int k_slot, bool begin, double tau) {
  k_plane_mask<<<dim3(c.d.n0, c.nm), 256, 0, c.stream>>>(c.mem, c.d, k_slot, begin ? 1 : 0, tau);
  if (c.use_planes) k_plane_bits<<<c.nm, 64, 0, c.stream>>>(c.mem, c.d);
  return (int)hipGetLastError();
}

}  // namespace glia
