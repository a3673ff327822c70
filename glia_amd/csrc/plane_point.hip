// plane_point.hip -- passes of the elasticity solver fused over x-planes (plane_fft.h).  Each takes the
// place of a Y pass and a Z pass (two of them around a product with a real field), and reads and writes
// its spectrum once instead of two or three times.
//
// Bound as the diffusion operator's plane pass: the vector units up to 128 points, the few waves a CU
// holds beyond; and at 160^3 and below by the number of blocks, three planes for each of n0.  160^3, one
// CG iteration: the three strain channels 197 -> 140 us, p's update and transform 59 -> 50, the screened
// output 68 -> 65, the preconditioner's output 53 -> 51, x and r's update and transform 79 -> 87
// (two rounds of blocks).  Whole solves: 32^3 5.41 -> 4.32 ms, 64^3 7.13 -> 5.92, 96^3 16.2 -> 12.6, 128^3 23.8 ->
// 20.3, 160^3 50.9 -> 46.6, 192^3 82.6 -> 77.5, 256^3 138 -> 130, 96 x 128 x 64 14.0 -> 12.0.
#include "plane_fft.h"

#include <type_traits>

namespace glia {
using namespace dev;

// the one-way kernels need fewer registers and take one plane a block
template <int N1, int N2>
struct PL1 : PL<N1, N2> {
  static constexpr int CH = 1, TB = PL<N1, N2>::T;
  static constexpr int MINW = 2;
  // Where more waves hold the lines than the columns at 40 entries a lane, 192 x 160 and 256 x 160, the separate
  // passes are the faster ones as soon as a launch takes a second round (128 x 192 x 160, a CG iteration 666
  // against 691 us, 192 x 192 x 160 934 against 1015; 80 x 256 x 160, one round, 605 against 570).
  using Q = PL<N1, N2>;
  static constexpr bool ONE_ROUND = Q::WZ > Q::WY && Q::RZ == 40;
};

// Whether a launch of this many blocks fills the chip well enough to beat the separate passes.  Up to four
// waves a plane several blocks share a CU and it always does.  From five on a CU runs one block at a time, so
// a launch takes whole rounds of 256 blocks: a last round that leaves the launch under two thirds full loses
// (96 planes of three lanes are 288 blocks in two rounds: 96 x 256 x 192 920 -> 857 us a CG iteration without
// the fused passes there, 96 x 128 x 256 626 -> 586), and so do fewer than 96 blocks of eight or ten waves
// (the one-lane coefficient pass at 64 x 256 x 256: 12 us over the separate passes).
template <class K>
static bool fills(int blocks) {
  const int rounds = (blocks + 255) / 256;
  return K::W <= 4 || ((K::W * K::CH < 8 || blocks >= 96) && (rounds == 1 || 3 * blocks >= 2 * 256 * rounds));
}

// block, plane and lane of the three kernels: CH planes a block, in order
template <class K>
struct PlaneOf {
  int wave, ch, plane;
  __device__ __forceinline__ PlaneOf() {
    wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    ch = wave / K::W;
    wave -= ch * K::W;
    plane = (int)blockIdx.x * K::CH + ch;
  }
};
template <class K, int HP>
__device__ __forceinline__ void y_load(GPtrT<HP> in, const PlaneLane& L, float2 (&v)[K::RY]) {
  if (!L.y_on) return;
#pragma unroll
  for (int j = 0; j < K::RY; j++) v[j] = (in + 4 * j * K::M)[(unsigned)(L.yt * K::M + L.yc)];
}
template <class K, int HP>
__device__ __forceinline__ void y_store(GPtrT<HP> out, const PlaneLane& L, const float2 (&v)[K::RY]) {
  if (!L.y_on) return;
#pragma unroll
  for (int j = 0; j < K::RY; j++) (out + 4 * j * K::M)[(unsigned)(L.yt * K::M + L.yc)] = v[j];
}

// all 32-line groups
template <class K>
constexpr unsigned kAllLines = (1u << K::WZ) - 1;

// out = F_yz(m F_yz^-1 in), m the real slot r_slot (a Lame coefficient times a strain term); in place
// when s_out is s_in
template <int N1, int N2>
__global__ void __launch_bounds__((PL<N1, N2>::TB), (PL<N1, N2>::MINW))
k_plane_coef(const MemberDev* __restrict__ mem, Dims d, const float2* __restrict__ tw1, const float2* __restrict__ twm,
             const float2* __restrict__ tw2, int s_in, int s_out, int r_slot, int honor) {
  using K = PL<N1, N2>;
  using RP = RealPart<K>;
  const MemberDev& Mb = mem[blockIdx.y];
  if (honor && Mb.st->done) return;
  __shared__ float lds_[K::CH][K::LDS];
  __shared__ float2 ty[N1], tm[K::M], t2[K::M];
  const PlaneOf<K> B;
  float* lds = lds_[B.ch];
  const bool z_on = B.wave < K::WZ;
  const int64_t base = (int64_t)B.plane * N1 * K::M;
  const auto mf = uniform(rptr2<0>(Mb, r_slot) + base);
  PlaneLane L = plane_lane<K>();
  float2 v[K::RY];
  float2 kq[RP::CNT];
  y_load<K>(uniform(cptr<0>(Mb, s_in) + base), L, v);
  if (!K::SPLIT && z_on) real_fetch<K, 0>(kq, mf, L);
  stage_plane_twiddles<K, N1>(ty, tm, t2, tw1, twm, tw2);
  if (L.y_on) lane_fft<K::RY, 4, +1>(v, L.yt, ty);
  float2 f[K::H], g[K::H];
  L.renew();
  turn_to_z<K>(lds, L, kAllLines<K>, z_on, v, f, g);
  L.renew();
  if (z_on) {
    float2 z[K::RZ];
    z_inverse<K>(f, g, z, L.zt, tm, t2);
    const float s = (float)(0.5 * d.inv_ng);
    auto mul = [&](int j, float2 m) { z[j] = make_float2(z[j].x * (m.x * s), z[j].y * (m.y * s)); };
    if constexpr (K::SPLIT) {
      real_stream<K>(lds, mf, L, mul);
    } else {
      real_use<K, 0>(lds, kq, L, mul);
    }
    L.renew();
    z_forward<K>(z, f, g, L.zt, tm, t2);
    wave_fence();
  }
  L.renew();
  turn_to_y<K>(lds, L, kAllLines<K>, z_on, f, g, v);
  L.renew();
  if (L.y_on) lane_fft<K::RY, 4, -1>(v, L.yt, ty);
  y_store<K>(uniform(cptr<0>(Mb, s_out) + base), L, v);
}

// Pairs a lane takes together: they divide its share of a part.  The last wave of 48 or 80 lines has half of
// its lines, which are the first half of every lane's pairs: it takes half of the groups (skipping the lines
// past the last one by one made every load a branch: 96 x 80 x 160, a CG iteration 447 -> 339 us).
template <class K>
struct PairGroup {
  static constexpr int CNT = RealPart<K>::CNT, LAST = K::LINES % 32 ? CNT / 2 : CNT;
  static constexpr int value = LAST % 8 == 0 ? 8 : (LAST % 6 == 0 ? 6 : (LAST % 5 == 0 ? 5 : 4));
  static_assert(LAST % value == 0, "a lane's pairs come in whole groups");
  static_assert(K::LINES % 32 == 0 || (K::LINES % 32 == 16 && CNT % 2 == 0 && RealPart<K>::PM % 4 == 0),
                "half of the last wave's lines are half of every lane's pairs");
  static __device__ __forceinline__ int count(int wave) { return wave == K::WZ - 1 ? LAST : CNT; }
};
// A group of the pairs of one part of the wave's lines in memory order: fn(i, offset in the plane, LDS
// index of the pair), i < PairGroup.
template <class K, int PART, class Fn>
__device__ __forceinline__ void line_pairs(int wave, int i0, Fn fn) {
  using RP = RealPart<K>;
  const int lane = (int)threadIdx.x & 63;
#pragma unroll
  for (int i = 0; i < PairGroup<K>::value; i++) {
    const int e = (i0 + i) * 64 + lane, row = wave * 32 + e / RP::PM, n = e % RP::PM;
    fn(i, (unsigned)(row * K::M + PART * RP::PM + n), K::SPLIT ? row * K::P + 2 * n : row * K::P + n);
  }
}
template <class K>
__device__ __forceinline__ void put_pair(float* lds, int at, float2 x) {
  if constexpr (!K::SPLIT) {
    reinterpret_cast<float2*>(lds)[at] = x;
  } else {
    lds[at] = x.x;
    lds[at + 1] = x.y;
  }
}
template <class K>
__device__ __forceinline__ float2 get_pair(const float* lds, int at) {
  if constexpr (!K::SPLIT) return reinterpret_cast<const float2*>(lds)[at];
  else return make_float2(lds[at], lds[at + 1]);
}
// LDS index of entry n = 2 j + t of this lane's line within its part
template <class K, int PART>
__device__ __forceinline__ int z_pair_at(const PlaneLane& L, int j) {
  const int n = 2 * j + L.zt - PART * RealPart<K>::PM;
  return K::SPLIT ? L.zl * K::P + 2 * n : L.zl * K::P + n;
}
// fn(std::integral_constant part) over the parts
template <class K, class Fn>
__device__ __forceinline__ void each_part(Fn fn) {
  fn(std::integral_constant<int, 0>{});
  if constexpr (RealPart<K>::PARTS == 4) {
    fn(std::integral_constant<int, 1>{});
    fn(std::integral_constant<int, 2>{});
    fn(std::integral_constant<int, 3>{});
  }
}

// real output c = F_yz^-1 in / N^3:
//   PO_SCREEN: r_out = c - a u with a in RS_RHO and u the real slot r_b; block partials of <u, r_out>
//   PO_DOT   : r_out = c; block partials of <c, c> and <c, r>, r the real slot r_b
enum { PO_SCREEN = 0, PO_DOT = 1 };
template <int N1, int N2, int MODE>
__global__ void __launch_bounds__((PL1<N1, N2>::TB), (PL1<N1, N2>::MINW))
k_plane_out(const MemberDev* __restrict__ mem, Dims d, const float2* __restrict__ tw1, const float2* __restrict__ twm,
            const float2* __restrict__ tw2, int s_in, int r_out, int r_b, int honor) {
  using K = PL1<N1, N2>;
  using RP = RealPart<K>;
  const MemberDev& Mb = mem[blockIdx.y];
  if (honor && Mb.st->done) return;
  __shared__ float lds_[K::CH][K::LDS];
  __shared__ float2 ty[N1], tm[K::M], t2[K::M];
  const PlaneOf<K> B;
  float* lds = lds_[B.ch];
  const bool z_on = B.wave < K::WZ;
  const int64_t base = (int64_t)B.plane * N1 * K::M;
  const auto out = uniform(rptr2<2>(Mb, r_out) + base);
  const auto pa = uniform(rptr2<0>(Mb, RS_RHO) + base), pb = uniform(rptr2<0>(Mb, r_b) + base);
  PlaneLane L = plane_lane<K>();
  float2 v[K::RY];
  y_load<K>(uniform(cptr<0>(Mb, s_in) + base), L, v);
  stage_plane_twiddles<K, N1>(ty, tm, t2, tw1, twm, tw2);
  if (L.y_on) lane_fft<K::RY, 4, +1>(v, L.yt, ty);
  float2 f[K::H], g[K::H];
  L.renew();
  turn_to_z<K>(lds, L, kAllLines<K>, z_on, v, f, g);
  L.renew();
  double acc[2] = {0.0, 0.0};
  if (z_on) {
    float2 z[K::RZ];
    z_inverse<K>(f, g, z, L.zt, tm, t2);
    const float s = (float)d.inv_ng;
    constexpr int J = K::RZ / RP::PARTS;
    each_part<K>([&](auto part) {
      constexpr int PART = decltype(part)::value;
      __builtin_amdgcn_sched_barrier(0);
      L.renew();
      wave_fence();
#pragma unroll
      for (int j = PART * J; j < PART * J + J; j++) put_pair<K>(lds, z_pair_at<K, PART>(L, j), cscale(z[j], s));
      wave_fence();
      constexpr int C = PairGroup<K>::value;
#pragma unroll 1
      for (int i0 = 0; i0 < PairGroup<K>::count(B.wave); i0 += C) {
        float2 a[C], b[C];
        line_pairs<K, PART>(B.wave, i0, [&](int i, unsigned at, int) {
          if (MODE == PO_SCREEN) a[i] = pa[at];
          b[i] = pb[at];
        });
        line_pairs<K, PART>(B.wave, i0, [&](int i, unsigned at, int la) {
          const float2 c = get_pair<K>(lds, la);
          if (MODE == PO_SCREEN) {
            const float2 w = make_float2(c.x - a[i].x * b[i].x, c.y - a[i].y * b[i].y);
            out[at] = w;
            acc[0] += (double)b[i].x * (double)w.x + (double)b[i].y * (double)w.y;
          } else {
            out[at] = c;
            acc[0] += (double)c.x * (double)c.x + (double)c.y * (double)c.y;
            acc[1] += (double)c.x * (double)b[i].x + (double)c.y * (double)b[i].y;
          }
        });
      }
    });
  }
  if (MODE == PO_SCREEN) {
    double a1[1] = {acc[0]};
    block_reduce_store<1>(a1, Mb.part + blockIdx.x);
  } else {
    block_reduce_store<2>(acc, Mb.part + (int64_t)blockIdx.x * 2);
  }
}

// spectrum of a real field that is first updated in place (the elasticity CG's vector work; the scalars
// and the rules are k_z_upd_r2c's):
//   PI_AXPBY: p = z + b p, out = F_yz p                       [ra = p, rb = z]
//   PI_CGUPD: x += t p, r -= t w, out = F_yz r                [ra = x, rb = r, rc = p, rd = w]
enum { PI_AXPBY = 0, PI_CGUPD = 1 };
template <int N1, int N2, int MODE>
__global__ void __launch_bounds__((PL1<N1, N2>::TB), (PL1<N1, N2>::MINW))
k_plane_in(const MemberDev* __restrict__ mem, Dims d, const float2* __restrict__ tw1, const float2* __restrict__ twm,
           const float2* __restrict__ tw2, int ra, int rb, int rc, int rd, const double* __restrict__ sc, int s_out,
           int honor) {
  using K = PL1<N1, N2>;
  using RP = RealPart<K>;
  const MemberDev& Mb = mem[blockIdx.y];
  if (honor && Mb.st->done) return;
  __shared__ float lds_[K::CH][K::LDS];
  __shared__ float2 ty[N1], tm[K::M], t2[K::M];
  const PlaneOf<K> B;
  float* lds = lds_[B.ch];
  const bool z_on = B.wave < K::WZ;
  const int64_t base = (int64_t)B.plane * N1 * K::M;
  const CgStep cg = cg_step<MODE == PI_CGUPD>(mem[0].st, sc);
  const auto A = uniform(rptr2<2>(Mb, ra) + base), R = uniform(rptr2<2>(Mb, rb) + base);
  const auto C = uniform(rptr2<0>(Mb, MODE == PI_CGUPD ? rc : ra) + base);
  const auto D = uniform(rptr2<0>(Mb, MODE == PI_CGUPD ? rd : rb) + base);
  PlaneLane L = plane_lane<K>();
  stage_plane_twiddles<K, N1>(ty, tm, t2, tw1, twm, tw2);
  float2 f[K::H], g[K::H];
  if (z_on) {
    float2 z[K::RZ];
    constexpr int J = K::RZ / RP::PARTS;
    each_part<K>([&](auto part) {
      constexpr int PART = decltype(part)::value;
      __builtin_amdgcn_sched_barrier(0);
      L.renew();
      wave_fence();
      constexpr int G = PairGroup<K>::value;
#pragma unroll 1
      for (int i0 = 0; i0 < PairGroup<K>::count(B.wave); i0 += G) {
        float2 q0[G], q1[G], q2[G], q3[G];
        line_pairs<K, PART>(B.wave, i0, [&](int i, unsigned at, int) {
          q0[i] = R[at];
          if (MODE == PI_AXPBY) {
            if (cg.upd) q1[i] = A[at];
          } else if (cg.upd) {
            q1[i] = A[at];
            q2[i] = C[at];
            q3[i] = D[at];
          }
        });
        line_pairs<K, PART>(B.wave, i0, [&](int i, unsigned at, int la) {
          float2 x = q0[i];
          if (MODE == PI_AXPBY) {
            if (cg.upd) x = make_float2(x.x + cg.t * q1[i].x, x.y + cg.t * q1[i].y);
            A[at] = x;
          } else if (cg.upd) {
            A[at] = make_float2(q1[i].x + cg.t * q2[i].x, q1[i].y + cg.t * q2[i].y);
            x = make_float2(x.x - cg.t * q3[i].x, x.y - cg.t * q3[i].y);
            R[at] = x;
          }
          put_pair<K>(lds, la, cscale(x, 0.5f));  // z_forward doubles
        });
      }
      wave_fence();
#pragma unroll
      for (int j = PART * J; j < PART * J + J; j++) z[j] = get_pair<K>(lds, z_pair_at<K, PART>(L, j));
    });
    L.renew();
    z_forward<K>(z, f, g, L.zt, tm, t2);
    wave_fence();
  }
  float2 v[K::RY];
  L.renew();
  turn_to_y<K>(lds, L, kAllLines<K>, z_on, f, g, v);
  L.renew();
  if (L.y_on) lane_fft<K::RY, 4, -1>(v, L.yt, ty);
  y_store<K>(uniform(cptr<0>(Mb, s_out) + base), L, v);
}

// ---------------------------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------------------------
int plane_blocks(const Dims& d) { return d.n0; }  // of the one-way kernels
template <int N1, int N2>
struct PlaneCoefFills {
  static int run(const LaunchCtx& c) { return fills<PL<N1, N2>>(c.nm * c.d.n0 / PL<N1, N2>::CH) ? 1 : 0; }
};
bool plane_coef_fills(const LaunchCtx& c) { return dispatch_plane<PlaneCoefFills>(c.d, c) == 1; }

template <int N1, int N2>
struct PlaneIoFills {
  // cgupd: the x and r update reads four fields and writes two, so little is left to gain but the launch;
  // one full round takes it, or two (192 x 256 x 192, three rounds: 49 us an iteration over the separate
  // passes; 160 x 96 x 160, 480 blocks: 13 us under them)
  static int run(const LaunchCtx& c, bool cgupd) {
    using K = PL1<N1, N2>;
    const int blocks = c.nm * c.d.n0;
    const bool few = blocks <= 256 || (blocks >= 448 && blocks <= 512);
    if (K::ONE_ROUND && blocks > 256) return 0;
    return fills<K>(blocks) && (!cgupd || K::W <= 4 || few) ? 1 : 0;
  }
};
bool plane_out_fills(const LaunchCtx& c) { return dispatch_plane<PlaneIoFills>(c.d, c, false) == 1; }
bool plane_in_fills(const LaunchCtx& c, int mode) {
  return dispatch_plane<PlaneIoFills>(c.d, c, mode == ZUM_CGUPD) == 1;
}

template <int N1, int N2>
struct RunPlaneCoef {
  static int run(const LaunchCtx& c, int s_in, int s_out, int r_slot, int honor) {
    const dim3 g(c.d.n0 / PL<N1, N2>::CH, c.nm);
    k_plane_coef<N1, N2><<<g, PL<N1, N2>::TB, 0, c.stream>>>(c.mem, c.d, c.tw1, c.twm, c.tw2, s_in, s_out, r_slot, honor);
    return (int)hipGetLastError();
  }
};
int launch_plane_coef(const LaunchCtx& c, int s_in, int s_out, int r_slot, bool honor_done) {
  return dispatch_plane<RunPlaneCoef>(c.d, c, s_in, s_out, r_slot, honor_done ? 1 : 0);
}

template <int N1, int N2>
struct RunPlaneOut {
  static int run(const LaunchCtx& c, int mode, int s_in, int r_out, int r_b, int honor) {
    const dim3 g(c.d.n0, c.nm);
    if (mode == ZPM_SCREEN)
      k_plane_out<N1, N2, PO_SCREEN><<<g, PL1<N1, N2>::TB, 0, c.stream>>>(c.mem, c.d, c.tw1, c.twm, c.tw2, s_in, r_out,
                                                                         r_b, honor);
    else if (mode == ZPM_C2R_DOT)
      k_plane_out<N1, N2, PO_DOT><<<g, PL1<N1, N2>::TB, 0, c.stream>>>(c.mem, c.d, c.tw1, c.twm, c.tw2, s_in, r_out, r_b,
                                                                      honor);
    else
      return -1;
    return (int)hipGetLastError();
  }
};
int launch_plane_out(const LaunchCtx& c, int mode, int s_in, int r_out, int r_b, bool honor_done) {
  return dispatch_plane<RunPlaneOut>(c.d, c, mode, s_in, r_out, r_b, honor_done ? 1 : 0);
}

template <int N1, int N2>
struct RunPlaneIn {
  static int run(const LaunchCtx& c, int mode, int ra, int rb, int rc, int rd, const double* sc, int s_out, int honor) {
    const dim3 g(c.d.n0, c.nm);
    if (mode == ZUM_AXPBY)
      k_plane_in<N1, N2, PI_AXPBY><<<g, PL1<N1, N2>::TB, 0, c.stream>>>(c.mem, c.d, c.tw1, c.twm, c.tw2, ra, rb, rc, rd, sc,
                                                                       s_out, honor);
    else if (mode == ZUM_CGUPD)
      k_plane_in<N1, N2, PI_CGUPD><<<g, PL1<N1, N2>::TB, 0, c.stream>>>(c.mem, c.d, c.tw1, c.twm, c.tw2, ra, rb, rc, rd, sc,
                                                                       s_out, honor);
    else
      return -1;
    return (int)hipGetLastError();
  }
};
int launch_plane_in(const LaunchCtx& c, int mode, int ra, int rb, int rc, int rd, const double* sc, int s_out,
                    bool honor_done) {
  if (mode == ZUM_CGUPD && !sc) return -1;
  return dispatch_plane<RunPlaneIn>(c.d, c, mode, ra, rb, rc, rd, sc, s_out, honor_done ? 1 : 0);
}

}  // namespace glia
