// lj_force_n3.hip -- the force pass with every unordered pair evaluated once
// (Newton's third law), for the FP32 and compensated modes of single boxes
// (k_force_n3, k_force_n3c) and for batches (k_batch_force_n3).
//
// Physics as the reference's pair loop (MDSystem.cu:21-138, MDSystem.cpp:
// 260-309); only the order of evaluation differs.
//
// Decomposition.  The particles form groups of G = 128 W (W = 4: 512, W = 2:
// 256).  A work item is a pair of groups (g, h), h >= g, run by one workgroup
// of W x W waves: wave (wi, wj) takes the 128 particles G g + 128 wi + [0, 128)
// as i (two per lane) and the 128 particles G h + 128 wj + [0, 128) as j.
//   * The j particles sit in LDS, stored twice in a row, so that at step t
//     lane l reads j = (l + t) mod 64 of a 64-particle sub-tile with a plain
//     immediate offset; after 64 steps every lane has met every j.
//   * i sums (force, (s/r)^6, (s/r)^6 (2 (s/r)^6 - 1)) stay in registers.
//   * j sums (minus the force, (s/r)^6 - w) travel with their j particle:
//     after each step every lane passes its j sums to the next lower lane
//     (ds_bpermute), so no atomics are involved and every sum is taken in a
//     fixed order (bit-reproducible results).
//   * Diagonal items (g == h): waves with wi < wj evaluate their tile pair
//     once as above, waves with wi == wj evaluate both orders of their own
//     tile (i sums only, self pair excluded by index), waves with wi > wj
//     are idle.  The time step's variant (W = 2) instead takes the diagonal
//     items two to a workgroup with every pair once (n3_diag_pair), so that
//     every workgroup carries the same work.
//   * Small items (groups of 128, W = 1; sizes whose items of 256 fill few of the
//     resident workgroups, n3_small_groups): the four waves of a workgroup
//     share one tile pair, each taking one 64-particle j sub-tile and half of its
//     64 steps, so the same pairs run on four times the waves.
// Output slots.  Particle p of group a receives exactly one entry per group s:
// s > a from the i side of item (a, s), s < a from the j side of item (s, a),
// s == a from the diagonal item.  The partial buffers are therefore the
// [S = groups][Npad] layout of the sliced kernel and the reduction and
// integrator kernels are shared (the time step's entries are the three force
// components only, store_part3).  Entry encoding (fx, fy, fz, bf) + af with
// e = (bf - af)/2 and W = 12 eps sum bf, as for the sliced kernel:
//   i side of a once-evaluated pair: bf = 2 b, af = b + a;
//   j side:                          bf = 0,   af = sum ((s/r)^6 - w);
//   both orders (self tile):         bf = b,   af = a.
// The time-step variant's loop is 24 VALU instructions per unordered pair
// (12.4 per ordered pair over the whole kernel, measured) against 21.5 per
// ordered pair for the sliced kernel, which evaluates each pair twice.
#include <algorithm>
#include <cstdlib>

#include "lj_device.h"

namespace lj {

namespace {

using namespace dev;

constexpr int kTile = 128;  // particles per wave tile
constexpr int kAccPerWave = 2 * 4 * 64;  // sub-tiles x components x tile

// LDS of one workgroup, declared once by each kernel: the diagonal-pair
// workgroups of the time step use the same bytes with their own layout
template <int W>
struct N3Lds {
  static constexpr int kG = kTile * W;
  static constexpr int kAcc = W * W * kAccPerWave > W * 5 * kG ? W * W * kAccPerWave : W * 5 * kG;
  uint4 pos[W * 2 * 128];  // [wj][sub-tile][doubled 64]
  // j sums [wave][sub-tile][component][64], then i sums [wj][component][G]
  float acc[kAcc];
  double ew[W * W][2];
};

// the pair's factors from its separation; returns r2
template <bool GUARD>
__device__ __forceinline__ float factors(float dx, float dy, float dz, float C1, bool ok, float& s,
                                         float& e6, float& w)
{
  const float r2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
  float ir2 = __builtin_amdgcn_rcpf(r2) * C1;
  if constexpr (GUARD) ir2 = ok ? ir2 : 0.f;
  e6 = ir2 * ir2 * ir2;
  w = e6 * __builtin_fmaf(e6, 2.f, -1.f);
  s = w * ir2;
  return r2;
}

template <bool PERIODIC, bool TIES, bool GUARD>
__device__ __forceinline__ void terms(const PosT<PERIODIC>& pi, const uint4& pj, float C1, bool ok,
                                      float& dx, float& dy, float& dz, float& s, float& e6,
                                      float& w)
{
  if constexpr (PERIODIC) {
    dx = mi_fixed<TIES>(pi.x, pj.x);
    dy = mi_fixed<TIES>(pi.y, pj.y);
    dz = mi_fixed<TIES>(pi.z, pj.z);
  } else {
    dx = pi.x - __uint_as_float(pj.x);
    dy = pi.y - __uint_as_float(pj.y);
    dz = pi.z - __uint_as_float(pj.z);
  }
  factors<GUARD>(dx, dy, dz, C1, ok, s, e6, w);
}

// The pairs with r2 <= thr, or not comparable, that a pass leaves out (EXCL):
// kLook notes the least r2 on the way (half an instruction a pair), kTest leaves
// them out pair by pair.
enum { kNone = 0, kLook = 1, kTest = 2 };
struct Excl {
  float thr, least;
};

// A lane's particle as the i of a pair.  Periodic boxes with exact ties take the
// mirrored frame (MirPos): no compare and select per axis, but the j side, whose
// sums travel through lanes of other frames, needs the frame's sign: g = -s_a,
// one select an axis (a full evaluation at N = 16384: 131 us with the
// compares and selects of the unmirrored form, 124 so).
template <bool PERIODIC, bool TIES>
struct SideI {
  LaneI<PERIODIC, TIES> li;
  __device__ __forceinline__ explicit SideI(const PosT<PERIODIC>& p) { li.set(p); }
  // separation and factors of the pair with pj, where ok (GUARD); returns r2
  template <bool GUARD, int EXCL>
  __device__ __forceinline__ float meet(const uint4& pj, float C1, float thr, bool ok, float& dx,
                                        float& dy, float& dz, float& s, float& e6, float& w) const
  {
    PosT<PERIODIC> p;
    if constexpr (PERIODIC) p.x = pj.x, p.y = pj.y, p.z = pj.z;
    else p.x = __uint_as_float(pj.x), p.y = __uint_as_float(pj.y), p.z = __uint_as_float(pj.z);
    sep(li.p, p, dx, dy, dz);
    if constexpr (EXCL == kTest)
      ok = ok && __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx)) > thr;
    return factors<GUARD || EXCL == kTest>(dx, dy, dz, C1, ok, s, e6, w);
  }
  // j sums minus this pair's force, from the frame
  __device__ __forceinline__ void react(float dx, float dy, float dz, float s, float& jx, float& jy,
                                        float& jz) const
  {
    jx = __builtin_fmaf(dx, li.p.mx ? -s : s, jx);
    jy = __builtin_fmaf(dy, li.p.my ? -s : s, jy);
    jz = __builtin_fmaf(dz, li.p.mz ? -s : s, jz);
  }
};

// rotate a value one lane down the wave: lane l receives lane (l + 1) mod 64.
// ds_bpermute does the gather in the LDS unit, off the VALU that bounds the
// pair loop: a DPP move (wave_rol:1, and row_ror alike) cost about 2.5 VALU
// issue slots here, and the kernel ran 92.6 us with it against 77.8 us with
// the permute (N = 16384, time-step variant, same box).  The LDS unit is nearly
// idle in the loop (one read per step), and the permute's latency overlaps the
// next step's i-side work.  Every lane of the wave must be active: the pair
// loops run with a full execution mask.
__device__ __forceinline__ float rot1(float v)
{
  const int lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  return __int_as_float(__builtin_amdgcn_ds_bpermute(((lane + 1) & 63) << 2, __float_as_int(v)));
}

// STEPS steps from t0 on of one j sub-tile P (64 particles, doubled): i sums in
// a1/a2 (in the lanes' frames), the j sums in j[] travelling with their j particle
template <bool PERIODIC, bool TIES, bool PARTIAL, bool ENERGY, int EXCL, int STEPS>
__device__ __forceinline__ void pair_steps(const uint4* P, int t0, int lane,
                                           const SideI<PERIODIC, TIES>& i1,
                                           const SideI<PERIODIC, TIES>& i2, bool v1, bool v2,
                                           float C1, Excl& ex, Acc& a1, Acc& a2, float (&j)[4])
{
  float jx = 0.f, jy = 0.f, jz = 0.f, jm = 0.f;
#pragma unroll 8
  for (int t = 0; t < STEPS; ++t) {
    const uint4 pj = P[lane + t0 + t];
    bool ok1 = true, ok2 = true;
    if constexpr (PARTIAL) {
      const bool jv = pj.w != 0u;
      ok1 = v1 && jv;
      ok2 = v2 && jv;
    }
    float dx1, dy1, dz1, s1, e1, w1, dx2, dy2, dz2, s2, e2, w2;
    const float r1 = i1.template meet<PARTIAL, EXCL>(pj, C1, ex.thr, ok1, dx1, dy1, dz1, s1, e1, w1);
    const float r2 = i2.template meet<PARTIAL, EXCL>(pj, C1, ex.thr, ok2, dx2, dy2, dz2, s2, e2, w2);
    if constexpr (EXCL == kLook) ex.least = __builtin_fminf(ex.least, __builtin_fminf(r1, r2));
    a1.fx = __builtin_fmaf(dx1, s1, a1.fx);
    a1.fy = __builtin_fmaf(dy1, s1, a1.fy);
    a1.fz = __builtin_fmaf(dz1, s1, a1.fz);
    a1.a += e1;
    a1.b += w1;
    a2.fx = __builtin_fmaf(dx2, s2, a2.fx);
    a2.fy = __builtin_fmaf(dy2, s2, a2.fy);
    a2.fz = __builtin_fmaf(dz2, s2, a2.fz);
    a2.a += e2;
    a2.b += w2;
    if constexpr (PERIODIC && TIES) {
      i1.react(dx1, dy1, dz1, s1, jx, jy, jz);
      i2.react(dx2, dy2, dz2, s2, jx, jy, jz);
    } else {
      jx = __builtin_fmaf(-dx2, s2, __builtin_fmaf(-dx1, s1, jx));
      jy = __builtin_fmaf(-dy2, s2, __builtin_fmaf(-dy1, s1, jy));
      jz = __builtin_fmaf(-dz2, s2, __builtin_fmaf(-dz1, s1, jz));
    }
    jx = rot1(jx);
    jy = rot1(jy);
    jz = rot1(jz);
    if constexpr (ENERGY) {
      jm += (e1 - w1) + (e2 - w2);
      jm = rot1(jm);
    }
  }
  j[0] = jx;
  j[1] = jy;
  j[2] = jz;
  j[3] = jm;
}

// One tile pair evaluated once, sub-tiles [0, nsub) of 64 j (SUBS = 2) or one
// (SUBS = 1), STEPS steps from t0 on each; i sums in a1/a2; j sums in registers
// that travel with their j particle (lane l holds the sums of j slot (l + t) mod
// 64 at step t and passes them to lane l - 1 afterwards), so after 64 steps lane
// l holds those of slot l.  J receives (-fx, -fy, -fz, sum (s/r)^6 - w) per
// sub-tile.
// nsub: sub-tiles holding a valid j (1 when the second one is past N)
template <bool PERIODIC, bool TIES, bool PARTIAL, bool ENERGY, int EXCL = kNone, int SUBS = 2,
          int STEPS = 64>
__device__ __forceinline__ void pair_tile(const uint4* P0, int lane, const PosT<PERIODIC>& pi1,
                                          const PosT<PERIODIC>& pi2, bool v1, bool v2, float C1,
                                          int nsub, Acc& a1, Acc& a2, float (&J)[SUBS][4],
                                          float thr = 0.f, int t0 = 0)
{
  const SideI<PERIODIC, TIES> i1(pi1), i2(pi2);
  Excl ex{thr, __builtin_inff()};
#pragma unroll
  for (int st = 0; st < SUBS; ++st) {
    if (st >= nsub) break;  // wave-uniform
    pair_steps<PERIODIC, TIES, PARTIAL, ENERGY, EXCL, STEPS>(P0 + st * 128, t0, lane, i1, i2, v1, v2,
                                                             C1, ex, a1, a2, J[st]);
  }
  if constexpr (EXCL == kLook) {
    // a pair to leave out shows in the least r2 or, with an r2 that is not a
    // number, in the sums: the tile is then taken again pair by pair, the same
    // sums without those pairs
    const bool bad = !(ex.least > thr) || a1.a != a1.a || a1.b != a1.b || a2.a != a2.a || a2.b != a2.b;
    if (__any(bad)) {
      acc_zero(a1);
      acc_zero(a2);
      for (int st = 0; st < SUBS; ++st) {
        if (st >= nsub) break;
        pair_steps<PERIODIC, TIES, true, ENERGY, kTest, STEPS>(P0 + st * 128, t0, lane, i1, i2, v1,
                                                               v2, C1, ex, a1, a2, J[st]);
      }
    }
  }
  i1.li.common_frame(a1);
  i2.li.common_frame(a2);
}

// both orders of the wave's own tile, i sums only, self pair (and with EXCL
// those to leave out) excluded; sub-tiles and steps as in pair_tile
template <bool PERIODIC, bool TIES, int EXCL = kNone, int SUBS = 2, int STEPS = 64>
__device__ __forceinline__ void self_tile(const uint4* P0, int lane, int i1, int i2, int jbase,
                                          const PosT<PERIODIC>& pi1, const PosT<PERIODIC>& pi2,
                                          bool v1, bool v2, float C1, int nsub, Acc& a1, Acc& a2,
                                          float thr = 0.f, int t0 = 0)
{
  const SideI<PERIODIC, TIES> s1(pi1), s2(pi2);
#pragma unroll
  for (int st = 0; st < SUBS; ++st) {
    if (st >= nsub) break;  // wave-uniform
    const uint4* P = P0 + st * 128;
#pragma unroll 8
    for (int t = 0; t < STEPS; ++t) {
      const int jx = lane + t0 + t;
      const uint4 pj = P[jx];
      const int j = jbase + st * 64 + (jx & 63);
      const bool jv = pj.w != 0u;
      const bool ok1 = v1 && jv && j != i1;
      const bool ok2 = v2 && jv && j != i2;
      float dx, dy, dz, s, e, w;
      s1.template meet<true, EXCL ? kTest : kNone>(pj, C1, thr, ok1, dx, dy, dz, s, e, w);
      a1.fx = __builtin_fmaf(dx, s, a1.fx);
      a1.fy = __builtin_fmaf(dy, s, a1.fy);
      a1.fz = __builtin_fmaf(dz, s, a1.fz);
      a1.a += e;
      a1.b += w;
      s2.template meet<true, EXCL ? kTest : kNone>(pj, C1, thr, ok2, dx, dy, dz, s, e, w);
      a2.fx = __builtin_fmaf(dx, s, a2.fx);
      a2.fy = __builtin_fmaf(dy, s, a2.fy);
      a2.fz = __builtin_fmaf(dz, s, a2.fz);
      a2.a += e;
      a2.b += w;
    }
  }
  s1.li.common_frame(a1);
  s2.li.common_frame(a2);
}

// rotate by k lanes: lane l receives lane (l + k) mod 64 (full execution mask)
__device__ __forceinline__ float rotk(float v, int k)
{
  const int lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  return __int_as_float(__builtin_amdgcn_ds_bpermute(((lane + k) & 63) << 2, __float_as_int(v)));
}

__device__ __forceinline__ void acc_two_sum(Acc& hi, Acc& lo, const Acc& x)
{
  two_sum(hi.fx, lo.fx, x.fx);
  two_sum(hi.fy, lo.fy, x.fy);
  two_sum(hi.fz, lo.fz, x.fz);
  two_sum(hi.a, lo.a, x.a);
  two_sum(hi.b, lo.b, x.b);
}

// Compensated mode (LJ_PREC_COMPENSATED): the sums of pair_tile in blocks of
// kJB = 32 pairs in FP32, each block added into a (hi, lo) pair by TwoSum, as
// the sliced kernel's j_range does.
//   i side: the lane's i meets one j per step, so a block is 32 steps; the
//   block sums go into (a1, l1) / (a2, l2) at t = 32 and t = 64.
//   j side: the travelling sums meet two i per step, so a block is 16 steps.
//   The (hi, lo) pairs of the j slots stay in their lanes between folds: at
//   the fold after step t = 16 k - 1 lane l's block holds slot (l + 16 k) mod
//   64 and its (hi, lo) slot (l + 16 (k - 1)), so the pairs are first rotated
//   by 16 lanes.  After the fold at t = 64 lane l holds slot l, as in
//   pair_tile.  The i (hi, lo) are added into a1 / a2 by the caller.
template <bool PERIODIC, bool TIES, bool PARTIAL, bool ENERGY>
__device__ __forceinline__ void pair_tile_c(const uint4* P0, int lane, const PosT<PERIODIC>& pi1,
                                            const PosT<PERIODIC>& pi2, bool v1, bool v2, float C1,
                                            int nsub, Acc& a1, Acc& a2, Acc& l1, Acc& l2,
                                            float (&J)[2][4])
{
  constexpr int NJ = ENERGY ? 4 : 3;
#pragma unroll
  for (int st = 0; st < 2; ++st) {
    if (st >= nsub) break;  // wave-uniform
    const uint4* P = P0 + st * 128;
    float jh[4] = {0.f, 0.f, 0.f, 0.f}, jl[4] = {0.f, 0.f, 0.f, 0.f};
    Acc b1, b2;
    acc_zero(b1);
    acc_zero(b2);
#pragma unroll 1
    for (int qt = 0; qt < 4; ++qt) {  // quarters of 16 steps
      float jb[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
      for (int u = 0; u < 16; ++u) {
        const uint4 pj = P[lane + 16 * qt + u];
        bool ok1 = true, ok2 = true;
        if constexpr (PARTIAL) {
          const bool jv = pj.w != 0u;
          ok1 = v1 && jv;
          ok2 = v2 && jv;
        }
        float dx1, dy1, dz1, s1, e1, w1, dx2, dy2, dz2, s2, e2, w2;
        terms<PERIODIC, TIES, PARTIAL>(pi1, pj, C1, ok1, dx1, dy1, dz1, s1, e1, w1);
        terms<PERIODIC, TIES, PARTIAL>(pi2, pj, C1, ok2, dx2, dy2, dz2, s2, e2, w2);
        b1.fx = __builtin_fmaf(dx1, s1, b1.fx);
        b1.fy = __builtin_fmaf(dy1, s1, b1.fy);
        b1.fz = __builtin_fmaf(dz1, s1, b1.fz);
        b1.a += e1;
        b1.b += w1;
        b2.fx = __builtin_fmaf(dx2, s2, b2.fx);
        b2.fy = __builtin_fmaf(dy2, s2, b2.fy);
        b2.fz = __builtin_fmaf(dz2, s2, b2.fz);
        b2.a += e2;
        b2.b += w2;
        jb[0] = rot1(__builtin_fmaf(-dx2, s2, __builtin_fmaf(-dx1, s1, jb[0])));
        jb[1] = rot1(__builtin_fmaf(-dy2, s2, __builtin_fmaf(-dy1, s1, jb[1])));
        jb[2] = rot1(__builtin_fmaf(-dz2, s2, __builtin_fmaf(-dz1, s1, jb[2])));
        if constexpr (ENERGY) jb[3] = rot1(jb[3] + ((e1 - w1) + (e2 - w2)));
      }
#pragma unroll
      for (int c = 0; c < NJ; ++c) {
        // (the first fold rotates zeros)
        jh[c] = rotk(jh[c], 16);
        jl[c] = rotk(jl[c], 16);
        two_sum(jh[c], jl[c], jb[c]);
      }
      if (qt & 1) {  // the end of a 32-step block of the i sums
        acc_two_sum(a1, l1, b1);
        acc_two_sum(a2, l2, b2);
        acc_zero(b1);
        acc_zero(b2);
      }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) J[st][c] = c < NJ ? jh[c] + jl[c] : 0.f;
  }
}

// Compensated form of self_tile: the i sums in blocks of 32 steps, each
// added into (a, l) by TwoSum
template <bool PERIODIC, bool TIES>
__device__ __forceinline__ void self_tile_c(const uint4* P0, int lane, int i1, int i2, int jbase,
                                            const PosT<PERIODIC>& pi1, const PosT<PERIODIC>& pi2,
                                            bool v1, bool v2, float C1, int nsub, Acc& a1, Acc& a2,
                                            Acc& l1, Acc& l2)
{
#pragma unroll
  for (int st = 0; st < 2; ++st) {
    if (st >= nsub) break;  // wave-uniform
    const uint4* P = P0 + st * 128;
#pragma unroll 1
    for (int half = 0; half < 2; ++half) {
      Acc b1, b2;
      acc_zero(b1);
      acc_zero(b2);
#pragma unroll 8
      for (int t = 32 * half; t < 32 * half + 32; ++t) {
        const int jx = lane + t;
        const uint4 pj = P[jx];
        const int j = jbase + st * 64 + (jx & 63);
        const bool jv = pj.w != 0u;
        const bool ok1 = v1 && jv && j != i1;
        const bool ok2 = v2 && jv && j != i2;
        float dx, dy, dz, s, e, w;
        terms<PERIODIC, TIES, true>(pi1, pj, C1, ok1, dx, dy, dz, s, e, w);
        b1.fx = __builtin_fmaf(dx, s, b1.fx);
        b1.fy = __builtin_fmaf(dy, s, b1.fy);
        b1.fz = __builtin_fmaf(dz, s, b1.fz);
        b1.a += e;
        b1.b += w;
        terms<PERIODIC, TIES, true>(pi2, pj, C1, ok2, dx, dy, dz, s, e, w);
        b2.fx = __builtin_fmaf(dx, s, b2.fx);
        b2.fy = __builtin_fmaf(dy, s, b2.fy);
        b2.fz = __builtin_fmaf(dz, s, b2.fz);
        b2.a += e;
        b2.b += w;
      }
      acc_two_sum(a1, l1, b1);
      acc_two_sum(a2, l2, b2);
    }
  }
}

__device__ __forceinline__ void encode(const Acc& a, int cls, float (&v)[5])
{
  v[0] = a.fx;
  v[1] = a.fy;
  v[2] = a.fz;
  if (cls == 1) {  // once-evaluated pairs
    v[3] = 2.f * a.b;
    v[4] = a.b + a.a;
  } else {
    v[3] = a.b;
    v[4] = a.a;
  }
}

// One step of two once-evaluated pair streams of a wave: the lane's i particle
// pi1 meets j slot (lane + t) mod 64 of sub-tile P1, pi2 that of P2 (LDS,
// doubled).  R1 / R2 hold the sums of those j slots (minus the force) and pass
// one lane down afterwards, as in pair_tile.  GUARD: pairs count only with a
// valid i (vi1, vi2) and j, and with HALF only on lanes 0-31 (the step t = 32
// of a triangle, where lanes l and l + 32 meet the same pair).
template <bool PERIODIC, bool GUARD, bool HALF>
__device__ __forceinline__ void dual_step(const uint4* P1, const uint4* P2, int lane, int t,
                                          const PosT<PERIODIC>& pi1, const PosT<PERIODIC>& pi2,
                                          bool vi1, bool vi2, float C1, float (&a1)[3],
                                          float (&a2)[3], float& ea, float& eb, float (&R1)[3],
                                          float (&R2)[3])
{
  const uint4 pj1 = P1[lane + t], pj2 = P2[lane + t];
  bool ok1 = true, ok2 = true;
  if constexpr (GUARD) {
    const bool h = !HALF || lane < 32;
    ok1 = vi1 && pj1.w != 0u && h;
    ok2 = vi2 && pj2.w != 0u && h;
  }
  float dx1, dy1, dz1, s1, e1, w1, dx2, dy2, dz2, s2, e2, w2;
  terms<PERIODIC, false, GUARD>(pi1, pj1, C1, ok1, dx1, dy1, dz1, s1, e1, w1);
  terms<PERIODIC, false, GUARD>(pi2, pj2, C1, ok2, dx2, dy2, dz2, s2, e2, w2);
  a1[0] = __builtin_fmaf(dx1, s1, a1[0]);
  a1[1] = __builtin_fmaf(dy1, s1, a1[1]);
  a1[2] = __builtin_fmaf(dz1, s1, a1[2]);
  a2[0] = __builtin_fmaf(dx2, s2, a2[0]);
  a2[1] = __builtin_fmaf(dy2, s2, a2[1]);
  a2[2] = __builtin_fmaf(dz2, s2, a2[2]);
  ea += e1 + e2;
  eb += w1 + w2;
  R1[0] = rot1(__builtin_fmaf(-dx1, s1, R1[0]));
  R1[1] = rot1(__builtin_fmaf(-dy1, s1, R1[1]));
  R1[2] = rot1(__builtin_fmaf(-dz1, s1, R1[2]));
  R2[0] = rot1(__builtin_fmaf(-dx2, s2, R2[0]));
  R2[1] = rot1(__builtin_fmaf(-dy2, s2, R2[1]));
  R2[2] = rot1(__builtin_fmaf(-dz2, s2, R2[2]));
}

// The pairs inside each 64-particle sub-tile of two sub-tiles at once
// (triangles): at step t = 1..32 lane l meets slot (l + t) mod 64, so every
// unordered pair of the sub-tile is met once (t = 32 on lanes 0-31 only).
// Afterwards lane l holds the j sums of slot (l + 33) mod 64.
// The loops of these two-stream steps advance two steps per iteration: with
// more the compiler reads further ahead from LDS and, at the 64 registers that
// eight waves per SIMD allow, spilled to scratch (the whole kernel then ran
// with a private segment).
template <bool PERIODIC, bool GUARD>
__device__ __forceinline__ void tri_pair(const uint4* P1, const uint4* P2, int lane,
                                         const PosT<PERIODIC>& pi1, const PosT<PERIODIC>& pi2,
                                         bool vi1, bool vi2, float C1, float (&a1)[3],
                                         float (&a2)[3], float& ea, float& eb, float (&R1)[3],
                                         float (&R2)[3])
{
#pragma nounroll
  for (int c = 0; c < 16; ++c) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int t = 2 * c + u + 1;
      if (u == 1 && c == 15)
        dual_step<PERIODIC, true, true>(P1, P2, lane, t, pi1, pi2, vi1, vi2, C1, a1, a2, ea, eb, R1,
                                                  R2);
      else
        dual_step<PERIODIC, GUARD, false>(P1, P2, lane, t, pi1, pi2, vi1, vi2, C1, a1, a2, ea, eb, R1,
                                                  R2);
    }
  }
}

// Every unordered pair of one group of 256 that the pair tile of its diagonal
// item leaves out (those inside sub-tiles 0-3 and between sub-tiles 0-1 and
// 2-3), once, by one wave; f[k] receives the sums of the lane's particle of
// sub-tile k (particles base + 64 k + [0, 64), at P + 128 k).  ea / eb: the
// wave's sums of (s/r)^6 and w.
//   1. triangles of sub-tiles 1 and 3; their i and (aligned) j sums become
//      the starting j sums of
//   2. sub-tile 0 x sub-tile 1 and sub-tile 2 x sub-tile 3 (64 steps), after
//      which lane l holds the totals of slot l of sub-tiles 1 and 3;
//   3. triangles of sub-tiles 0 and 2, adding to the i sums of step 2.
template <bool PERIODIC, bool GUARD>
__device__ __forceinline__ void tri_tiles(const uint4* P, const uint4* __restrict__ q,
                                          const float4* __restrict__ pf, int base, int N, float C1,
                                          int lane, float (&f)[4][3], float& ea, float& eb)
{
  const int i0 = base + lane;
  const bool v0 = i0 < N, v1 = i0 + 64 < N, v2 = i0 + 128 < N, v3 = i0 + 192 < N;
  {
    const PosT<PERIODIC> pi1 = load_pos<PERIODIC>(q, pf, v1 ? i0 + 64 : N - 1);
    const PosT<PERIODIC> pi3 = load_pos<PERIODIC>(q, pf, v3 ? i0 + 192 : N - 1);
    float h1[3] = {0.f, 0.f, 0.f}, h3[3] = {0.f, 0.f, 0.f};
    tri_pair<PERIODIC, GUARD>(P + 128, P + 384, lane, pi1, pi3, v1, v3, C1, f[1], f[3], ea, eb, h1,
                              h3);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      f[1][c] += rotk(h1[c], 31);
      f[3][c] += rotk(h3[c], 31);
    }
  }
  const PosT<PERIODIC> pi0 = load_pos<PERIODIC>(q, pf, v0 ? i0 : N - 1);
  const PosT<PERIODIC> pi2 = load_pos<PERIODIC>(q, pf, v2 ? i0 + 128 : N - 1);
#pragma unroll 2
  for (int t = 0; t < 64; ++t)
    dual_step<PERIODIC, GUARD, false>(P + 128, P + 384, lane, t, pi0, pi2, v0, v2, C1, f[0], f[2],
                                      ea, eb, f[1], f[3]);
  float h0[3] = {0.f, 0.f, 0.f}, h2[3] = {0.f, 0.f, 0.f};
  tri_pair<PERIODIC, GUARD>(P, P + 256, lane, pi0, pi2, v0, v2, C1, f[0], f[2], ea, eb, h0, h2);
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    f[0][c] += rotk(h0[c], 31);
    f[2][c] += rotk(h2[c], 31);
  }
}

// Two diagonal items (A, A) and (B, B) of the time step's variant (W = 2) in
// one workgroup, every unordered pair of a group once: waves 0 / 1 pair the
// first 128 particles of A / B with the last 128 (pair_tile), waves 2 / 3 take
// the remaining pairs of A / B (tri_tiles) and pass their sums through LDS to
// waves 0 / 1, which add them to their own and write slot A / B of the
// group's particles.  All four waves carry the same work, so with the off-diagonal items a group count of 64 gives
// 2016 + 32 = 2048 equal workgroups, as many as are resident at once (eight
// 4-wave workgroups per CU): the 2080 items of the other decomposition leave
// 32 for a second round.  B < 0: A alone (waves 1 and 3 idle).
template <bool PERIODIC>
__device__ __forceinline__ void n3_diag_pair(N3Lds<2>& lds, const uint4* __restrict__ q,
                                             const float4* __restrict__ pf,
                                             float4* __restrict__ fpart, double* __restrict__ ew,
                                             int N, int Npad, float C1, int A, int B)
{
  static_assert(sizeof(N3Lds<2>::acc) >= 512 * sizeof(uint4), "group B's positions fit in acc");
  const int T = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(T >> 6);
  const int lane = T & 63;
  uint4* const posA = lds.pos;                            // [sub-tile][doubled 64]
  uint4* const posB = reinterpret_cast<uint4*>(lds.acc);  // same layout
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int grp = r ? B : A;
    if (grp < 0) continue;
    const int j = 256 * grp + T;
    const int jl = j < N ? j : 0;
    uint4 p;
    if constexpr (PERIODIC) {
      p = q[jl];
    } else {
      const float4 f = pf[jl];
      p = make_uint4(__float_as_uint(f.x), __float_as_uint(f.y), __float_as_uint(f.z), 0u);
    }
    p.w = j < N ? 1u : 0u;
    uint4* d = (r ? posB : posA) + (T >> 6) * 128;
    d[T & 63] = p;
    d[(T & 63) + 64] = p;
  }
  __syncthreads();

  const int grp = (wave & 1) ? B : A;
  const uint4* P = (wave & 1) ? posB : posA;
  const int base = 256 * grp;
  const bool partial = base + 256 > N;
  double se = 0., sw = 0.;
  // per lane: the sums of its particle of sub-tile k = 0..3 of the group
  float f[4][3] = {{0.f, 0.f, 0.f}, {0.f, 0.f, 0.f}, {0.f, 0.f, 0.f}, {0.f, 0.f, 0.f}};
  if (grp >= 0) {
    if (wave < 2) {
      const int i1 = base + lane, i2 = i1 + 64, jt0 = base + 128;
      if (jt0 < N) {  // the last 128 hold a particle
        const bool v1 = i1 < N, v2 = i2 < N;
        const PosT<PERIODIC> pi1 = load_pos<PERIODIC>(q, pf, v1 ? i1 : N - 1);
        const PosT<PERIODIC> pi2 = load_pos<PERIODIC>(q, pf, v2 ? i2 : N - 1);
        Acc a1, a2;
        acc_zero(a1);
        acc_zero(a2);
        float J[2][4] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
        if (partial)
          pair_tile<PERIODIC, false, true, false>(P + 256, lane, pi1, pi2, v1, v2, C1,
                                                  jt0 + 64 < N ? 2 : 1, a1, a2, J);
        else
          pair_tile<PERIODIC, false, false, false>(P + 256, lane, pi1, pi2, v1, v2, C1, 2, a1, a2,
                                                   J);
        f[0][0] = a1.fx, f[0][1] = a1.fy, f[0][2] = a1.fz;
        f[1][0] = a2.fx, f[1][1] = a2.fy, f[1][2] = a2.fz;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          f[2][c] = J[0][c];
          f[3][c] = J[1][c];
        }
        se = (double)a1.a + (double)a2.a;
        sw = (double)a1.b + (double)a2.b;
      }
    } else {
      float ea = 0.f, eb = 0.f;
      if (partial)
        tri_tiles<PERIODIC, true>(P, q, pf, base, N, C1, lane, f, ea, eb);
      else
        tri_tiles<PERIODIC, false>(P, q, pf, base, N, C1, lane, f, ea, eb);
      se = (double)ea;
      sw = (double)eb;
    }
  }
  // the triangle waves' sums to the pair-tile waves through LDS (the position
  // tiles are free once every wave is done): [group][sub-tile][component][64]
  float* const tri = reinterpret_cast<float*>(lds.pos);
  static_assert(sizeof(lds.pos) + sizeof(lds.acc) >= 2 * 4 * 3 * 64 * sizeof(float), "room");
  __syncthreads();
  if (wave >= 2 && grp >= 0) {
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int c = 0; c < 3; ++c) tri[(((wave & 1) * 4 + k) * 3 + c) * 64 + lane] = f[k][c];
  }
  __syncthreads();
  if (wave < 2 && grp >= 0) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float* t = tri + ((wave * 4 + k) * 3) * 64 + lane;
      if (base + 64 * k + lane < N)
        store_part3(fpart, (size_t)grp * Npad + base + 64 * k + lane, f[k][0] + t[0],
                    f[k][1] + t[64], f[k][2] + t[128]);
    }
  }
  // totals in the ordered-pair convention: every pair here was met once
  double te = sw - se, tw = 2. * sw;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    te += __shfl_xor(te, o, 64);
    tw += __shfl_xor(tw, o, 64);
  }
  if (lane == 0) {
    lds.ew[wave][0] = te;
    lds.ew[wave][1] = tw;
  }
  __syncthreads();
  if (T == 0) {
    ew[0] = lds.ew[0][0] + lds.ew[1][0] + lds.ew[2][0] + lds.ew[3][0];
    ew[1] = lds.ew[0][1] + lds.ew[1][1] + lds.ew[2][1] + lds.ew[3][1];
  }
}

// W x W waves per workgroup, groups of G = 128 W particles.  Eight waves per
// SIMD (at most 64 VGPRs; the loop body is unchanged by the limit, no spills).
// ENERGY = false (the time step): no per-particle energies; the partial
// entries carry the force only (three floats, store_part3; no apart), and each
// workgroup writes its
// totals ew[2 item] = sum over ordered pairs of ((s/r)^12 - (s/r)^6) and
// ew[2 item + 1] = sum of w = (s/r)^6 (2 (s/r)^6 - 1), the finaliser's E and W
// terms.  The j side then carries three sums instead of four.
// One group pair (g, h) of one box: q/pf/fpart/apart point at the box's
// arrays, ew (ENERGY = false) at the workgroup's two totals.
// COMP: the compensated mode's sums (pair_tile_c, self_tile_c; W = 2).
// EXCL (kLook): pairs with r2 <= thr are left out.
template <bool PERIODIC, bool TIES, int W, bool ENERGY, bool COMP = false, int EXCL = kNone>
__device__ __forceinline__ void n3_item(N3Lds<W>& lds, const uint4* __restrict__ q,
                                        const float4* __restrict__ pf,
                                        float4* __restrict__ fpart, float* __restrict__ apart,
                                        double* __restrict__ ew, int N, int Npad, float C1, int g,
                                        int h, float thr = 0.f)
{
  constexpr int kG = kTile * W;
  uint4* const s_pos = lds.pos;
  float* const s_acc = lds.acc;
  const int T = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(T >> 6);
  const int lane = T & 63;
  const int wi = wave / W, wj = wave % W;
  const bool diag = g == h;
  const bool partial = kG * (h + 1) > N;

  if (T < kG) {
    const int j = kG * h + T;
    const int jl = j < N ? j : 0;
    uint4 p;
    if constexpr (PERIODIC) {
      p = q[jl];
    } else {
      const float4 f = pf[jl];
      p = make_uint4(__float_as_uint(f.x), __float_as_uint(f.y), __float_as_uint(f.z), 0u);
    }
    p.w = j < N ? 1u : 0u;
    uint4* d = s_pos + (T >> 6) * 128;  // (wj, sub-tile) = (T >> 7, (T >> 6) & 1)
    d[T & 63] = p;
    d[(T & 63) + 64] = p;
  }
  __syncthreads();

  // tiles entirely past N (the last group of a box, partial) are idle, and a
  // second sub-tile past N is skipped: wave-uniform tests
  const int jt0 = kG * h + kTile * wj, it0 = kG * g + kTile * wi;
  const bool live = jt0 < N && it0 < N;
  const int nsub = jt0 + 64 < N ? 2 : 1;
  // pair tile / self tile / idle
  const int cls = !live ? 0 : (diag ? (wi < wj ? 1 : (wi == wj ? 2 : 0)) : 1);
  const int i1 = kG * g + kTile * wi + lane, i2 = i1 + 64;
  const bool v1 = i1 < N, v2 = i2 < N;
  const PosT<PERIODIC> pi1 = load_pos<PERIODIC>(q, pf, v1 ? i1 : N - 1);
  const PosT<PERIODIC> pi2 = load_pos<PERIODIC>(q, pf, v2 ? i2 : N - 1);
  Acc a1, a2;
  acc_zero(a1);
  acc_zero(a2);
  const uint4* P0 = s_pos + wj * 256;
  float J[2][4] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
  if constexpr (COMP) {
    static_assert(W == 2, "compensated items: groups of 256");
    Acc l1, l2;
    acc_zero(l1);
    acc_zero(l2);
    if (cls == 1) {
      if (partial)
        pair_tile_c<PERIODIC, TIES, true, ENERGY>(P0, lane, pi1, pi2, v1, v2, C1, nsub, a1, a2, l1,
                                                  l2, J);
      else
        pair_tile_c<PERIODIC, TIES, false, ENERGY>(P0, lane, pi1, pi2, v1, v2, C1, 2, a1, a2, l1,
                                                   l2, J);
    } else if (cls == 2) {
      self_tile_c<PERIODIC, TIES>(P0, lane, i1, i2, kG * h + kTile * wj, pi1, pi2, v1, v2, C1, nsub,
                                  a1, a2, l1, l2);
    }
    a1.fx += l1.fx, a1.fy += l1.fy, a1.fz += l1.fz, a1.a += l1.a, a1.b += l1.b;
    a2.fx += l2.fx, a2.fy += l2.fy, a2.fz += l2.fz, a2.a += l2.a, a2.b += l2.b;
  } else if (cls == 1) {
    if (partial)
      pair_tile<PERIODIC, TIES, true, ENERGY, EXCL>(P0, lane, pi1, pi2, v1, v2, C1, nsub, a1, a2, J,
                                                    thr);
    else
      pair_tile<PERIODIC, TIES, false, ENERGY, EXCL>(P0, lane, pi1, pi2, v1, v2, C1, 2, a1, a2, J,
                                                     thr);
  } else if (cls == 2) {
    self_tile<PERIODIC, TIES, EXCL>(P0, lane, i1, i2, kG * h + kTile * wj, pi1, pi2, v1, v2, C1, nsub,
                                    a1, a2, thr);
  }
  {
    float* A = s_acc + wave * kAccPerWave;
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
      for (int c = 0; c < 4; ++c) A[(st * 4 + c) * 64 + lane] = J[st][c];
  }
  __syncthreads();

  // j sums of particle G h + T over the W i rows, in row order
  float jf[4] = {0.f, 0.f, 0.f, 0.f};
  if (T < kG) {
    const int col = T >> 7, st = (T >> 6) & 1, idx = T & 63;
    for (int r = 0; r < W; ++r) {
      const float* A = s_acc + (r * W + col) * kAccPerWave + st * 256;
#pragma unroll
      for (int c = 0; c < 4; ++c) jf[c] += A[c * 64 + idx];
    }
  }
  __syncthreads();

  if constexpr (!ENERGY) {
    // E and W totals of the item in the ordered-pair convention: pairs of a
    // pair tile count twice, those of a self tile (both orders) once
    double(*s_ew)[2] = lds.ew;
    const double m = cls == 1 ? 2. : (cls == 2 ? 1. : 0.);
    const double se = (double)a1.a + (double)a2.a, sw = (double)a1.b + (double)a2.b;
    double te = m * 0.5 * (sw - se), tw = m * sw;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      te += __shfl_xor(te, o, 64);
      tw += __shfl_xor(tw, o, 64);
    }
    if (lane == 0) {
      s_ew[wave][0] = te;
      s_ew[wave][1] = tw;
    }
    __syncthreads();
    if (T == 0) {
      double E = 0., Wv = 0.;
      for (int w = 0; w < W * W; ++w) {
        E += s_ew[w][0];
        Wv += s_ew[w][1];
      }
      ew[0] = E;
      ew[1] = Wv;
    }
  }

  // i sums through LDS: ib[wj][component][G]
  float* ib = s_acc;
  {
    float e1[5], e2[5];
    if (cls == 0) {
      for (int c = 0; c < 5; ++c) e1[c] = e2[c] = 0.f;
    } else {
      encode(a1, cls, e1);
      encode(a2, cls, e2);
    }
#pragma unroll
    for (int c = 0; c < 5; ++c) {
      ib[(wj * 5 + c) * kG + kTile * wi + lane] = e1[c];
      ib[(wj * 5 + c) * kG + kTile * wi + lane + 64] = e2[c];
    }
  }
  __syncthreads();

  if (T < kG) {
    float v[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
    for (int c2 = 0; c2 < W; ++c2)
#pragma unroll
      for (int c = 0; c < 5; ++c) v[c] += ib[(c2 * 5 + c) * kG + T];
    if (diag) {
      v[0] += jf[0];
      v[1] += jf[1];
      v[2] += jf[2];
      v[4] += jf[3];
    }
    const int i = kG * g + T;
    const size_t si = h, sj = g;
    if (i < N) {
      if constexpr (ENERGY) {
        store_part(fpart + si * Npad + i, v[0], v[1], v[2], v[3]);
        store_part(apart + si * Npad + i, v[4]);
      } else {
        store_part3(fpart, si * Npad + i, v[0], v[1], v[2]);
      }
    }
    if (!diag) {
      const int j = kG * h + T;
      if (j < N) {
        if constexpr (ENERGY) {
          store_part(fpart + sj * Npad + j, jf[0], jf[1], jf[2], 0.f);
          store_part(apart + sj * Npad + j, jf[3]);
        } else {
          store_part3(fpart, sj * Npad + j, jf[0], jf[1], jf[2]);
        }
      }
    }
  }
}

// item k of ng groups in row order: (g, h) with h >= g; row g starts at
// g ng - g (g - 1) / 2
__device__ __forceinline__ int2 row_item(int k, int ng)
{
  const float b = ng + 0.5f;
  int g = max(0, min(ng - 1, (int)(b - sqrtf(fmaxf(b * b - 2.f * k, 0.f)))));
  while (g > 0 && g * ng - g * (g - 1) / 2 > k) --g;
  while ((g + 1) * ng - (g + 1) * g / 2 <= k) ++g;
  return make_int2(g, g + k - (g * ng - g * (g - 1) / 2));
}

// EXCL (single evaluations that leave out pairs with r2 <= thr): no item table,
// items in row order
// The tie rule's frames take about six more registers: seven waves per SIMD then.
template <bool PERIODIC, bool TIES, int W, bool ENERGY, int EXCL = kNone>
__global__ __launch_bounds__(64 * W * W) __attribute__((amdgpu_waves_per_eu(TIES && W == 2 ? 7 : 8))) void k_force_n3(
    const uint4* __restrict__ q, const float4* __restrict__ pf, const int2* __restrict__ items,
    float4* __restrict__ fpart, float* __restrict__ apart, double* __restrict__ ew, int N, int Npad,
    float C1, int ng, float thr)
{
  __shared__ N3Lds<W> lds;
  const int k = blockIdx.x;  // item
  const int2 it = EXCL ? row_item(k, ng) : items[k];
  if constexpr (!ENERGY && W == 2) {
    if (it.y < 0) {  // diagonal pair (it.x, -2 - it.y), the second one absent when -1
      n3_diag_pair<PERIODIC>(lds, q, pf, fpart, ew + 2 * (size_t)k, N, Npad, C1, it.x, -2 - it.y);
      return;
    }
  }
  n3_item<PERIODIC, TIES, W, ENERGY, false, EXCL>(lds, q, pf, fpart, apart,
                                                  ENERGY ? nullptr : ew + 2 * (size_t)k, N, Npad, C1,
                                                  it.x, it.y, thr);
}

// Small items: a pair of groups of 128 per workgroup of four waves; wave w takes
// j sub-tile w / 2 and its steps 32 (w & 1) + [0, 32) for the 128 i (two per
// lane).  Entries, slots and totals as n3_item's; the last group may lie past N
// (the group count is even): its items write zeros.
// Why: a box of N = 5003 has 210 items of 256, 420 workgroups when halved by j
// sub-tile, one or two waves on a SIMD, which then waits for its own latency
// (13.6 us against 7.6 us of issue).  As 820 small items the waves are half as
// long and three or four share a SIMD; the partial slots are those of the
// halved items.
template <bool PERIODIC, bool TIES, bool ENERGY, int EXCL = kNone>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) void k_force_n3s(
    const uint4* __restrict__ q, const float4* __restrict__ pf, const int2* __restrict__ items,
    float4* __restrict__ fpart, float* __restrict__ apart, double* __restrict__ ew, int N, int Npad,
    float C1, int ng, float thr)
{
  constexpr int NI = ENERGY ? 5 : 3, NJ = ENERGY ? 4 : 3;
  __shared__ uint4 s_pos[2 * 128];       // [sub-tile][doubled 64]
  __shared__ float s_j[4][NJ][64];       // j sums [wave][component][slot]
  __shared__ float s_i[4][NI][kTile];    // i sums [wave][component][i]
  __shared__ double s_ew[4][2];
  const int2 it = EXCL ? row_item(blockIdx.x, ng) : items[blockIdx.x];
  const int g = it.x, h = it.y;
  const int T = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(T >> 6);
  const int lane = T & 63;
  const bool diag = g == h;
  const int i1 = kTile * g + lane, i2 = i1 + 64;
  const bool v1 = i1 < N, v2 = i2 < N;
  const PosT<PERIODIC> pi1 = load_pos<PERIODIC>(q, pf, v1 ? i1 : N - 1);
  const PosT<PERIODIC> pi2 = load_pos<PERIODIC>(q, pf, v2 ? i2 : N - 1);
  if (T < kTile) {
    const int j = kTile * h + T;
    const int jl = j < N ? j : 0;
    uint4 p;
    if constexpr (PERIODIC) {
      p = q[jl];
    } else {
      const float4 f = pf[jl];
      p = make_uint4(__float_as_uint(f.x), __float_as_uint(f.y), __float_as_uint(f.z), 0u);
    }
    p.w = j < N ? 1u : 0u;
    uint4* d = s_pos + (T >> 6) * 128;
    d[T & 63] = p;
    d[(T & 63) + 64] = p;
  }
  __syncthreads();

  const int st = wave >> 1, t0 = 32 * (wave & 1);
  const int jb = kTile * h + 64 * st;  // the wave's j sub-tile
  const bool live = jb < N;            // wave-uniform
  const int cls = !live ? 0 : (diag ? 2 : 1);
  Acc a1, a2;
  acc_zero(a1);
  acc_zero(a2);
  float J[1][4] = {{0.f, 0.f, 0.f, 0.f}};
  if (cls == 1) {  // g < h: every i is valid
    if (jb + 64 > N)
      pair_tile<PERIODIC, TIES, true, ENERGY, EXCL, 1, 32>(s_pos + st * 128, lane, pi1, pi2, v1, v2, C1,
                                                           1, a1, a2, J, thr, t0);
    else
      pair_tile<PERIODIC, TIES, false, ENERGY, EXCL, 1, 32>(s_pos + st * 128, lane, pi1, pi2, v1, v2,
                                                            C1, 1, a1, a2, J, thr, t0);
  } else if (cls == 2) {
    self_tile<PERIODIC, TIES, EXCL, 1, 32>(s_pos + st * 128, lane, i1, i2, jb, pi1, pi2, v1, v2, C1, 1,
                                           a1, a2, thr, t0);
  }
  // after the steps lane l holds the sums of j slot (l + t0 + 32) mod 64
#pragma unroll
  for (int c = 0; c < NJ; ++c) s_j[wave][c][(lane + t0 + 32) & 63] = J[0][c];
  {
    float e1[5], e2[5];
    encode(a1, cls, e1);
    encode(a2, cls, e2);
#pragma unroll
    for (int c = 0; c < NI; ++c) {
      s_i[wave][c][lane] = e1[c];
      s_i[wave][c][lane + 64] = e2[c];
    }
  }
  if constexpr (!ENERGY) {
    // ordered-pair convention, as in n3_item
    const double m = cls == 1 ? 2. : 1.;
    const double se = (double)a1.a + (double)a2.a, sw = (double)a1.b + (double)a2.b;
    double te = m * 0.5 * (sw - se), tw = m * sw;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      te += __shfl_xor(te, o, 64);
      tw += __shfl_xor(tw, o, 64);
    }
    if (lane == 0) {
      s_ew[wave][0] = te;
      s_ew[wave][1] = tw;
    }
  }
  __syncthreads();

  if constexpr (!ENERGY)
    if (T < 2)
      ew[2 * (size_t)blockIdx.x + T] = s_ew[0][T] + s_ew[1][T] + s_ew[2][T] + s_ew[3][T];
  if (T < kTile) {  // i side: slot h
    const int i = kTile * g + T;
    float v[NI];
#pragma unroll
    for (int c = 0; c < NI; ++c) v[c] = (s_i[0][c][T] + s_i[1][c][T]) + (s_i[2][c][T] + s_i[3][c][T]);
    if (i < N) {
      if constexpr (ENERGY) {
        store_part(fpart + (size_t)h * Npad + i, v[0], v[1], v[2], v[3]);
        store_part(apart + (size_t)h * Npad + i, v[4]);
      } else {
        store_part3(fpart, (size_t)h * Npad + i, v[0], v[1], v[2]);
      }
    }
  } else if (!diag) {  // j side: slot g
    const int u = T - kTile, j = kTile * h + u, w = 2 * (u >> 6), x = u & 63;
    float v[NJ];
#pragma unroll
    for (int c = 0; c < NJ; ++c) v[c] = s_j[w][c][x] + s_j[w + 1][c][x];
    if (j < N) {
      if constexpr (ENERGY) {
        store_part(fpart + (size_t)g * Npad + j, v[0], v[1], v[2], 0.f);
        store_part(apart + (size_t)g * Npad + j, v[3]);
      } else {
        store_part3(fpart, (size_t)g * Npad + j, v[0], v[1], v[2]);
      }
    }
  }
}

// Compensated mode: one workgroup per item of the unpaired list (the diagonal
// items through self_tile_c), groups of 256.  The (hi, lo) pairs of the
// compensated sums take about 26 more registers than the FP32 loop, which
// holds eight waves per SIMD at 64; the kernel runs at the occupancy its
// registers allow.
template <bool PERIODIC, bool TIES, bool ENERGY>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5))) void k_force_n3c(const uint4* __restrict__ q,
                                                   const float4* __restrict__ pf,
                                                   const int2* __restrict__ items,
                                                   float4* __restrict__ fpart,
                                                   float* __restrict__ apart,
                                                   double* __restrict__ ew, int N, int Npad,
                                                   float C1)
{
  __shared__ N3Lds<2> lds;
  const int2 it = items[blockIdx.x];
  n3_item<PERIODIC, TIES, 2, ENERGY, true>(lds, q, pf, fpart, apart,
                                                  ENERGY ? nullptr : ew + 2 * (size_t)blockIdx.x, N,
                                                  Npad, C1, it.x, it.y);
}

// batched ensemble: item = (box, g, h) over all boxes; each box's partials at
// its own rows (pbase, S = groups of 256, Npad); ENERGY: per-particle energies
// kept (single evaluations), else the time step's variant with the item's
// (E, W) totals at ew[2 e].
// PERSIST: a grid of resident workgroups drains the item queue (longest items
// first): each takes the next item from the queue head until the head passes
// nitems, which every workgroup reaches; the head is reset by the kernel that
// precedes every force pass (prep, drift, or the previous step's kick).
// Otherwise workgroup b runs item b.
template <bool PERIODIC, bool TIES, bool ENERGY>
__device__ __forceinline__ void batch_n3_item(N3Lds<2>& lds, const uint4* __restrict__ q,
                                              const float4* __restrict__ pf,
                                              float4* __restrict__ fpart, float* __restrict__ apart,
                                              const BoxParam* __restrict__ box,
                                              const BatchItem& w, double* __restrict__ ew)
{
  const BoxParam bp = box[w.box];
  n3_item<PERIODIC, TIES, 2, ENERGY>(lds, q + bp.off, pf + bp.off, fpart + bp.pbase, apart + bp.pbase,
                                     ENERGY ? nullptr : ew + 2 * (size_t)w.e, bp.N, bp.Npad, bp.C1,
                                     w.i0, w.s);
}

template <bool PERIODIC, bool TIES, bool ENERGY, bool PERSIST>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) void k_batch_force_n3(
    const uint4* __restrict__ q, const float4* __restrict__ pf, float4* __restrict__ fpart,
    float* __restrict__ apart, const BoxParam* __restrict__ box, const BatchItem* __restrict__ items,
    double* __restrict__ ew, unsigned* __restrict__ counter, int nitems)
{
  __shared__ N3Lds<2> lds;
  if constexpr (PERSIST) {
    __shared__ unsigned s_item;
    for (;;) {
      if (threadIdx.x == 0) s_item = atomicAdd(counter, 1u);
      __syncthreads();  // also: every thread is done with the previous item's LDS
      const unsigned it = s_item;
      __syncthreads();  // s_item read by all before thread 0 writes it again
      if (it >= (unsigned)nitems) break;  // uniform in the workgroup
      batch_n3_item<PERIODIC, TIES, ENERGY>(lds, q, pf, fpart, apart, box, items[it], ew);
    }
  } else {
    batch_n3_item<PERIODIC, TIES, ENERGY>(lds, q, pf, fpart, apart, box, items[blockIdx.x], ew);
  }
}

}  // namespace

int n3_waves(int /*N*/)
{
  // W = 2 (groups of 256, 4-wave workgroups, up to 8 resident per CU) measured
  // 116 us at N = 16384 against 145 us for W = 4 (groups of 512, 16-wave
  // workgroups, at most 2 per CU); LJ_PAIR_ONCE_WAVES=4 selects the latter
  const char* e = std::getenv("LJ_PAIR_ONCE_WAVES");
  if (e && std::atoi(e) == 4) return 4;
  return 2;
}

// Relative pair rate of one CU holding w four-wave workgroups of the pair
// loop (one wave per SIMD each), measured on the time step's pass at
// rho* = 0.85: 1 : 2.0 : 2.15 : 2.6 for w = 1, 2, 3 and >= 4 (one wave per
// SIMD is bound by its own latency; from four on the VALU is nearly full).
double n3_cu_rate(int w) { return w <= 1 ? 1.0 : w == 2 ? 2.0 : w == 3 ? 2.15 : 2.6; }

// modelled duration of a pass of n workgroups, each `work` items of pairs,
// spread evenly over `cus` CUs: the busiest CU holds ceil(n / cus) of them
double n3_pass_time(long n, double work, int cus)
{
  const int w = (int)((n + cus - 1) / cus);
  return w * work / n3_cu_rate(w);
}

bool n3_small_groups(int W, int ng)
{
  // LJ_PAIR_ONCE_SPLIT=0 / 1 turns the small items off / on (groups of 256)
  if (W != 2) return false;
  const char* e = std::getenv("LJ_PAIR_ONCE_SPLIT");
  if (e && (e[0] == '0' || e[0] == '1')) return e[0] == '1';
  int cus = 256, dev = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      cus <= 0)
    cus = 256;
  // where halves of the items on two workgroups each would by the model take at
  // least 10% less time (twice as many partial slots cost the integrator about
  // that much)
  const long full = (long)ng * (ng + 1) / 2, paired = (long)ng * (ng - 1) / 2 + (ng + 1) / 2;
  return n3_pass_time(2 * full, 0.5, cus) < 0.9 * n3_pass_time(paired, 1.0, cus);
}

ForcePlan make_n3_plan(int N, bool comp)
{
  ForcePlan pl;
  int W = comp ? 2 : n3_waves(N);
  int ng = (N + kTile * W - 1) / (kTile * W);
  if (!comp && n3_small_groups(W, ng)) {
    W = 1;
    ng *= 2;
  }
  pl.N = N;
  pl.n3 = W;
  pl.comp = comp ? 1 : 0;
  pl.ng = ng;
  pl.S = ng;
  pl.jchunk = kTile * W;
  pl.Npad = (N + 63) & ~63;
  pl.nitems = ng * (ng + 1) / 2;
  // the time step of the groups of 256 pairs its diagonal items
  // (n3_step_items), unless compensated
  pl.nitems_step = W == 2 && !comp ? ng * (ng - 1) / 2 + (ng + 1) / 2 : pl.nitems;
  return pl;
}

ForcePlan compat_plan(int N, const PairScalars& ps)
{
  if (n3_eligible(N) && N <= kCompatOnceMaxN && ps.thr > 0.f) {
    const ForcePlan pl = make_n3_plan(N);
    if (pl.n3 != 4 && (size_t)pl.S * pl.Npad <= kCompatSlots) return pl;
  }
  return make_force_plan(N, 0, 1);
}

bool n3_comp_enabled()
{
  // LJ_PAIR_ONCE_COMP=0 keeps the compensated mode on the sliced kernel
  const char* e = std::getenv("LJ_PAIR_ONCE_COMP");
  return !(e && e[0] == '0');
}

bool n3_eligible(int N)
{
  // LJ_PAIR_ONCE=0 / 1 turns the kernel off / on at any size (tuning)
  const char* e = std::getenv("LJ_PAIR_ONCE");
  if (e && (e[0] == '0' || e[0] == '1')) return e[0] == '1' && N >= 256;
  // Up to N = 4096 this decides single evaluations (steps are one launch there).
  // Measured at rho* = 0.85, us, pair-once / sliced: lj_compute_forces N = 2048
  // 38.8 / 38.4, 2560 41.0 / 42.1, 3072 42.6 / 44.4, 3584 43.2 / 48.1, 5003 50.0 /
  // 57.8, most of it launches and the wait; the step's force pass 6.8 / 6.0 at 2560,
  // 8.0 / 7.1 at 3072, 8.1 / 8.9 at 3584, 12.3 / 17.4 at 5003.
  return N >= 3072;
}

void n3_items(int ng, int2* out)
{
  // off-diagonal items first, the lighter diagonal ones last
  int k = 0;
  for (int g = 0; g < ng; ++g)
    for (int h = g + 1; h < ng; ++h) out[k++] = make_int2(g, h);
  for (int g = 0; g < ng; ++g) out[k++] = make_int2(g, g);
}

void n3_step_items(const ForcePlan& pl, int2* out)
{
  if (pl.nitems_step == pl.nitems) {
    n3_items(pl.ng, out);
    return;
  }
  // the diagonal items in pairs (g, g + half) encoded as (g, -2 - (g + half)),
  // a last odd one alone as (g, -1), first: when the workgroups outnumber the
  // resident slots the longer ones should start in the first round; then the
  // off-diagonal items
  const int ng = pl.ng, half = (ng + 1) / 2;
  int k = 0;
  for (int g = 0; g < half; ++g) out[k++] = make_int2(g, g + half < ng ? -2 - (g + half) : -1);
  for (int g = 0; g < ng; ++g)
    for (int h = g + 1; h < ng; ++h) out[k++] = make_int2(g, h);
}

namespace {

template <int W, bool ENERGY, int EXCL = kNone>
hipError_t launch_n3_w(hipStream_t st, const ForcePlan& pl, const PairScalars& ps, const uint4* q,
                       const float4* posf, float4* fpart, float* apart, double* ew, bool ties)
{
  // the time step's variant runs its own item list (diagonal items paired)
  const int nitems = ENERGY ? pl.nitems : pl.nitems_step;
  const int2* items = ENERGY ? pl.items : pl.items_step;
  dim3 grid(nitems), block(W == 1 ? 256 : 64 * W * W);
  const LaunchStamp ts = tl_force_stamp;
#define LJ_N3(P, T)                                                                               \
  do {                                                                                            \
    if constexpr (W == 1)                                                                         \
      hipExtLaunchKernelGGL((k_force_n3s<P, T, ENERGY, EXCL>), grid, block, 0, st, ts.start,      \
                            ts.stop, 0, q, posf, items, fpart, apart, ew, pl.N, pl.Npad, ps.C1,   \
                            pl.ng, ps.thr);                                                       \
    else                                                                                          \
      hipExtLaunchKernelGGL((k_force_n3<P, T, W, ENERGY, EXCL>), grid, block, 0, st, ts.start,    \
                            ts.stop, 0, q, posf, items, fpart, apart, ew, pl.N, pl.Npad, ps.C1,   \
                            pl.ng, ps.thr);                                                       \
  } while (0)
  if (!ps.periodic) LJ_N3(false, false);
  else if (!ties) LJ_N3(true, false);
  else if constexpr (ENERGY) LJ_N3(true, true);
  else return hipErrorInvalidValue;  // the time step has no exact-tie rule
#undef LJ_N3
  return hipGetLastError();
}

template <bool ENERGY>
hipError_t launch_n3_c(hipStream_t st, const ForcePlan& pl, const PairScalars& ps, const uint4* q,
                       const float4* posf, float4* fpart, float* apart, double* ew, bool ties)
{
  // both variants run the unpaired item list (items_step equals it)
  const int nitems = ENERGY ? pl.nitems : pl.nitems_step;
  const int2* items = ENERGY ? pl.items : pl.items_step;
  dim3 grid(nitems), block(256);
  const LaunchStamp ts = tl_force_stamp;
  if (ps.periodic) {
    if (ties)
      hipExtLaunchKernelGGL((k_force_n3c<true, true, ENERGY>), grid, block, 0, st, ts.start, ts.stop,
                            0, q, posf, items, fpart, apart, ew, pl.N, pl.Npad, ps.C1);
    else
      hipExtLaunchKernelGGL((k_force_n3c<true, false, ENERGY>), grid, block, 0, st, ts.start, ts.stop,
                            0, q, posf, items, fpart, apart, ew, pl.N, pl.Npad, ps.C1);
  } else {
    hipExtLaunchKernelGGL((k_force_n3c<false, false, ENERGY>), grid, block, 0, st, ts.start, ts.stop,
                          0, q, posf, items, fpart, apart, ew, pl.N, pl.Npad, ps.C1);
  }
  return hipGetLastError();
}

}  // namespace

template <bool PERIODIC, bool TIES, bool ENERGY>
void launch_batch_n3_t(hipStream_t st, const BatchArgs& a)
{
  const int pg = a.persistent_grid > 0 ? std::min(a.persistent_grid, a.nitems) : 0;
  if (pg > 0)
    hipLaunchKernelGGL((k_batch_force_n3<PERIODIC, TIES, ENERGY, true>), dim3(pg), dim3(256), 0, st,
                       a.q, a.pos, a.fpart, a.apart, a.box, a.items, a.ew, a.counter, a.nitems);
  else
    hipLaunchKernelGGL((k_batch_force_n3<PERIODIC, TIES, ENERGY, false>), dim3(a.nitems),
                       dim3(256), 0, st, a.q, a.pos, a.fpart, a.apart, a.box, a.items, a.ew,
                       a.counter, a.nitems);
}

hipError_t launch_batch_force_n3(hipStream_t st, const BatchArgs& a, bool periodic, bool ties)
{
  if (a.lean) {  // the time step (no exact-tie rule there)
    if (ties || !a.ew) return hipErrorInvalidValue;
    if (periodic) launch_batch_n3_t<true, false, false>(st, a);
    else launch_batch_n3_t<false, false, false>(st, a);
    return hipGetLastError();
  }
  if (periodic) {
    if (ties) launch_batch_n3_t<true, true, true>(st, a);
    else launch_batch_n3_t<true, false, true>(st, a);
  } else {
    launch_batch_n3_t<false, false, true>(st, a);
  }
  return hipGetLastError();
}

hipError_t launch_force_n3_step_items(hipStream_t st, const ForcePlan& pl, const PairScalars& ps,
                                      const uint4* q, const float4* posf, float4* fpart, double* ew,
                                      int first, int count)
{
  // the step variant's items [first, first + count), each writing its own
  // partial entries and (E, W) totals: one GPU's share of a pass whose items
  // are dealt out (W = 2, diagonal items paired)
  if (pl.n3 != 2 || pl.comp || first < 0 || count < 1 ||
      first + count > pl.nitems_step)
    return hipErrorInvalidValue;
  const LaunchStamp ts = tl_force_stamp;
  const int2* items = pl.items_step + first;
  double* e = ew + 2 * (size_t)first;
  if (ps.periodic)
    hipExtLaunchKernelGGL((k_force_n3<true, false, 2, false>), dim3(count), dim3(256), 0, st,
                          ts.start, ts.stop, 0, q, posf, items, fpart, nullptr, e, pl.N, pl.Npad,
                          ps.C1, pl.ng, 0.f);
  else
    hipExtLaunchKernelGGL((k_force_n3<false, false, 2, false>), dim3(count), dim3(256), 0,
                          st, ts.start, ts.stop, 0, q, posf, items, fpart, nullptr, e, pl.N, pl.Npad,
                          ps.C1, pl.ng, 0.f);
  return hipGetLastError();
}

hipError_t launch_force_n3(hipStream_t st, const ForcePlan& pl, const PairScalars& ps,
                           const uint4* q, const float4* posf, float4* fpart, float* apart,
                           bool ties, double* ew)
{
  // ew != null: the time step's variant (force partials + per-workgroup totals)
  if (ps.thr > 0.f && (pl.comp || ew)) return hipErrorInvalidValue;
  if (pl.comp) {
    if (pl.n3 != 2 || pl.nitems_step != pl.nitems) return hipErrorInvalidValue;
    return ew ? launch_n3_c<false>(st, pl, ps, q, posf, fpart, apart, ew, false)
              : launch_n3_c<true>(st, pl, ps, q, posf, fpart, apart, nullptr, ties);
  }
  if (ew) {
    if (pl.n3 == 1) return launch_n3_w<1, false>(st, pl, ps, q, posf, fpart, apart, ew, false);
    if (pl.n3 == 2) return launch_n3_w<2, false>(st, pl, ps, q, posf, fpart, apart, ew, false);
    return launch_n3_w<4, false>(st, pl, ps, q, posf, fpart, apart, ew, false);
  }
  if (ps.thr > 0.f) {  // pairs with r2 <= thr left out
    if (pl.n3 == 1)
      return launch_n3_w<1, true, kLook>(st, pl, ps, q, posf, fpart, apart, nullptr, ties);
    if (pl.n3 == 2)
      return launch_n3_w<2, true, kLook>(st, pl, ps, q, posf, fpart, apart, nullptr, ties);
    return hipErrorInvalidValue;
  }
  if (pl.n3 == 1) return launch_n3_w<1, true>(st, pl, ps, q, posf, fpart, apart, nullptr, ties);
  if (pl.n3 == 2) return launch_n3_w<2, true>(st, pl, ps, q, posf, fpart, apart, nullptr, ties);
  return launch_n3_w<4, true>(st, pl, ps, q, posf, fpart, apart, nullptr, ties);
}

}  // namespace lj
