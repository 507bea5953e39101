// lj_small.h -- the complete force on T particles by one workgroup: the
// device part shared by the one-launch time steps of small boxes
// (lj_small.hip).
#pragma once

#include "lj_device.h"

namespace lj {
namespace dev {

// One workgroup of kSmallThreads threads takes T particles against all N of
// their box: lane tid holds particle i0 + tid % T and meets every P-th j,
// P = kSmallThreads / T, from phase tid / T on.  The j particles pass through
// LDS in chunks; a lane's FP32 sums cover at most 32 pairs, are then added in
// double, and everything across lanes is added in double in a fixed order (so
// the FP32 and the compensated mode share the kernel).
//   One particle per lane: two per lane halve the LDS reads but leave half the
// phases, twice the sums to reduce and a few spills (N = 2048, T = 8, EVN step:
// 8.75 against 7.67 us; four per lane 13 us and more).
constexpr int kSmallThreads = 1024;

template <int T>
struct SmallGeo {
  static_assert(T <= 16 && 16 % T == 0, "a row of 16 lanes holds whole phases");
  static constexpr int P = kSmallThreads / T;               // phases
  static constexpr int CH = 32 * P < 2048 ? 32 * P : 2048;  // j per LDS chunk
  static constexpr int E = kSmallThreads / 16;              // rows of 16 lanes
};

template <int T>
union SmallLds {
  uint4 j[SmallGeo<T>::CH];
  double red[5][SmallGeo<T>::E][T];
};

// v of the lane N below in the row of 16 (rotated), for a double
template <int N>
__device__ __forceinline__ double row_ror(double v)
{
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x120 + N, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x120 + N, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}

// internal coordinates of a box copy: fixed point, or the bits of the floats
template <bool PERIODIC>
__device__ __forceinline__ PosT<PERIODIC> small_pos(const uint4& v)
{
  PosT<PERIODIC> p;
  if constexpr (PERIODIC) {
    p.x = v.x;
    p.y = v.y;
    p.z = v.z;
  } else {
    p.x = __uint_as_float(v.x);
    p.y = __uint_as_float(v.y);
    p.z = __uint_as_float(v.z);
  }
  return p;
}

// Totals of NV sums over the workgroup's lanes of each particle, left in every
// lane of wave 0 (lane % T: the particle); the other waves leave with undefined
// sums and no barrier follows.  The lanes' other LDS data is done with.
template <int NV, int T>
__device__ __forceinline__ void small_reduce(double (&d)[NV],
                                             double (*red)[SmallGeo<T>::E][T])
{
  using G = SmallGeo<T>;
  const int tid = threadIdx.x;
  // the phases of a row of 16 lanes, then the rows through LDS
#pragma unroll
  for (int c = 0; c < NV; ++c) {
    if constexpr (T <= 8) d[c] += row_ror<8>(d[c]);
    if constexpr (T <= 4) d[c] += row_ror<4>(d[c]);
  }
  __syncthreads();
  if (tid % 16 < T)
#pragma unroll
    for (int c = 0; c < NV; ++c) red[c][tid / 16][tid % T] = d[c];
  __syncthreads();
  if (tid >= 64) return;
  constexpr int EG = G::E * T / 64;  // rows per lane
#pragma unroll
  for (int c = 0; c < NV; ++c) d[c] = 0.;
#pragma unroll
  for (int e = 0; e < EG; ++e)
#pragma unroll
    for (int c = 0; c < NV; ++c) d[c] += red[c][(tid / T) * EG + e][tid % T];
#pragma unroll
  for (int o = T; o < 64; o <<= 1)
#pragma unroll
    for (int c = 0; c < NV; ++c) d[c] += __shfl_xor(d[c], o, 64);
}

// Sums over all j of the pairs of particle i0 + lane % T, returned in every
// lane of wave 0 (the other waves return with undefined sums; no barrier
// follows).  i0 is a multiple of T; q holds the box's N particles.
template <bool PERIODIC, int T>
__device__ __forceinline__ Partial small_forces(SmallLds<T>& lds, const uint4* __restrict__ q,
                                                int N, int i0, float C1)
{
  using G = SmallGeo<T>;
  const int tid = threadIdx.x, ph = tid / T, i = i0 + tid % T;
  const PosT<PERIODIC> pi = small_pos<PERIODIC>(q[min(i, N - 1)]);
  double d[5] = {0., 0., 0., 0., 0.};
  for (int c0 = 0; c0 < N; c0 += G::CH) {
    const int n = min(G::CH, N - c0);
    if (c0 > 0) __syncthreads();
#pragma unroll
    for (int t = 0; t < G::CH; t += kSmallThreads)
      if (t + tid < n) lds.j[t + tid] = q[c0 + t + tid];
    __syncthreads();
    Acc a;
    acc_zero(a);
    // rows of P particles; the T particles of the tile are met in one row
    // (T divides P), which alone looks for the self pair; a last, shorter row
    // looks for its end
    const int rows = n / G::P;
    const int self = i0 >= c0 && i0 < c0 + G::CH ? (i0 - c0) / G::P : -1;
    const auto open = [&](int k0, int k1) {
#pragma unroll 4
      for (int k = k0; k < k1; ++k)
        pair<0>(pi, small_pos<PERIODIC>(lds.j[k * G::P + ph]), 0, 0, C1, 0.f, a);
    };
    const auto guarded = [&](int k) {
      const int j = k * G::P + ph;
      pair<1>(pi, small_pos<PERIODIC>(lds.j[min(j, n - 1)]), i, j < n ? c0 + j : i, C1,
                        0.f, a);
    };
    if (self >= 0 && self < rows) {
      open(0, self);
      guarded(self);
      open(self + 1, rows);
    } else {
      open(0, rows);
    }
    if (rows * G::P < n) guarded(rows);
    d[0] += a.fx;
    d[1] += a.fy;
    d[2] += a.fz;
    d[3] += a.a;
    d[4] += a.b;
  }
  small_reduce<5, T>(d, lds.red);
  return Partial{d[0], d[1], d[2], d[3], d[4]};
}

// totals of NV values over the T lead lanes of wave 0 (the others hold zeros)
template <int NV, int T>
__device__ __forceinline__ void small_row_sum(double (&v)[NV])
{
#pragma unroll
  for (int o = 1; o < T; o <<= 1)
#pragma unroll
    for (int k = 0; k < NV; ++k) v[k] += __shfl_xor(v[k], o, 64);
}

// the copy of a particle's coordinates that the next force pass reads
template <bool PERIODIC>
__device__ __forceinline__ uint4 small_q(const float4& p, double qs)
{
  if constexpr (PERIODIC) return make_uint4(fixq(p.x, qs), fixq(p.y, qs), fixq(p.z, qs), 0u);
  else return make_uint4(__float_as_uint(p.x), __float_as_uint(p.y), __float_as_uint(p.z), 0u);
}

}  // namespace dev
}  // namespace lj
