// lj_fp64.hip -- the FP64 precision mode: double positions, velocities and
// forces, double pair arithmetic, and the reference integrator's formulas
// (MDSystem.cpp:442-510) evaluated in double. It is the device reference of
// the precision study: the FP32 and compensated modes are measured against it
// over long trajectories that a CPU cannot follow at N = 131072.
//
// Pair pass: every unordered pair once over pairs of 256-particle groups
// (k_force64_n3), or, with an explicit j-slice count and where the groups' slots
// would take too much memory, the sliced decomposition (one i per lane, grid =
// i-tiles x j-slices, j streamed through SGPRs by uniform scalar loads); minimum
// image dx -= L rint(dx / L) in double; self pair excluded by index
// (MDSystem.cpp:267).  Partial entries are summed per particle in fixed order.
#include "lj_fp64.h"
#include "lj_small.h"

namespace lj {

namespace {

using namespace dev;

// 1 / x in double: the hardware estimate (v_rcp_f64, good to about 2^-23)
// refined by one third-order step, y + y (e + e^2) with e = 1 - x y, to within
// an ulp or two of the quotient (e^3 is below 2^-60; the IEEE division's scaling
// and fix-up sequence cost several times as much in the pair loop, two Newton
// steps one instruction more)
__device__ __forceinline__ double rcp64(double x)
{
  const double y = __builtin_amdgcn_rcp(x);
  const double e = __builtin_fma(-x, y, 1.);
  return __builtin_fma(y, __builtin_fma(e, e, e), y);
}

// the terms of one pair: sc d is the force on i (internal units), ir6 and w the
// energy and virial terms; GUARD: ok = false leaves the pair out
template <bool PERIODIC, bool GUARD>
__device__ __forceinline__ void terms64(double xi, double yi, double zi, double xj, double yj,
                                        double zj, double L, double invL, double s2, bool ok,
                                        double& dx, double& dy, double& dz, double& sc, double& ir6,
                                        double& w)
{
  dx = xi - xj;
  dy = yi - yj;
  dz = zi - zj;
  if constexpr (PERIODIC) {
    dx -= L * __builtin_rint(dx * invL);
    dy -= L * __builtin_rint(dy * invL);
    dz -= L * __builtin_rint(dz * invL);
  }
  const double r2 = dx * dx + dy * dy + dz * dz;
  double ir2 = s2 * rcp64(GUARD && !ok ? 1. : r2);
  if constexpr (GUARD) ir2 = ok ? ir2 : 0.;
  ir6 = ir2 * ir2 * ir2;
  w = ir6 * (2. * ir6 - 1.);
  sc = w * ir2;
}

// a particle's sums over its pairs: force, a = sum ir6, b = sum w
struct Acc64 {
  double fx, fy, fz, a, b;
};

__device__ __forceinline__ void add64(Acc64& c, double dx, double dy, double dz, double sc, double ir6,
                                      double w)
{
  c.fx += sc * dx;
  c.fy += sc * dy;
  c.fz += sc * dz;
  c.a += ir6;
  c.b += w;
}

// pairs (i, j), j in [jb, je), j streamed through SGPRs (uniform scalar
// loads), four j loaded ahead of their pairs: a loop of one j waited on each
// scalar load in turn.  GUARD: j may be i (the self pair, excluded)
template <bool PERIODIC, bool GUARD>
__device__ __forceinline__ void force64_range(const double4* __restrict__ x, const double4& xi,
                                              int i, int jb, int je, double L, double invL,
                                              double s2, Acc64& c)
{
  const auto one = [&](const double4& xj, int j) {
    double dx, dy, dz, sc, ir6, w;
    terms64<PERIODIC, GUARD>(xi.x, xi.y, xi.z, xj.x, xj.y, xj.z, L, invL, s2, j != i, dx, dy, dz, sc,
                             ir6, w);
    add64(c, dx, dy, dz, sc, ir6, w);
  };
  int j = __builtin_amdgcn_readfirstlane(jb);
  for (; j + 4 <= je; j += 4) {
    const double4 x0 = x[j], x1 = x[j + 1], x2 = x[j + 2], x3 = x[j + 3];
    one(x0, j);
    one(x1, j + 1);
    one(x2, j + 2);
    one(x3, j + 3);
  }
  for (; j < je; ++j) one(x[j], j);
}

// Partial entries of every pass here: (fx, fy, fz, m), m = sum (ir6 - w), so
// that e_i = -m / 2; the virial needs no per-particle sums: each wave (sliced)
// or workgroup (pair-once) writes its total of w over ordered pairs to wt.
template <bool PERIODIC>
__global__ __launch_bounds__(kBlock) void k_force64(const double4* __restrict__ x, int N, int Npad,
                                                    int jchunk, double L, double invL, double s2,
                                                    double4* __restrict__ part,
                                                    double* __restrict__ wt)
{
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i0 = (blockIdx.x * kWaves + wv) * 64;
  const int s = blockIdx.y;
  const int j0 = s * jchunk;
  const int j1 = min(N, j0 + jchunk);
  const int i = i0 + lane;
  Acc64 c{0., 0., 0., 0., 0.};
  if (i0 < N) {
    const double4 xi = x[min(i, N - 1)];
    // the self pair can only lie in the wave's own 64 j: the guard runs there
    const int d0 = max(j0, i0), d1 = min(j1, i0 + 64);
    if (d0 >= d1) {
      force64_range<PERIODIC, false>(x, xi, i, j0, j1, L, invL, s2, c);
    } else {
      force64_range<PERIODIC, false>(x, xi, i, j0, d0, L, invL, s2, c);
      force64_range<PERIODIC, true>(x, xi, i, d0, d1, L, invL, s2, c);
      force64_range<PERIODIC, false>(x, xi, i, d1, j1, L, invL, s2, c);
    }
  }
  if (i < N) store_part(part + (size_t)s * Npad + i, c.fx, c.fy, c.fz, c.a - c.b);
  double b = i < N ? c.b : 0.;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) b += __shfl_xor(b, o, 64);
  if (lane == 0) wt[((size_t)s * gridDim.x + blockIdx.x) * kWaves + wv] = b;
}

// ---- every unordered pair once (the decomposition of lj_force_n3.hip) ----
// Work item (g, h), h >= g, of two groups of 256 particles, one workgroup of
// 2 x 2 waves: wave (wi, wj) holds 128 i of group g (two per lane) and meets the
// 128 j of group h in two sub-tiles of 64, which sit in LDS twice in a row, so
// that at step t lane l reads j (l + t) mod 64; the sums of the j travel with
// them, one lane down per step (ds_bpermute).  Slot h of a particle of group g
// receives its i sums, slot g of one of group h its j sums.
//   35 FP64 instructions and one v_rcp_f64 (four issue slots) per unordered pair of
// a periodic box against 2 x 33 of the sliced pass; bound by their issue (N = 40000:
// 1671 -> 1046 us on one card, 912 on a faster one, 77 to 88% of the slots; 16384:
// 301 -> 197 us, where the last, partly filled round of workgroups shows; 8000:
// 75 -> 55).  SPLIT: two workgroups per item, one j
// sub-tile of every wave each (2 ng slots), for sizes whose items leave most
// SIMDs a wave or less.
constexpr int kG64 = 256;

struct N64Lds {
  double x[3][4 * 128];  // [sub-tile][doubled 64]
  double acc[4 * 512];   // j sums [wave][sub-tile][4][64], then i sums [wj][4][256]
  double w[4];
};

__device__ __forceinline__ double rot64(double v, int src4)
{
  const int lo = __builtin_amdgcn_ds_bpermute(src4, __double2loint(v));
  const int hi = __builtin_amdgcn_ds_bpermute(src4, __double2hiint(v));
  return __hiloint2double(hi, lo);
}

// PARTIAL: only pairs with a valid i (v1, v2) and j (first j of the sub-tile +
// slot < N) count
template <bool PERIODIC, bool PARTIAL>
__device__ __forceinline__ void pair_tile64(const N64Lds& lds, int sub, int lane, int jb, int N,
                                            const double4& x1, const double4& x2, bool v1, bool v2,
                                            double L, double invL, double s2, Acc64& a1, Acc64& a2,
                                            double (&J)[4])
{
  const int src4 = ((lane + 1) & 63) << 2;
  const double *px = lds.x[0] + sub * 128, *py = lds.x[1] + sub * 128, *pz = lds.x[2] + sub * 128;
  double jx = 0., jy = 0., jz = 0., jm = 0.;
#pragma unroll 2
  for (int t = 0; t < 64; ++t) {
    const double xj = px[lane + t], yj = py[lane + t], zj = pz[lane + t];
    const bool jv = !PARTIAL || jb + ((lane + t) & 63) < N;
    double dx, dy, dz, sc, ir6, w;
    terms64<PERIODIC, PARTIAL>(x1.x, x1.y, x1.z, xj, yj, zj, L, invL, s2, v1 && jv, dx, dy, dz, sc,
                               ir6, w);
    add64(a1, dx, dy, dz, sc, ir6, w);
    jx -= sc * dx;
    jy -= sc * dy;
    jz -= sc * dz;
    jm += ir6 - w;
    terms64<PERIODIC, PARTIAL>(x2.x, x2.y, x2.z, xj, yj, zj, L, invL, s2, v2 && jv, dx, dy, dz, sc,
                               ir6, w);
    add64(a2, dx, dy, dz, sc, ir6, w);
    jx -= sc * dx;
    jy -= sc * dy;
    jz -= sc * dz;
    jm += ir6 - w;
    jx = rot64(jx, src4);
    jy = rot64(jy, src4);
    jz = rot64(jz, src4);
    jm = rot64(jm, src4);
  }
  J[0] = jx;
  J[1] = jy;
  J[2] = jz;
  J[3] = jm;
}

// both orders of the wave's own tile, i sums only, self pair excluded
template <bool PERIODIC>
__device__ __forceinline__ void self_tile64(const N64Lds& lds, int sub, int lane, int jb, int N, int i1,
                                            int i2, const double4& x1, const double4& x2, double L,
                                            double invL, double s2, Acc64& a1, Acc64& a2)
{
  const double *px = lds.x[0] + sub * 128, *py = lds.x[1] + sub * 128, *pz = lds.x[2] + sub * 128;
#pragma unroll 2
  for (int t = 0; t < 64; ++t) {
    const double xj = px[lane + t], yj = py[lane + t], zj = pz[lane + t];
    const int j = jb + ((lane + t) & 63);
    double dx, dy, dz, sc, ir6, w;
    terms64<PERIODIC, true>(x1.x, x1.y, x1.z, xj, yj, zj, L, invL, s2, i1 < N && j < N && j != i1, dx,
                            dy, dz, sc, ir6, w);
    add64(a1, dx, dy, dz, sc, ir6, w);
    terms64<PERIODIC, true>(x2.x, x2.y, x2.z, xj, yj, zj, L, invL, s2, i2 < N && j < N && j != i2, dx,
                            dy, dz, sc, ir6, w);
    add64(a2, dx, dy, dz, sc, ir6, w);
  }
}

template <bool PERIODIC, bool SPLIT>
__global__ __launch_bounds__(256) void k_force64_n3(const double4* __restrict__ x,
                                                    const int2* __restrict__ items, int N, int Npad,
                                                    double L, double invL, double s2,
                                                    double4* __restrict__ part,
                                                    double* __restrict__ wt)
{
  __shared__ N64Lds lds;
  const int wg = blockIdx.x;
  const int2 it = items[SPLIT ? wg >> 1 : wg];
  const int half = SPLIT ? wg & 1 : 0;
  const int g = it.x, h = it.y;
  const int T = threadIdx.x, lane = T & 63;
  const int wave = __builtin_amdgcn_readfirstlane(T >> 6);
  const int wi = wave >> 1, wj = wave & 1;
  const bool diag = g == h;
  {
    const double4 p = x[min(kG64 * h + T, N - 1)];
    const int o = wave * 128 + lane;
    lds.x[0][o] = lds.x[0][o + 64] = p.x;
    lds.x[1][o] = lds.x[1][o + 64] = p.y;
    lds.x[2][o] = lds.x[2][o + 64] = p.z;
  }
  __syncthreads();
  const int jt0 = kG64 * h + 128 * wj, it0 = kG64 * g + 128 * wi;
  // pair tile / self tile / idle (a diagonal item's lower wave, tiles past N)
  const int cls = jt0 >= N || it0 >= N ? 0 : !diag || wi < wj ? 1 : wi == wj ? 2 : 0;
  const bool partial = kG64 * (h + 1) > N;
  const int i1 = it0 + lane, i2 = i1 + 64;
  const double4 x1 = x[min(i1, N - 1)], x2 = x[min(i2, N - 1)];
  Acc64 a1{0., 0., 0., 0., 0.}, a2{0., 0., 0., 0., 0.};
  double J[2][4] = {};
#pragma unroll
  for (int st = 0; st < 2; ++st) {
    const int jb = jt0 + 64 * st;
    if ((SPLIT && st != half) || cls == 0 || jb >= N) continue;  // wave-uniform
    if (cls == 2)
      self_tile64<PERIODIC>(lds, 2 * wj + st, lane, jb, N, i1, i2, x1, x2, L, invL, s2, a1, a2);
    else if (partial)
      pair_tile64<PERIODIC, true>(lds, 2 * wj + st, lane, jb, N, x1, x2, i1 < N, i2 < N, L, invL, s2,
                                  a1, a2, J[st]);
    else
      pair_tile64<PERIODIC, false>(lds, 2 * wj + st, lane, jb, N, x1, x2, true, true, L, invL, s2, a1,
                                   a2, J[st]);
  }
#pragma unroll
  for (int st = 0; st < 2; ++st)
#pragma unroll
    for (int c = 0; c < 4; ++c) lds.acc[((wave * 2 + st) * 4 + c) * 64 + lane] = J[st][c];
  // total of w over ordered pairs: a pair tile's count twice
  double w = (cls == 1 ? 2. : 1.) * (a1.b + a2.b);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) w += __shfl_xor(w, o, 64);
  if (lane == 0) lds.w[wave] = w;
  __syncthreads();
  if (T == 0) wt[wg] = lds.w[0] + lds.w[1] + lds.w[2] + lds.w[3];
  // j sums of particle 256 h + T over the two i rows
  double jf[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int o = ((wave & 1) * 4 + c) * 64 + lane, col = wave >> 1;
    jf[c] = lds.acc[col * 512 + o] + lds.acc[(2 + col) * 512 + o];
  }
  __syncthreads();
  {
    double* ib = lds.acc + wj * 1024 + 128 * wi + lane;
    const double v1[4] = {a1.fx, a1.fy, a1.fz, a1.a - a1.b}, v2[4] = {a2.fx, a2.fy, a2.fz, a2.a - a2.b};
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      ib[c * 256] = v1[c];
      ib[c * 256 + 64] = v2[c];
    }
  }
  __syncthreads();
  double v[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    v[c] = lds.acc[c * 256 + T] + lds.acc[1024 + c * 256 + T];
    if (diag) v[c] += jf[c];
  }
  const int i = kG64 * g + T, j = kG64 * h + T;
  const size_t si = SPLIT ? 2 * h + half : h, sj = SPLIT ? 2 * g + half : g;
  if (i < N) store_part(part + si * Npad + i, v[0], v[1], v[2], v[3]);
  if (!diag && j < N) store_part(part + sj * Npad + j, jf[0], jf[1], jf[2], jf[3]);
}

// ---- integrator: four lanes share a particle's slot sums and a block holds
// kRowParticles particles, one block row each (as the FP32 kernels) ----

constexpr int kLanes64 = kBlock / kRowParticles;

struct Sum64 {
  double fx, fy, fz, m;
};

// every lane of the wave calls this; i < 0: no particle
__device__ __forceinline__ Sum64 sum_slices64(const Step64& a, int i, int r)
{
  constexpr int B = 8;
  Sum64 p{0., 0., 0., 0.};
  const int C = (a.S + kLanes64 - 1) / kLanes64;
  const int s0 = i >= 0 ? min(a.S, r * C) : 0, s1 = i >= 0 ? min(a.S, s0 + C) : 0;
  for (int s = s0; s < s1; s += B) {
    double4 f[B];
#pragma unroll
    for (int k = 0; k < B; ++k) f[k] = a.part[(size_t)min(s + k, s1 - 1) * a.Npad + i];
#pragma unroll
    for (int k = 0; k < B; ++k) {
      const bool in = s + k < s1;
      p.fx += in ? f[k].x : 0.;
      p.fy += in ? f[k].y : 0.;
      p.fz += in ? f[k].z : 0.;
      p.m += in ? f[k].w : 0.;
    }
  }
#pragma unroll
  for (int o = 1; o < kLanes64; o <<= 1) {
    p.fx += __shfl_xor(p.fx, o, 64);
    p.fy += __shfl_xor(p.fy, o, 64);
    p.fz += __shfl_xor(p.fz, o, 64);
    p.m += __shfl_xor(p.m, o, 64);
  }
  return p;
}

// this thread's share of the force pass's totals of w, for a grid of a.nrow rows
__device__ __forceinline__ double w_share(const Step64& a, int row)
{
  double w = 0.;
  for (int k = row * kBlock + (int)threadIdx.x; k < a.nwt; k += a.nrow * kBlock) w += a.wt[k];
  return w;
}

// forces of particle i from its sums, into f and the FP32 mirror
__device__ __forceinline__ double4 finish_force(const Step64& a, int i, const Sum64& p)
{
  const double e = -0.5 * p.m;
  const double4 f = make_double4(a.FS * p.fx, a.FS * p.fy, a.FS * p.fz, e);
  a.f[i] = f;
  a.force[i] = make_float4((float)f.x, (float)f.y, (float)f.z, (float)e);
  return f;
}

__device__ __forceinline__ void bc64(double4& x, double4& v, int bc, double L)
{
  if (bc == LJ_BC_PERIODIC) {  // MDSystem.cpp:414-424
    if (x.x < 0.) x.x += L;
    if (x.x > L) x.x -= L;
    if (x.y < 0.) x.y += L;
    if (x.y > L) x.y -= L;
    if (x.z < 0.) x.z += L;
    if (x.z > L) x.z -= L;
  } else if (bc == LJ_BC_WALL) {  // MDSystem.cpp:425-435
    if (x.x < 0. && v.x < 0.) v.x = -v.x;
    if (x.x > L && v.x > 0.) v.x = -v.x;
    if (x.y < 0. && v.y < 0.) v.y = -v.y;
    if (x.y > L && v.y > 0.) v.y = -v.y;
    if (x.z < 0. && v.z < 0.) v.z = -v.z;
    if (x.z > L && v.z > 0.) v.z = -v.z;
  }
}

// written out, so that every kernel contracts it alike
__device__ __forceinline__ double sq3(const double4& v)
{
  return __builtin_fma(v.z, v.z, __builtin_fma(v.y, v.y, v.x * v.x));
}

__device__ __forceinline__ float4 narrow(const double4& d)
{
  return make_float4((float)d.x, (float)d.y, (float)d.z, (float)d.w);
}

// MDSystem.cpp:447-453 (EVN) and :473-479 (TVN) in double.  Run by the drift
// kernel or at the end of the previous step; without contraction, so that both
// give the same bits.
template <int CANON>
__device__ __forceinline__ void drift64(const Step64& a, int i, double4 x, double4 v, const double4& f)
{
#pragma clang fp contract(off)
  const double dt = a.dt;
  x.x += dt * v.x + dt * dt * f.x / 2.;
  x.y += dt * v.y + dt * dt * f.y / 2.;
  x.z += dt * v.z + dt * dt * f.z / 2.;
  a.x[i] = x;
  if constexpr (CANON == LJ_EVN) {
    v.x += dt * f.x / 2.;
    v.y += dt * f.y / 2.;
    v.z += dt * f.z / 2.;
    v.w = 0.;
    a.v[i] = v;
  } else {
    a.tf[i] = make_double4(0.5 * f.x, 0.5 * f.y, 0.5 * f.z, 0.);
  }
}

// the state at the end of a step of a run: the next step's drift, or the
// final state with its FP32 mirrors
template <bool DRIFT, int CANON>
__device__ __forceinline__ void end_step64(const Step64& a, int i, const double4& x, const double4& v,
                                           const double4& f)
{
  if constexpr (DRIFT) {
    if constexpr (CANON == LJ_TVN) a.v[i] = v;
    drift64<CANON>(a, i, x, v, f);
  } else {
    if (a.bc == LJ_BC_PERIODIC) a.x[i] = x;
    a.v[i] = v;
    a.pos[i] = narrow(x);
    a.vel[i] = narrow(v);
  }
}

__global__ __launch_bounds__(kBlock) void k_reduce64(Step64 a)
{
  const int r = threadIdx.x % kLanes64, i = blockIdx.x * kRowParticles + threadIdx.x / kLanes64;
  const Sum64 p = sum_slices64(a, i < a.N ? i : -1, r);
  double v[2] = {0., w_share(a, blockIdx.x)};
  if (i < a.N && r == 0) v[0] = finish_force(a, i, p).w;
  const int fld[2] = {BLK_E, BLK_B};
  block_sum_store<2>(v, a.blk + (size_t)blockIdx.x * kBlkFields, fld);
}

template <int CANON>
__global__ __launch_bounds__(kBlock) void k_drift64(Step64 a)
{
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < a.N) drift64<CANON>(a, i, a.x[i], a.v[i], a.f[i]);
}

// MDSystem.cpp:458-462, then the boundary conditions (:406-436, called at :578).
// DRIFT: also the next step's drift; FIN: block 0 computes the observables of
// the run's previous step.
template <bool DRIFT, bool FIN>
__global__ __launch_bounds__(kBlock) void k_kick64(Step64 a, StepArgs fin)
{
#pragma clang fp contract(off)
  if constexpr (FIN) {
    if (blockIdx.x == 0) {
      step_observables<kWaves>(fin, fin.nrow, true, true);
      return;
    }
  }
  const int row = (int)blockIdx.x - (FIN ? 1 : 0);
  const int r = threadIdx.x % kLanes64, i = row * kRowParticles + threadIdx.x / kLanes64;
  const bool lead = r == 0 && i < a.N;
  double4 v = {}, x = {};
  if (lead) {
    v = a.v[i];
    x = a.x[i];
  }
  const Sum64 p = sum_slices64(a, i < a.N ? i : -1, r);
  double v3[3] = {0., 0., w_share(a, row)};
  if (lead) {
    const double4 f = finish_force(a, i, p);
    const double dt = a.dt;
    v.x += dt * f.x / 2.;
    v.y += dt * f.y / 2.;
    v.z += dt * f.z / 2.;
    bc64(x, v, a.bc, a.L);
    v3[0] = sq3(v);
    v3[1] = f.w;
    end_step64<DRIFT, LJ_EVN>(a, i, x, v, f);
  }
  const int fld[3] = {BLK_K2, BLK_E, BLK_B};
  block_sum_store<3>(v3, a.blk + (size_t)row * kBlkFields, fld);
}

// MDSystem.cpp:484-495: the averaged force and the half-step velocities
template <bool FIN>
__global__ __launch_bounds__(kBlock) void k_tvn64_a(Step64 a, StepArgs fin)
{
#pragma clang fp contract(off)
  if constexpr (FIN) {
    if (blockIdx.x == 0) {
      step_observables<kWaves>(fin, fin.nrow, true, true);
      return;
    }
  }
  const int row = (int)blockIdx.x - (FIN ? 1 : 0);
  const int r = threadIdx.x % kLanes64, i = row * kRowParticles + threadIdx.x / kLanes64;
  const bool lead = r == 0 && i < a.N;
  double4 v = {}, tf = {};
  if (lead) {
    v = a.v[i];
    tf = a.tf[i];
  }
  const Sum64 p = sum_slices64(a, i < a.N ? i : -1, r);
  double v3[3] = {0., 0., w_share(a, row)};
  if (lead) {
    const double4 f = finish_force(a, i, p);
    tf.x += 0.5 * f.x;
    tf.y += 0.5 * f.y;
    tf.z += 0.5 * f.z;
    a.tf[i] = tf;
    const double dt = a.dt;
    const double4 tv = make_double4(v.x + dt * tf.x / 2., v.y + dt * tf.y / 2., v.z + dt * tf.z / 2., 0.);
    v3[0] = sq3(tv);
    v3[1] = f.w;
  }
  const int fld[3] = {BLK_TV2, BLK_E, BLK_B};
  block_sum_store<3>(v3, a.blk + (size_t)row * kBlkFields, fld);
}

// MDSystem.cpp:497-505 (T_kin over 3N, :370), then the boundary conditions; one
// particle per thread, each wave writes the K2 field of its row
template <bool DRIFT>
__global__ __launch_bounds__(kBlock) void k_tvn64_b(Step64 a)
{
#pragma clang fp contract(off)
  const int i = blockIdx.x * kBlock + threadIdx.x;
  double4 v = {}, x = {}, tf = {}, f = {};
  if (i < a.N) {
    v = a.v[i];
    x = a.x[i];
    tf = a.tf[i];
    if (DRIFT) f = a.f[i];
  }
  const double tv2 = blk_total(a.blk, a.nrow, BLK_TV2);
  const double chi = sqrt(a.T0 / (tv2 * (1. / 3. / a.N)));
  double k2 = 0.;
  if (i < a.N) {
    const double dt = a.dt;
    v.x = (2. * chi - 1.) * v.x + chi * dt * tf.x;
    v.y = (2. * chi - 1.) * v.y + chi * dt * tf.y;
    v.z = (2. * chi - 1.) * v.z + chi * dt * tf.z;
    bc64(x, v, a.bc, a.L);
    k2 = sq3(v);
    end_step64<DRIFT, LJ_TVN>(a, i, x, v, f);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) k2 += __shfl_xor(k2, o, 64);
  const int row = i / kRowParticles;
  if ((threadIdx.x & 63) == 0 && row < a.nrow) a.blk[(size_t)row * kBlkFields + BLK_K2] = k2;
}

// ---- one-launch steps (lj_small.h) in double: N <= 4096 ----

template <int T>
union Small64Lds {
  double x[3][SmallGeo<T>::CH];
  double red[5][SmallGeo<T>::E][T];
};

// (fx, fy, fz, m, b) of particle i0 + lane % T in wave 0, as small_forces
template <bool PERIODIC, int T>
__device__ __forceinline__ void small_forces64(Small64Lds<T>& lds, const double4* __restrict__ xs,
                                               int N, int i0, double L, double s2, double (&d)[5])
{
  using G = SmallGeo<T>;
  const int tid = threadIdx.x, ph = tid / T, i = i0 + tid % T;
  const double4 xi = xs[min(i, N - 1)];
  const double invL = 1. / L;
  Acc64 a{0., 0., 0., 0., 0.};
  for (int c0 = 0; c0 < N; c0 += G::CH) {
    const int n = min(G::CH, N - c0);
    if (c0 > 0) __syncthreads();
#pragma unroll
    for (int t = 0; t < G::CH; t += kSmallThreads)
      if (t + tid < n) {
        const double4 p = xs[c0 + t + tid];
        lds.x[0][t + tid] = p.x;
        lds.x[1][t + tid] = p.y;
        lds.x[2][t + tid] = p.z;
      }
    __syncthreads();
    const int rows = n / G::P;
    const int self = i0 >= c0 && i0 < c0 + G::CH ? (i0 - c0) / G::P : -1;
    const auto one = [&](auto guard, int j, bool ok) {
      double dx, dy, dz, sc, ir6, w;
      terms64<PERIODIC, decltype(guard)::value>(xi.x, xi.y, xi.z, lds.x[0][j], lds.x[1][j], lds.x[2][j],
                                                L, invL, s2, ok, dx, dy, dz, sc, ir6, w);
      add64(a, dx, dy, dz, sc, ir6, w);
    };
    const auto open = [&](int k0, int k1) {
#pragma unroll 2
      for (int k = k0; k < k1; ++k) one(std::false_type{}, k * G::P + ph, true);
    };
    const auto guarded = [&](int k) {
      const int j = k * G::P + ph;
      one(std::true_type{}, min(j, n - 1), j < n && c0 + j != i);
    };
    if (self >= 0 && self < rows) {
      open(0, self);
      guarded(self);
      open(self + 1, rows);
    } else {
      open(0, rows);
    }
    if (rows * G::P < n) guarded(rows);
  }
  d[0] = a.fx;
  d[1] = a.fy;
  d[2] = a.fz;
  d[3] = a.a - a.b;
  d[4] = a.b;
  small_reduce<5, T>(d, lds.red);
}

template <int CANON>
__global__ __launch_bounds__(kBlock) void k_small_drift64(Step64 a)
{
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= a.N) return;
  drift64<CANON>(a, i, a.x[i], a.v[i], a.f[i]);
  a.xn[i] = a.x[i];
}

template <bool PERIODIC, int T, bool DRIFT, bool FIN>
__global__ __launch_bounds__(kSmallThreads) void k_small64_evn(Step64 a, StepArgs fin)
{
#pragma clang fp contract(off)
  __shared__ Small64Lds<T> lds;
  if constexpr (FIN) {
    if (blockIdx.x == 0) {
      if (threadIdx.x < kBlock) step_observables<kWaves>(fin, fin.nrow, true, true);
      return;
    }
  }
  const int row = (int)blockIdx.x - (FIN ? 1 : 0);
  const int i = row * T + threadIdx.x;
  const bool lead = threadIdx.x < T && i < a.N;
  double s[5];
  small_forces64<PERIODIC, T>(lds, a.xs, a.N, row * T, a.L, a.sigma * a.sigma, s);
  if (threadIdx.x >= 64) return;
  double v3[3] = {0., 0., 0.};
  if (lead) {
    double4 v = a.v[i], x = a.x[i];
    const double4 f = finish_force(a, i, Sum64{s[0], s[1], s[2], s[3]});
    const double dt = a.dt;
    v.x += dt * f.x / 2.;
    v.y += dt * f.y / 2.;
    v.z += dt * f.z / 2.;
    bc64(x, v, a.bc, a.L);
    v3[0] = sq3(v);
    v3[1] = f.w;
    v3[2] = s[4];
    end_step64<DRIFT, LJ_EVN>(a, i, x, v, f);
    if constexpr (DRIFT) a.xn[i] = a.x[i];
  }
  small_row_sum<3, T>(v3);
  if (threadIdx.x == 0) {
    double* r = a.blk + (size_t)row * kBlkFields;
    r[BLK_K2] = v3[0];
    r[BLK_E] = v3[1];
    r[BLK_B] = v3[2];
  }
}

template <bool PERIODIC, int T, bool FIN>
__global__ __launch_bounds__(kSmallThreads) void k_small64_tvn(Step64 a, StepArgs fin)
{
#pragma clang fp contract(off)
  __shared__ Small64Lds<T> lds;
  if constexpr (FIN) {
    if (blockIdx.x == 0) {
      if (threadIdx.x < kBlock) step_observables<kWaves>(fin, fin.nrow, true, true);
      return;
    }
  }
  const int row = (int)blockIdx.x - (FIN ? 1 : 0);
  const int i = row * T + threadIdx.x;
  const bool lead = threadIdx.x < T && i < a.N;
  double s[5];
  small_forces64<PERIODIC, T>(lds, a.xs, a.N, row * T, a.L, a.sigma * a.sigma, s);
  if (threadIdx.x >= 64) return;
  double v3[3] = {0., 0., 0.};
  if (lead) {
    const double4 v = a.v[i];
    double4 tf = a.tf[i];
    const double4 f = finish_force(a, i, Sum64{s[0], s[1], s[2], s[3]});
    tf.x += 0.5 * f.x;
    tf.y += 0.5 * f.y;
    tf.z += 0.5 * f.z;
    a.tf[i] = tf;
    const double dt = a.dt;
    const double4 tv = make_double4(v.x + dt * tf.x / 2., v.y + dt * tf.y / 2., v.z + dt * tf.z / 2., 0.);
    v3[0] = sq3(tv);
    v3[1] = f.w;
    v3[2] = s[4];
  }
  small_row_sum<3, T>(v3);
  if (threadIdx.x == 0) {
    double* r = a.blk + (size_t)row * kBlkFields;
    r[BLK_K2] = 0.;  // k_tvn64_b writes the first rows' totals
    r[BLK_TV2] = v3[0];
    r[BLK_E] = v3[1];
    r[BLK_B] = v3[2];
  }
}

template <bool PERIODIC, int T>
void small64_evn_t(hipStream_t st, const Step64& a, bool drift_next, const StepArgs* fin)
{
  const dim3 g(a.nrow + (fin ? 1 : 0)), b(kSmallThreads);
  const StepArgs none{};
  if (drift_next) {
    if (fin) hipLaunchKernelGGL((k_small64_evn<PERIODIC, T, true, true>), g, b, 0, st, a, *fin);
    else hipLaunchKernelGGL((k_small64_evn<PERIODIC, T, true, false>), g, b, 0, st, a, none);
  } else {
    if (fin) hipLaunchKernelGGL((k_small64_evn<PERIODIC, T, false, true>), g, b, 0, st, a, *fin);
    else hipLaunchKernelGGL((k_small64_evn<PERIODIC, T, false, false>), g, b, 0, st, a, none);
  }
}

template <bool PERIODIC, int T>
void small64_tvn_t(hipStream_t st, const Step64& a, const StepArgs* fin)
{
  const dim3 g(a.nrow + (fin ? 1 : 0)), b(kSmallThreads);
  if (fin) hipLaunchKernelGGL((k_small64_tvn<PERIODIC, T, true>), g, b, 0, st, a, *fin);
  else hipLaunchKernelGGL((k_small64_tvn<PERIODIC, T, false>), g, b, 0, st, a, StepArgs{});
}

__global__ __launch_bounds__(kBlock) void k_widen(const float4* __restrict__ s, double4* __restrict__ d, int N)
{
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < N) {
    const float4 p = s[i];
    d[i] = make_double4(p.x, p.y, p.z, p.w);
  }
}

__global__ __launch_bounds__(kBlock) void k_narrow(const double4* __restrict__ s, float4* __restrict__ d, int N)
{
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < N) d[i] = narrow(s[i]);
}

__global__ __launch_bounds__(kBlock) void k_kinetic64(const double4* __restrict__ v, int N, double* blk)
{
  const int i = blockIdx.x * kBlock + threadIdx.x;
  double s[1] = {i < N ? sq3(v[i]) : 0.};
  const int fld[1] = {BLK_K2};
  block_sum_store<1>(s, blk + (size_t)blockIdx.x * kBlkFields, fld);
}

// RenormalizeVelocities (MDSystem.cpp:375-389) on the double velocities
__global__ __launch_bounds__(kBlock) void k_scale64(double4* __restrict__ v, float4* __restrict__ vel,
                                                    int N, const double* __restrict__ blk, int nblk,
                                                    double T0, double factor, lj_obs* obs)
{
  double Tkin = 0.;
  if (!(factor > 0.)) {
    Tkin = blk_total(blk, nblk, BLK_K2) * (1. / 3. / N);
    factor = sqrt(T0 / Tkin);
  }
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < N) {
    double4 w = v[i];
    w.x *= factor;
    w.y *= factor;
    w.z *= factor;
    v[i] = w;
    vel[i] = narrow(w);
  }
  if (blockIdx.x == 0 && threadIdx.x == 0 && obs) {
    if (Tkin > 0.) {
      obs->K *= T0 / Tkin;
      obs->T = T0;
    } else {
      obs->K *= factor * factor;
      obs->T *= factor * factor;
    }
    obs->U = obs->K + obs->V;
  }
}

__global__ __launch_bounds__(kBlock) void k_bc64(double4* __restrict__ x, double4* __restrict__ v,
                                                 float4* __restrict__ pos, float4* __restrict__ vel,
                                                 int N, int bc, double L)
{
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= N) return;
  double4 p = x[i], w = v[i];
  bc64(p, w, bc, L);
  x[i] = p;
  v[i] = w;
  pos[i] = narrow(p);
  vel[i] = narrow(w);
}

inline int nb(int n) { return (n + kBlock - 1) / kBlock; }

}  // namespace

// Pair-once from N = 4097 on, as long as its slots stay within 4 GiB (N about
// 180,000; a context that finds no room for them takes the sliced pass); measured
// steps (EVN, periodic, us; sliced / pair-once): N = 3000 26.5 /
// 24.1, 4000 31.0 / 32.5, 5000 42.0 / 35.9, 8000 77.9 / 62.2, 16384 273 / 190,
// 131072 16900 / 10700.  Split while the items fit two rounds of the 1024 workgroups
// that the kernel's registers let the device hold: their length is the granularity of the
// last round (split / unsplit: 8000 62 / 71, 12000 109 / 116, 16384 191 / 194, 40000
// 1104 / 1052, where the second set of slots costs more).
ForcePlan make_plan64(int N, int jslices)
{
  const int ng = (N + kG64 - 1) / kG64, nitems = ng * (ng + 1) / 2;
  const int split = nitems <= 2080 ? 2 : 1;
  const int Npad = (N + 63) & ~63;
  if (jslices > 0 || N <= 4096 || (double)ng * split * Npad * sizeof(double4) > 4294967296.)
    return make_force_plan(N, jslices, 1);
  ForcePlan pl;
  pl.N = N;
  pl.n3 = 2;
  pl.ng = ng;
  pl.nitems = pl.nitems_step = nitems;
  pl.split = split;
  pl.S = ng * split;
  pl.jchunk = kG64;
  pl.Npad = Npad;
  return pl;
}

int force64_totals(const ForcePlan& pl)
{
  return pl.n3 ? pl.nitems * pl.split : pl.gx * pl.S * kWaves;
}

hipError_t launch_force64(hipStream_t st, const ForcePlan& pl, const double4* x, bool periodic,
                          double L, double sigma, double4* part, double* wt)
{
  const double s2 = sigma * sigma;
  if (pl.n3) {
    const dim3 grid(pl.nitems * pl.split), b(kG64);
#define LJ_ARGS grid, b, 0, st, x, pl.items, pl.N, pl.Npad, L, 1. / L, s2, part, wt
    if (pl.split == 2) {
      if (periodic) hipLaunchKernelGGL((k_force64_n3<true, true>), LJ_ARGS);
      else hipLaunchKernelGGL((k_force64_n3<false, true>), LJ_ARGS);
    } else {
      if (periodic) hipLaunchKernelGGL((k_force64_n3<true, false>), LJ_ARGS);
      else hipLaunchKernelGGL((k_force64_n3<false, false>), LJ_ARGS);
    }
#undef LJ_ARGS
    return hipGetLastError();
  }
  dim3 grid(pl.gx, pl.S);
  if (periodic)
    hipLaunchKernelGGL(k_force64<true>, grid, dim3(kBlock), 0, st, x, pl.N, pl.Npad, pl.jchunk, L,
                       1. / L, s2, part, wt);
  else
    hipLaunchKernelGGL(k_force64<false>, grid, dim3(kBlock), 0, st, x, pl.N, pl.Npad, pl.jchunk,
                       L, 1. / L, s2, part, wt);
  return hipGetLastError();
}

hipError_t launch_reduce64(hipStream_t st, const Step64& a)
{
  hipLaunchKernelGGL(k_reduce64, dim3(a.nrow), dim3(kBlock), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_drift64(hipStream_t st, const Step64& a, int canonical)
{
  if (canonical == LJ_EVN)
    hipLaunchKernelGGL(k_drift64<LJ_EVN>, dim3(nb(a.N)), dim3(kBlock), 0, st, a);
  else
    hipLaunchKernelGGL(k_drift64<LJ_TVN>, dim3(nb(a.N)), dim3(kBlock), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_kick64(hipStream_t st, const Step64& a, bool drift_next, const StepArgs* fin)
{
  const dim3 g(a.nrow + (fin ? 1 : 0)), b(kBlock);
  const StepArgs none{};
  if (drift_next) {
    if (fin) hipLaunchKernelGGL((k_kick64<true, true>), g, b, 0, st, a, *fin);
    else hipLaunchKernelGGL((k_kick64<true, false>), g, b, 0, st, a, none);
  } else {
    if (fin) hipLaunchKernelGGL((k_kick64<false, true>), g, b, 0, st, a, *fin);
    else hipLaunchKernelGGL((k_kick64<false, false>), g, b, 0, st, a, none);
  }
  return hipGetLastError();
}

hipError_t launch_tvn64_a(hipStream_t st, const Step64& a, const StepArgs* fin)
{
  if (fin) hipLaunchKernelGGL(k_tvn64_a<true>, dim3(a.nrow + 1), dim3(kBlock), 0, st, a, *fin);
  else hipLaunchKernelGGL(k_tvn64_a<false>, dim3(a.nrow), dim3(kBlock), 0, st, a, StepArgs{});
  return hipGetLastError();
}

hipError_t launch_tvn64_b(hipStream_t st, const Step64& a, bool drift_next)
{
  if (drift_next) hipLaunchKernelGGL(k_tvn64_b<true>, dim3(nb(a.N)), dim3(kBlock), 0, st, a);
  else hipLaunchKernelGGL(k_tvn64_b<false>, dim3(nb(a.N)), dim3(kBlock), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_small_drift64(hipStream_t st, const Step64& a, int canonical)
{
  if (canonical == LJ_EVN)
    hipLaunchKernelGGL(k_small_drift64<LJ_EVN>, dim3(nb(a.N)), dim3(kBlock), 0, st, a);
  else
    hipLaunchKernelGGL(k_small_drift64<LJ_TVN>, dim3(nb(a.N)), dim3(kBlock), 0, st, a);
  return hipGetLastError();
}

#define LJ_SMALL_T(CALL)                  \
  switch (T) {                            \
    case 4: CALL(4); break;               \
    case 8: CALL(8); break;               \
    case 16: CALL(16); break;             \
    default: return hipErrorInvalidValue; \
  }

hipError_t launch_small64_evn(hipStream_t st, int T, const Step64& a, bool drift_next,
                              const StepArgs* fin)
{
#define LJ_CALL(K)                                                              \
  a.bc == LJ_BC_PERIODIC ? small64_evn_t<true, K>(st, a, drift_next, fin)       \
                         : small64_evn_t<false, K>(st, a, drift_next, fin)
  LJ_SMALL_T(LJ_CALL)
#undef LJ_CALL
  return hipGetLastError();
}

hipError_t launch_small64_tvn(hipStream_t st, int T, const Step64& a, const StepArgs* fin)
{
#define LJ_CALL(K)                                                  \
  a.bc == LJ_BC_PERIODIC ? small64_tvn_t<true, K>(st, a, fin)       \
                         : small64_tvn_t<false, K>(st, a, fin)
  LJ_SMALL_T(LJ_CALL)
#undef LJ_CALL
  return hipGetLastError();
}
#undef LJ_SMALL_T

hipError_t launch_widen(hipStream_t st, const float4* src, double4* dst, int N)
{
  hipLaunchKernelGGL(k_widen, dim3(nb(N)), dim3(kBlock), 0, st, src, dst, N);
  return hipGetLastError();
}

hipError_t launch_narrow(hipStream_t st, const double4* src, float4* dst, int N)
{
  hipLaunchKernelGGL(k_narrow, dim3(nb(N)), dim3(kBlock), 0, st, src, dst, N);
  return hipGetLastError();
}

hipError_t launch_kinetic64(hipStream_t st, const double4* v, int N, double* blk)
{
  hipLaunchKernelGGL(k_kinetic64, dim3(nb(N)), dim3(kBlock), 0, st, v, N, blk);
  return hipGetLastError();
}

hipError_t launch_scale64(hipStream_t st, double4* v, float4* vel, int N, const double* blk,
                          int nblk, double T0, double factor, lj_obs* obs)
{
  hipLaunchKernelGGL(k_scale64, dim3(nb(N)), dim3(kBlock), 0, st, v, vel, N, blk, nblk, T0, factor,
                     obs);
  return hipGetLastError();
}

hipError_t launch_bc64(hipStream_t st, double4* x, double4* v, float4* pos, float4* vel, int N,
                       int bc, double L)
{
  hipLaunchKernelGGL(k_bc64, dim3(nb(N)), dim3(kBlock), 0, st, x, v, pos, vel, N, bc, L);
  return hipGetLastError();
}

}  // namespace lj
