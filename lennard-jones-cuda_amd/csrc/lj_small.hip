// lj_small.hip -- the time step of small boxes in one launch (EVN) or two
// (TVN): the workgroup that computes the whole force on its particles also
// runs their integrator (reference MDSystem.cpp:438-583), so that no partial
// sums pass through memory and no launch waits for another inside a step.
//
// A step of a small box is a chain of latencies: at N = 400 its 80,000 pairs
// are 0.05 us of the device's FP32 rate, an empty kernel in a chain of graph
// nodes takes 1.8 us, and the force pass, kick and finaliser took 11.0 us.
// Here the step is 4.6 us: the launch, one load of all coordinates, the pairs
// of a lane, two passes through LDS and the stores.  From about N = 1500 on the
// pair loop is visible, and at N = 4096 it is 9.4 us of the 14, which is the issue
// time of its 22 slots per ordered pair.
#include "lj_small.h"

namespace lj {

namespace {

using namespace dev;

template <bool PERIODIC, int CANON>
__global__ __launch_bounds__(kBlock) void k_small_drift(StepArgs a)
{
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= a.N) return;
  float4 p = a.pos[i];
  float4 v = a.vel[i];
  float4 tf;
  drift_one<CANON>(p, v, tf, a.force[i], a.dt);
  if constexpr (CANON == LJ_EVN) a.vel[i] = v;
  else a.tF[i] = tf;
  a.pos[i] = p;
  a.q[i] = small_q<PERIODIC>(p, a.qscale);
}

// DRIFT: also the next step's drift (its coordinates go to a.qn, since other
// workgroups still read a.q); FIN: block 0 computes the observables of the
// run's previous step.
template <bool PERIODIC, int T, bool DRIFT, bool FIN>
__global__ __launch_bounds__(kSmallThreads) __attribute__((amdgpu_waves_per_eu(8))) void k_small_evn(
    StepArgs a, StepArgs fin, float C1)
{
#pragma clang fp contract(off)
  __shared__ SmallLds<T> lds;
  if constexpr (FIN) {
    if (blockIdx.x == 0) {
      // by the threads of the stand-alone finaliser: the same bits
      if (threadIdx.x < kBlock) step_observables<kWaves>(fin, fin.nrow, true, true);
      return;
    }
  }
  const int row = (int)blockIdx.x - (FIN ? 1 : 0);
  const int i = row * T + threadIdx.x;
  const bool lead = threadIdx.x < T && i < a.N;
  // the particles' own loads go out ahead of the pair loop
  float4 v = {}, p = {};
  if (lead) {
    v = a.vel[i];
    p = a.pos[i];
  }
  const Partial s = small_forces<PERIODIC, T>(lds, a.q, a.N, row * T, C1);
  if (threadIdx.x >= 64) return;
  double v3[3] = {0., 0., 0.};
  if (lead) {
    const double e = 0.5 * (s.b - s.a);
    const float fx = (float)(a.FS * s.fx), fy = (float)(a.FS * s.fy), fz = (float)(a.FS * s.fz);
    a.force[i] = make_float4(fx, fy, fz, a.keep_w ? (float)e : 0.f);
    const double dt = a.dt;
    v.x = (float)(v.x + dt * fx / 2.);  // MDSystem.cpp:460-462
    v.y = (float)(v.y + dt * fy / 2.);
    v.z = (float)(v.z + dt * fz / 2.);
    apply_bc_one(p, v, a.bc, a.L);
    if (!DRIFT && PERIODIC) a.pos[i] = p;
    v3[0] = kin2(v);
    v3[1] = e;
    v3[2] = s.b;
    if constexpr (DRIFT) {
      float4 tf;
      drift_one<LJ_EVN>(p, v, tf, make_float4(fx, fy, fz, 0.f), dt);
      a.pos[i] = p;
      a.qn[i] = small_q<PERIODIC>(p, a.qscale);
    }
    a.vel[i] = v;
  }
  small_row_sum<3, T>(v3);
  if (threadIdx.x == 0) {
    double* r = a.blk + (size_t)row * kBlkFields;
    r[BLK_K2] = v3[0];
    r[BLK_E] = v3[1];
    r[BLK_B] = v3[2];
  }
}

// first half of the TVN step (k_tvn_b follows): forces, half-step velocities
template <bool PERIODIC, int T, bool FIN>
__global__ __launch_bounds__(kSmallThreads) __attribute__((amdgpu_waves_per_eu(8))) void k_small_tvn(
    StepArgs a, StepArgs fin, float C1)
{
#pragma clang fp contract(off)
  __shared__ SmallLds<T> lds;
  if constexpr (FIN) {
    if (blockIdx.x == 0) {
      // by the threads of the stand-alone finaliser: the same bits
      if (threadIdx.x < kBlock) step_observables<kWaves>(fin, fin.nrow, true, true);
      return;
    }
  }
  const int row = (int)blockIdx.x - (FIN ? 1 : 0);
  const int i = row * T + threadIdx.x;
  const bool lead = threadIdx.x < T && i < a.N;
  float4 v = {}, tf = {};
  if (lead) {
    v = a.vel[i];
    tf = a.tF[i];
  }
  const Partial s = small_forces<PERIODIC, T>(lds, a.q, a.N, row * T, C1);
  if (threadIdx.x >= 64) return;
  double v3[3] = {0., 0., 0.};
  if (lead) {
    const double e = 0.5 * (s.b - s.a);
    const float fx = (float)(a.FS * s.fx), fy = (float)(a.FS * s.fy), fz = (float)(a.FS * s.fz);
    a.force[i] = make_float4(fx, fy, fz, a.keep_w ? (float)e : 0.f);
    tf.x += 0.5f * fx;  // MDSystem.cpp:486-488
    tf.y += 0.5f * fy;
    tf.z += 0.5f * fz;
    a.tF[i] = tf;
    const double dt = a.dt;
    float4 tv;
    tv.x = (float)(v.x + dt * tf.x / 2.);  // MDSystem.cpp:493-495
    tv.y = (float)(v.y + dt * tf.y / 2.);
    tv.z = (float)(v.z + dt * tf.z / 2.);
    tv.w = 0.f;
    v3[0] = kin2(tv);
    v3[1] = e;
    v3[2] = s.b;
  }
  small_row_sum<3, T>(v3);
  if (threadIdx.x == 0) {
    double* r = a.blk + (size_t)row * kBlkFields;
    r[BLK_K2] = 0.;  // k_tvn_b writes the first step_rows(N) rows' totals
    r[BLK_TV2] = v3[0];
    r[BLK_E] = v3[1];
    r[BLK_B] = v3[2];
  }
}

template <bool PERIODIC, int T>
void small_evn_t(hipStream_t st, const StepArgs& a, float C1, bool drift_next, const StepArgs* fin)
{
  const dim3 g(a.nrow + (fin ? 1 : 0)), b(kSmallThreads);
  if (drift_next) {
    if (fin) hipLaunchKernelGGL((k_small_evn<PERIODIC, T, true, true>), g, b, 0, st, a, *fin, C1);
    else hipLaunchKernelGGL((k_small_evn<PERIODIC, T, true, false>), g, b, 0, st, a, a, C1);
  } else {
    if (fin) hipLaunchKernelGGL((k_small_evn<PERIODIC, T, false, true>), g, b, 0, st, a, *fin, C1);
    else hipLaunchKernelGGL((k_small_evn<PERIODIC, T, false, false>), g, b, 0, st, a, a, C1);
  }
}

template <bool PERIODIC, int T>
void small_tvn_t(hipStream_t st, const StepArgs& a, float C1, const StepArgs* fin)
{
  const dim3 g(a.nrow + (fin ? 1 : 0)), b(kSmallThreads);
  if (fin) hipLaunchKernelGGL((k_small_tvn<PERIODIC, T, true>), g, b, 0, st, a, *fin, C1);
  else hipLaunchKernelGGL((k_small_tvn<PERIODIC, T, false>), g, b, 0, st, a, a, C1);
}

}  // namespace

// The smallest tile that gives at most one workgroup per CU (256), up to 16
// particles: a smaller tile shortens every lane's chain of pairs, a second
// workgroup on a CU doubles it.  Measured EVN steps at T = 4 / 8 / 16 (us; the
// separate kernels in brackets): N = 400 4.6 / 4.7 / 5.2 [11.0], 1000 4.9 / 5.3 /
// 6.5 [11.3], 1500 6.6 / 5.9 / 7.6 [11.7], 2048 8.8 / 7.6 / 8.7 [12.6], 3000
// 12.0 / 11.0 / 11.2 [15.3], 4096 18.1 / 14.4 / 14.2 [18.2]; TVN steps are 2.5
// to 3 us longer (4096: 17.3 [21.3]).  Beyond 4096 every pair from both sides
// costs more than the pair-once pass and its sums save (5003: 21.7 [19.3]).
int small_tile(int N)
{
  for (int T = 4; T <= 16; T *= 2)
    if (N <= 256 * T) return T;
  return 0;
}

hipError_t launch_small_drift(hipStream_t st, const StepArgs& a)
{
  const dim3 g((a.N + kBlock - 1) / kBlock), b(kBlock);
  const bool per = a.bc == LJ_BC_PERIODIC;
  if (a.canonical == LJ_EVN) {
    if (per) hipLaunchKernelGGL((k_small_drift<true, LJ_EVN>), g, b, 0, st, a);
    else hipLaunchKernelGGL((k_small_drift<false, LJ_EVN>), g, b, 0, st, a);
  } else {
    if (per) hipLaunchKernelGGL((k_small_drift<true, LJ_TVN>), g, b, 0, st, a);
    else hipLaunchKernelGGL((k_small_drift<false, LJ_TVN>), g, b, 0, st, a);
  }
  return hipGetLastError();
}

#define LJ_SMALL_T(CALL)                  \
  switch (T) {                            \
    case 4: CALL(4); break;               \
    case 8: CALL(8); break;               \
    case 16: CALL(16); break;             \
    default: return hipErrorInvalidValue; \
  }

hipError_t launch_small_evn(hipStream_t st, int T, const StepArgs& a, float C1, bool drift_next,
                            const StepArgs* fin)
{
#define LJ_CALL(K)                                                                        \
  do {                                                                                    \
    if (a.bc == LJ_BC_PERIODIC) small_evn_t<true, K>(st, a, C1, drift_next, fin);         \
    else small_evn_t<false, K>(st, a, C1, drift_next, fin);                               \
  } while (0)
  LJ_SMALL_T(LJ_CALL)
#undef LJ_CALL
  return hipGetLastError();
}

hipError_t launch_small_tvn(hipStream_t st, int T, const StepArgs& a, float C1, const StepArgs* fin)
{
#define LJ_CALL(K)                                                        \
  do {                                                                    \
    if (a.bc == LJ_BC_PERIODIC) small_tvn_t<true, K>(st, a, C1, fin);     \
    else small_tvn_t<false, K>(st, a, C1, fin);                           \
  } while (0)
  LJ_SMALL_T(LJ_CALL)
#undef LJ_CALL
  return hipGetLastError();
}

}  // namespace lj
