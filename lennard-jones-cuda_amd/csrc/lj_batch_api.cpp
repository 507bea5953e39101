// lj_batch_api.cpp -- C-ABI of the batched ensemble (many boxes, one launch
// per kernel per step, captured in a HIP graph) and its autotuner.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <fstream>
#include <sstream>
#include <string>
#include <vector>

#include "lj_fluct.h"
#include "lj_internal.h"
#include "lj_util.h"

using namespace lj;

namespace {
// the tuning of a new batch: its steps are one launch where that is faster
// (small_steps), else this tiling's; single evaluations use the tiling
constexpr lj_batch_tuning kDefaultTuning{1, 512, 8, 0};
}  // namespace

struct lj_batch {
  int device = 0;
  int nboxes = 0;
  int canonical = LJ_EVN;
  int boundary = LJ_BC_PERIODIC;
  double eps = 1.0;
  int ncu = 256;
  std::vector<int> N;
  std::vector<double> rho, T0, L;
  std::vector<int> off;
  int Ntot = 0;
  double sub_fraction = 0.5;
  lj_batch_tuning tune = kDefaultTuning;
  bool ready = false;  // the tuning's tables stand
  hipStream_t stream = nullptr;
  // device
  float4 *pos = nullptr, *vel = nullptr, *force = nullptr, *tF = nullptr;
  uint4* q = nullptr;
  float4* fpart = nullptr;
  float* apart = nullptr;
  size_t part_cap = 0;
  double* blk = nullptr;
  // one-launch steps (small; with the default tuning): the other coordinate buffer,
  // the tiles, the boxes with the tiles' rows, and two buffers of block rows that
  // the steps alternate between
  bool small = false;
  uint4* q2 = nullptr;
  BoxParam* box_s = nullptr;
  int2* tiles = nullptr;
  double* blk_s = nullptr;
  int ntiles = 0;
  lj_obs* obs = nullptr;
  double* stats = nullptr;
  BoxParam* box = nullptr;
  int2* pblock = nullptr;
  BatchItem* items = nullptr;
  size_t items_cap = 0;
  double* ew = nullptr;  // pair-once: (E, W) per item, boxes' runs contiguous
  size_t ew_cap = 0;
  unsigned* counter = nullptr;
  int nblocks = 0, nitems = 0;
  std::vector<BoxParam> hbox;
  hipGraph_t graph = nullptr;  // one step
  hipGraphExec_t gexec = nullptr;
  hipGraph_t graph_run = nullptr;  // kGraphSteps steps back to back
  hipGraphExec_t gexec_run = nullptr;
  double g_dt = 0.;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  // fluctuation counters of every box (lj_batch_fl_*), sampled after every
  // step when smp_fl is set
  FlSampler fl;
  int smp_fl = 0;
  // per-step history of lj_batch_integrate_hist (hist_cap steps of nboxes rows)
  double* hist = nullptr;
  int64_t* hist_base = nullptr;
  int hist_cap = 0;
};

namespace {

void bdrop_graph(lj_batch* b)
{
  if (b->gexec) (void)hipGraphExecDestroy(b->gexec);
  if (b->graph) (void)hipGraphDestroy(b->graph);
  if (b->gexec_run) (void)hipGraphExecDestroy(b->gexec_run);
  if (b->graph_run) (void)hipGraphDestroy(b->graph_run);
  b->gexec = nullptr;
  b->graph = nullptr;
  b->gexec_run = nullptr;
  b->graph_run = nullptr;
}

int bsetdev(lj_batch* b)
{
  if (!b) return fail(LJ_ERR_ARG, "null batch");
  LJ_HIP(hipSetDevice(b->device));
  return LJ_OK;
}

int bready(lj_batch* b)
{
  LJ_TRY(bsetdev(b));
  if (!b->ready) return fail(LJ_ERR_STATE, "the batch has no tables (no room at lj_batch_set_tuning)");
  return LJ_OK;
}

// lean: the time step's force pass (force-only partials and per-item totals
// when the pair-once decomposition is tuned in)
BatchArgs bargs(lj_batch* b, double dt, bool lean = false)
{
  BatchArgs a{};
  a.pos = b->pos;
  a.vel = b->vel;
  a.force = b->force;
  a.tF = b->tF;
  a.q = b->q;
  a.fpart = b->fpart;
  a.apart = b->apart;
  a.blk = b->blk;
  a.obs = b->obs;
  a.stats = b->stats;
  a.box = b->box;
  a.pblock = b->pblock;
  a.items = b->items;
  a.counter = b->counter;
  a.nboxes = b->nboxes;
  a.nblocks = b->nblocks;
  a.nitems = b->nitems;
  a.dt = dt;
  a.eps = b->eps;
  a.bc = b->boundary;
  a.canonical = b->canonical;
  a.ipl = b->tune.ipl;
  a.persistent_grid = b->tune.blocks_per_cu > 0 ? b->tune.blocks_per_cu * b->ncu : 0;
  a.pair_once = b->tune.pair_once;
  a.lean = lean && a.pair_once ? 1 : 0;
  a.ew = b->ew;
  a.hist = b->hist;
  a.hist_base = b->hist_base;
  a.hist_cap = b->hist_cap;
  return a;
}

// a one-launch step; par: its parity in the run
BatchArgs small_args(lj_batch* b, double dt, int par)
{
  BatchArgs a = bargs(b, dt);
  const bool swap = par && b->canonical == LJ_EVN;
  a.q = swap ? b->q2 : b->q;
  a.qn = swap ? b->q : b->q2;
  a.box = b->box_s;
  a.blk = b->blk_s + (size_t)par * b->ntiles * kBlkFields;
  a.ntiles = b->ntiles;
  a.tiles = b->tiles;
  return a;
}

bool default_tuning(const lj_batch_tuning& t)
{
  const lj_batch_tuning& d = kDefaultTuning;
  return t.ipl == d.ipl && t.jchunk == d.jchunk && t.blocks_per_cu == d.blocks_per_cu &&
         t.pair_once == d.pair_once;
}

// Whether a batch with the default tuning takes the one-launch step.  A tile costs it a workgroup
// of 1024 threads, 8.7e-3 us however few particles its box has; the four launches
// of the default tiling cost 105 to 145 us a step and then less per tile: 4.4e-3 us
// up to 512 particles a box, 7.5e-3 (one launch: 11.8e-3) at 1000, 14.2e-3 (16.3e-3) at
// 2000.  EVN steps, us, one launch / tiling: 327 boxes of 200 41 / 130, 1310 154 / 186,
// 2621 300 / 261, 5242 594 / 407; 655 of 400 157 / 193, 1310 308 / 268; 262 of 1000
// 202 / 262, 524 393 / 390, 1048 778 / 640; 262 of 2000 539 / 617, 524 1068 / 1071; 131 of
// 4000 1005 / 1057; one of 100,000 4388 / 4397.  So the line lies at 24,576 tiles of
// boxes up to 512 particles, 32,768 up to 1200 and 49,152 above.
bool small_steps(const std::vector<int>& N)
{
  long units = 0;
  for (int n : N) units += (long)((n + kBatchTile - 1) / kBatchTile) * (n <= 512 ? 4 : n <= 1200 ? 3 : 2);
  return units <= 4 * 24576;
}

// tables of the one-launch steps, from the boxes' parameters
int build_small(lj_batch* b, const std::vector<BoxParam>& bp)
{
  b->small = default_tuning(b->tune) && small_steps(b->N);
  if (!b->small) return LJ_OK;
  const int T = kBatchTile;
  std::vector<BoxParam> bs = bp;
  std::vector<int2> tiles;
  for (int k = 0; k < b->nboxes; ++k) {
    bs[k].blk0 = (int)tiles.size();
    bs[k].nblk = (b->N[k] + T - 1) / T;
    for (int t = 0; t < bs[k].nblk; ++t) tiles.push_back(make_int2(k, t * T));
  }
  // the boxes' rows stay in box order; the tiles with the longest chains first
  std::stable_sort(tiles.begin(), tiles.end(),
                   [&](const int2& x, const int2& y) { return b->N[x.x] > b->N[y.x]; });
  b->ntiles = (int)tiles.size();
  if (!b->q2) LJ_TRY(dev_alloc(&b->q2, b->Ntot));
  if (!b->box_s) LJ_TRY(dev_alloc(&b->box_s, b->nboxes));
  if (!b->tiles) LJ_TRY(dev_alloc(&b->tiles, tiles.size()));
  if (!b->blk_s) LJ_TRY(dev_alloc(&b->blk_s, (size_t)2 * tiles.size() * kBlkFields));
  LJ_HIP(hipMemcpyAsync(b->box_s, bs.data(), sizeof(BoxParam) * bs.size(), hipMemcpyHostToDevice,
                        b->stream));
  LJ_HIP(hipMemcpyAsync(b->tiles, tiles.data(), sizeof(int2) * tiles.size(), hipMemcpyHostToDevice,
                        b->stream));
  LJ_HIP(hipStreamSynchronize(b->stream));
  return LJ_OK;
}

// (re)build the per-box tables and the work items for the current tuning
int build_tables(lj_batch* b)
{
  const int ipl = b->tune.ipl;
  const int tile = 64 * ipl;
  const int jc0 = b->tune.jchunk;
  std::vector<BoxParam> bp(b->nboxes);
  std::vector<int2> pblock;
  std::vector<BatchItem> items;
  size_t pbase = 0;
  int blk0 = 0;
  for (int k = 0; k < b->nboxes; ++k) {
    const int N = b->N[k];
    BoxParam& p = bp[k];
    std::memset(&p, 0, sizeof(p));
    p.N = N;
    p.off = b->off[k];
    int jc = std::min(jc0, (N + 7) & ~7);
    jc = (jc + 7) & ~7;
    if (b->tune.pair_once) jc = kPairOnceGroup;  // one partial slot per group
    p.jchunk = jc;
    p.S = (N + jc - 1) / jc;
    p.Npad = (N + 63) & ~63;
    p.pbase = (int)pbase;
    pbase += (size_t)p.S * p.Npad;
    p.nblk = (N + kBlock - 1) / kBlock;
    p.blk0 = blk0;
    for (int t = 0; t < p.nblk; ++t) pblock.push_back(make_int2(k, t * kBlock));
    blk0 += p.nblk;
    const PairScalars ps = make_pair_scalars(b->L[k], b->boundary == LJ_BC_PERIODIC, b->eps, 1.0, false);
    p.L = b->L[k];
    p.qscale = ps.qscale;
    p.FS = ps.FS;
    p.C1 = ps.C1;
    p.rho = b->rho[k];
    p.T0 = b->T0[k];
    const double side = b->L[k] * std::cbrt(b->sub_fraction);  // MDSystem.cpp:711
    p.sub_lo = 0.5 * b->L[k] - 0.5 * side;
    p.sub_hi = 0.5 * b->L[k] + 0.5 * side;
    if (b->tune.pair_once) {
      p.ew0 = (int)items.size();
      for (int g = 0; g < p.S; ++g)
        for (int h = g; h < p.S; ++h) items.push_back(BatchItem{k, g, h, (int)items.size()});
      p.nitem = (int)items.size() - p.ew0;
    } else {
      for (int t = 0; t < (N + tile - 1) / tile; ++t)
        for (int s = 0; s < p.S; ++s) items.push_back(BatchItem{k, t * tile, s, 0});
    }
  }
  if (pbase > (size_t)0x7fffffff) return fail(LJ_ERR_UNSUPPORTED, "batch partial buffer too large");
  // longest items first (pairs per item), boxes with larger N first on ties
  std::stable_sort(items.begin(), items.end(), [&](const BatchItem& x, const BatchItem& y) {
    auto cost = [&](const BatchItem& w) {
      const BoxParam& p = bp[w.box];
      if (b->tune.pair_once) {  // pairs of the two groups (a diagonal item has half)
        const long long G = kPairOnceGroup;
        const long long ni = std::min(G, (long long)p.N - w.i0 * G);
        const long long nj = std::min(G, (long long)p.N - w.s * G);
        return w.i0 == w.s ? ni * nj / 2 : ni * nj;
      }
      const long long ni = std::min(tile, p.N - w.i0);
      const long long nj = std::min(p.jchunk, p.N - w.s * p.jchunk);
      return ni * nj;
    };
    const long long cx = cost(x), cy = cost(y);
    if (cx != cy) return cx > cy;
    return bp[x.box].N > bp[y.box].N;
  });
  LJ_HIP(hipStreamSynchronize(b->stream));
  // the captured steps hold the tables' addresses; a failure below leaves none
  bdrop_graph(b);
  b->ready = false;
  if (pbase > b->part_cap) {
    dev_free(b->fpart);
    dev_free(b->apart);
    b->part_cap = 0;
    LJ_TRY(dev_alloc(&b->fpart, pbase));
    LJ_TRY(dev_alloc(&b->apart, pbase));
    b->part_cap = pbase;
  }
  if (items.size() > b->items_cap) {
    dev_free(b->items);
    b->items_cap = 0;
    LJ_TRY(dev_alloc(&b->items, items.size()));
    b->items_cap = items.size();
  }
  if (b->tune.pair_once && items.size() > b->ew_cap) {
    dev_free(b->ew);
    b->ew_cap = 0;
    LJ_TRY(dev_alloc(&b->ew, 2 * items.size()));
    b->ew_cap = items.size();
  }
  if (!b->box) LJ_TRY(dev_alloc(&b->box, b->nboxes));
  if (!b->pblock) LJ_TRY(dev_alloc(&b->pblock, pblock.size()));
  if (!b->blk) LJ_TRY(dev_alloc(&b->blk, (size_t)blk0 * kBlkFields));
  // on the batch's stream: a null-stream copy can break another thread's capture
  LJ_HIP(hipMemcpyAsync(b->box, bp.data(), sizeof(BoxParam) * bp.size(), hipMemcpyHostToDevice,
                        b->stream));
  LJ_HIP(hipMemcpyAsync(b->pblock, pblock.data(), sizeof(int2) * pblock.size(), hipMemcpyHostToDevice,
                        b->stream));
  LJ_HIP(hipMemcpyAsync(b->items, items.data(), sizeof(BatchItem) * items.size(),
                        hipMemcpyHostToDevice, b->stream));
  LJ_HIP(hipStreamSynchronize(b->stream));
  LJ_TRY(build_small(b, bp));
  b->hbox = bp;
  b->nblocks = (int)pblock.size();
  b->nitems = (int)items.size();
  b->ready = true;
  return LJ_OK;
}

// one step of a run captured together: the first starts with the drift, each
// later one finds it done by the previous step's kick kernel (drift_next), with
// the same arithmetic, so a run gives the bits of single steps
int enqueue_batch_step(lj_batch* b, hipStream_t st, double dt, bool first = true, bool last = true,
                       int par = 0)
{
  if (b->small) {
    const BatchArgs a = small_args(b, dt, par), prev = small_args(b, dt, par ^ 1);
    if (first) LJ_HIP(launch_batch_drift(st, a));
    if (b->canonical == LJ_EVN) {
      LJ_HIP(launch_batch_small_evn(st, a, !last, first ? nullptr : &prev));
    } else {
      LJ_HIP(launch_batch_small_tvn(st, a, first ? nullptr : &prev));
      LJ_HIP(launch_batch_tvn_b(st, a, !last));
    }
    if (last) LJ_HIP(launch_batch_finalize(st, a, 1));
    if (b->smp_fl)
      LJ_HIP(launch_fl_sample(st, b->fl, b->pos, b->vel, 0, b->box, b->pblock, b->nblocks));
    return LJ_OK;
  }
  const BatchArgs a = bargs(b, dt, true);
  if (first) LJ_HIP(launch_batch_drift(st, a));
  LJ_HIP(launch_batch_force(st, a, b->boundary == LJ_BC_PERIODIC, false));
  if (b->canonical == LJ_EVN) {
    LJ_HIP(launch_batch_kick_evn(st, a, !last));
  } else {
    LJ_HIP(launch_batch_tvn_a(st, a));
    LJ_HIP(launch_batch_tvn_b(st, a, !last));
  }
  LJ_HIP(launch_batch_finalize(st, a, 1));
  if (b->smp_fl)
    LJ_HIP(launch_fl_sample(st, b->fl, b->pos, b->vel, 0, b->box, b->pblock, b->nblocks));
  return LJ_OK;
}

int capture_batch_steps(lj_batch* b, double dt, int steps, hipGraph_t* graph, hipGraphExec_t* exec)
{
  hipStream_t st = b->stream;
  LJ_HIP(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
  int rc = LJ_OK;
  // steps that sample end with their own final state (no drift of the next
  // step fused into their kick kernels)
  const bool alone = b->smp_fl != 0;
  for (int k = 0; k < steps && rc == LJ_OK; ++k)
    rc = enqueue_batch_step(b, st, dt, alone || k == 0, alone || k == steps - 1, k & 1);
  hipGraph_t g = nullptr;
  hipError_t ee = hipStreamEndCapture(st, &g);
  if (rc != LJ_OK) {
    if (g) (void)hipGraphDestroy(g);
    return rc;
  }
  LJ_HIP(ee);
  *graph = g;
  LJ_HIP(hipGraphInstantiate(exec, g, nullptr, nullptr, 0));
  return LJ_OK;
}

// lean: the time step's pass (with pair_once: force-only partials and
// per-item totals), as timed by lj_batch_time_force and the autotuner
int enqueue_batch_forces(lj_batch* b, hipStream_t st, bool ties, bool lean = false)
{
  const BatchArgs a = bargs(b, 0., lean);
  LJ_HIP(launch_batch_prep_q(st, a));  // also resets the queue head
  LJ_HIP(launch_batch_force(st, a, b->boundary == LJ_BC_PERIODIC, ties));
  return LJ_OK;
}

// us of one of the batch's steps as it is tuned now: replays of a captured run, on
// copies of the state
int time_steps(lj_batch* b, int reps, double* us)
{
  struct Copies {
    lj_batch* b;
    float4 *pos = b->pos, *vel = b->vel, *force = b->force, *tF = b->tF;  // the batch's own
    lj_obs* own_obs = b->obs;
    double *own_stats = b->stats, *hist = b->hist;
    int smp_fl = b->smp_fl;
    float4* state = nullptr;
    lj_obs* obs = nullptr;
    double* stats = nullptr;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    ~Copies()
    {
      (void)hipStreamSynchronize(b->stream);
      b->pos = pos, b->vel = vel, b->force = force, b->tF = tF;
      b->obs = own_obs, b->stats = own_stats, b->hist = hist, b->smp_fl = smp_fl;
      if (exec) (void)hipGraphExecDestroy(exec);
      if (graph) (void)hipGraphDestroy(graph);
      dev_free(state);
      dev_free(obs);
      dev_free(stats);
    }
  } c{b};
  const size_t n = b->Ntot;
  hipStream_t st = b->stream;
  LJ_TRY(dev_alloc(&c.state, 4 * n));
  LJ_TRY(dev_alloc(&c.obs, b->nboxes));
  LJ_TRY(dev_alloc(&c.stats, (size_t)b->nboxes * kNStat));
  const auto copy = [st](void* d, const void* s, size_t bytes) {
    return hipMemcpyAsync(d, s, bytes, hipMemcpyDeviceToDevice, st);
  };
  LJ_HIP(copy(c.state, b->pos, sizeof(float4) * n));
  LJ_HIP(copy(c.state + n, b->vel, sizeof(float4) * n));
  LJ_HIP(copy(c.state + 2 * n, b->force, sizeof(float4) * n));
  LJ_HIP(copy(c.state + 3 * n, b->tF, sizeof(float4) * n));
  LJ_HIP(copy(c.obs, b->obs, sizeof(lj_obs) * b->nboxes));
  LJ_HIP(copy(c.stats, b->stats, sizeof(double) * b->nboxes * kNStat));
  b->pos = c.state, b->vel = c.state + n, b->force = c.state + 2 * n, b->tF = c.state + 3 * n;
  b->obs = c.obs, b->stats = c.stats, b->hist = nullptr, b->smp_fl = 0;
  LJ_HIP(hipStreamSynchronize(st));
  LJ_TRY(capture_batch_steps(b, 0., kGraphSteps, &c.graph, &c.exec));
  LJ_HIP(hipGraphLaunch(c.exec, st));  // warm
  LJ_HIP(hipEventRecord(b->e0, st));
  for (int k = 0; k < reps; ++k) LJ_HIP(hipGraphLaunch(c.exec, st));
  LJ_HIP(hipEventRecord(b->e1, st));
  LJ_HIP(hipEventSynchronize(b->e1));
  float ms = 0.f;
  LJ_HIP(hipEventElapsedTime(&ms, b->e0, b->e1));
  *us = 1000.0 * ms / reps / kGraphSteps;
  return LJ_OK;
}

std::string tune_key(lj_batch* b)
{
  hipDeviceProp_t prop;
  std::string dev = "gfx";
  if (hipGetDeviceProperties(&prop, b->device) == hipSuccess) dev = prop.gcnArchName;
  unsigned long long h = 1469598103934665603ull;  // FNV-1a over the box sizes
  for (int n : b->N) {
    h ^= (unsigned long long)n;
    h *= 1099511628211ull;
  }
  std::ostringstream os;
  os << "v5:" << dev << ":" << b->ncu << ":" << b->nboxes << ":" << b->boundary << ":" << std::hex << h;
  return os.str();
}

}  // namespace

extern "C" {

int lj_batch_create(int nboxes, const int* N, const double* rho, const double* T0, int canonical,
                    int boundary, int device, lj_batch** out)
{
  if (!out || !N || !rho || !T0) return fail(LJ_ERR_ARG, "lj_batch_create: null argument");
  *out = nullptr;
  if (nboxes <= 0) return fail(LJ_ERR_ARG, "lj_batch_create: nboxes must be positive");
  if (canonical != 0 && canonical != 1) return fail(LJ_ERR_ARG, "lj_batch_create: canonical must be 0 or 1");
  if (boundary < 0 || boundary > 2) return fail(LJ_ERR_ARG, "lj_batch_create: boundary must be 0, 1 or 2");
  long long tot = 0;
  for (int k = 0; k < nboxes; ++k) {
    if (N[k] <= 0 || !(rho[k] > 0.) || !(T0[k] >= 0.))
      return fail(LJ_ERR_ARG, "lj_batch_create: box %d has N=%d rho=%g T0=%g", k, N[k], rho[k], T0[k]);
    tot += N[k];
  }
  if (tot > (1ll << 28)) return fail(LJ_ERR_ARG, "lj_batch_create: too many particles (%lld)", tot);
  LJ_TRY(check_device());
  LJ_HIP(hipSetDevice(device));
  lj_batch* b = new lj_batch();
  b->device = device;
  b->nboxes = nboxes;
  b->canonical = canonical;
  b->boundary = boundary;
  b->N.assign(N, N + nboxes);
  b->rho.assign(rho, rho + nboxes);
  b->T0.assign(T0, T0 + nboxes);
  int off = 0;
  for (int k = 0; k < nboxes; ++k) {
    b->off.push_back(off);
    off += N[k];
    b->L.push_back(box_length(N[k], rho[k]));
  }
  b->Ntot = off;
  int ncu = 0;
  if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess && ncu > 0)
    b->ncu = ncu;
  int rc = LJ_OK;
  auto A = [&](int r) { if (rc == LJ_OK) rc = r; };
  if (hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess) {
    b->stream = nullptr;
    A(fail(LJ_ERR_DEVICE, "hipStreamCreate failed"));
  }
  A(dev_alloc(&b->pos, off));
  A(dev_alloc(&b->vel, off));
  A(dev_alloc(&b->force, off));
  A(dev_alloc(&b->tF, off));
  A(dev_alloc(&b->q, off));
  A(dev_alloc(&b->obs, nboxes));
  A(dev_alloc(&b->stats, (size_t)nboxes * kNStat));
  A(dev_alloc(&b->counter, 1));
  if (rc == LJ_OK && (hipEventCreate(&b->e0) != hipSuccess || hipEventCreate(&b->e1) != hipSuccess))
    A(fail(LJ_ERR_DEVICE, "hipEventCreate failed"));
  if (rc == LJ_OK) A(build_tables(b));
  if (rc == LJ_OK) {
    std::vector<float> z((size_t)4 * off, 0.f);
    std::vector<lj_obs> o(nboxes);
    std::memset(o.data(), 0, sizeof(lj_obs) * nboxes);
    std::vector<double> zs((size_t)nboxes * kNStat, 0.);
    const size_t bytes = sizeof(float4) * (size_t)off;
    hipStream_t st = b->stream;
    const auto up = [st](void* d, const void* h, size_t n) {
      return hipMemcpyAsync(d, h, n, hipMemcpyHostToDevice, st) == hipSuccess;
    };
    if (!up(b->pos, z.data(), bytes) || !up(b->vel, z.data(), bytes) ||
        !up(b->force, z.data(), bytes) || !up(b->tF, z.data(), bytes) ||
        !up(b->obs, o.data(), sizeof(lj_obs) * nboxes) ||
        !up(b->stats, zs.data(), sizeof(double) * zs.size()) || hipStreamSynchronize(st) != hipSuccess)
      A(fail(LJ_ERR_DEVICE, "initial upload failed"));
  }
  if (rc != LJ_OK) {
    std::string msg = last_error();
    lj_batch_destroy(b);
    fail(rc, "%s", msg.c_str());
    return rc;
  }
  *out = b;
  return LJ_OK;
}

int lj_batch_destroy(lj_batch* b)
{
  if (!b) return LJ_OK;
  (void)hipSetDevice(b->device);
  if (b->stream) (void)hipStreamSynchronize(b->stream);
  bdrop_graph(b);
  dev_free(b->pos);
  dev_free(b->vel);
  dev_free(b->force);
  dev_free(b->tF);
  dev_free(b->q);
  dev_free(b->q2);
  dev_free(b->box_s);
  dev_free(b->tiles);
  dev_free(b->blk_s);
  dev_free(b->fpart);
  dev_free(b->apart);
  dev_free(b->blk);
  dev_free(b->obs);
  dev_free(b->stats);
  dev_free(b->box);
  dev_free(b->pblock);
  dev_free(b->items);
  dev_free(b->ew);
  dev_free(b->counter);
  fl_free(b->fl);
  dev_free(b->hist);
  dev_free(b->hist_base);
  if (b->e0) (void)hipEventDestroy(b->e0);
  if (b->e1) (void)hipEventDestroy(b->e1);
  if (b->stream) (void)hipStreamDestroy(b->stream);
  delete b;
  return LJ_OK;
}

int lj_batch_num_particles(const lj_batch* b) { return b ? b->Ntot : 0; }

int lj_batch_set_array(lj_batch* b, int box, int type, const float* host4N)
{
  LJ_TRY(bsetdev(b));
  if (box < -1 || box >= b->nboxes || !host4N) return fail(LJ_ERR_ARG, "lj_batch_set_array: bad box or pointer");
  float4* d = type == LJ_ARRAY_POS ? b->pos : type == LJ_ARRAY_VEL ? b->vel : type == LJ_ARRAY_FORCE ? b->force : nullptr;
  if (!d) return fail(LJ_ERR_ARG, "lj_batch_set_array: unknown array type %d", type);
  const size_t o = box < 0 ? 0 : b->off[box];
  const size_t n = box < 0 ? b->Ntot : b->N[box];
  LJ_HIP(hipMemcpyAsync(d + o, host4N, sizeof(float4) * n, hipMemcpyHostToDevice, b->stream));
  LJ_HIP(hipStreamSynchronize(b->stream));
  return LJ_OK;
}

int lj_batch_get_array(lj_batch* b, int box, int type, float* host4N)
{
  LJ_TRY(bsetdev(b));
  if (box < -1 || box >= b->nboxes || !host4N) return fail(LJ_ERR_ARG, "lj_batch_get_array: bad box or pointer");
  float4* d = type == LJ_ARRAY_POS ? b->pos : type == LJ_ARRAY_VEL ? b->vel : type == LJ_ARRAY_FORCE ? b->force : nullptr;
  if (!d) return fail(LJ_ERR_ARG, "lj_batch_get_array: unknown array type %d", type);
  const size_t o = box < 0 ? 0 : b->off[box];
  const size_t n = box < 0 ? b->Ntot : b->N[box];
  LJ_HIP(hipMemcpyAsync(host4N, d + o, sizeof(float4) * n, hipMemcpyDeviceToHost, b->stream));
  LJ_HIP(hipStreamSynchronize(b->stream));
  return LJ_OK;
}

int lj_batch_compute_forces(lj_batch* b)
{
  LJ_TRY(bready(b));
  hipStream_t st = b->stream;
  LJ_TRY(enqueue_batch_forces(b, st, true));
  const BatchArgs a = bargs(b, 0.);
  LJ_HIP(launch_batch_reduce_forces(st, a));
  LJ_HIP(launch_batch_kinetic(st, a));
  LJ_HIP(launch_batch_finalize(st, a, 0));
  LJ_HIP(hipStreamSynchronize(st));
  return LJ_OK;
}

int lj_batch_sample_initial_state(lj_batch* b, uint64_t seed)
{
  LJ_TRY(bsetdev(b));
  std::vector<float> p((size_t)4 * b->Ntot), v((size_t)4 * b->Ntot);
  for (int k = 0; k < b->nboxes; ++k) {
    const size_t o = (size_t)4 * b->off[k];
    lattice_positions(b->N[k], b->L[k], p.data() + o);
    gaussian_velocities(b->N[k], b->T0[k], seed + (uint64_t)k, v.data() + o);
  }
  LJ_TRY(lj_batch_set_array(b, -1, LJ_ARRAY_POS, p.data()));
  LJ_TRY(lj_batch_set_array(b, -1, LJ_ARRAY_VEL, v.data()));
  LJ_TRY(lj_batch_compute_forces(b));
  return lj_batch_reset_stats(b);
}

int lj_batch_set_subvolume(lj_batch* b, double fraction)
{
  LJ_TRY(bsetdev(b));
  if (!(fraction > 0.) || fraction > 1.) return fail(LJ_ERR_ARG, "lj_batch_set_subvolume: fraction must be in (0, 1]");
  b->sub_fraction = fraction;
  return build_tables(b);
}

int lj_batch_reset_stats(lj_batch* b)
{
  LJ_TRY(bsetdev(b));
  LJ_HIP(launch_batch_zero_stats(b->stream, bargs(b, 0.)));
  LJ_HIP(hipStreamSynchronize(b->stream));
  return LJ_OK;
}

int lj_batch_get_stats(lj_batch* b, double* out)
{
  LJ_TRY(bsetdev(b));
  if (!out) return fail(LJ_ERR_ARG, "lj_batch_get_stats: null output");
  LJ_HIP(hipMemcpyAsync(out, b->stats, sizeof(double) * kNStat * b->nboxes, hipMemcpyDeviceToHost, b->stream));
  LJ_HIP(hipStreamSynchronize(b->stream));
  return LJ_OK;
}

int lj_batch_get_observables(lj_batch* b, lj_obs* out)
{
  LJ_TRY(bsetdev(b));
  if (!out) return fail(LJ_ERR_ARG, "lj_batch_get_observables: null output");
  LJ_HIP(hipMemcpyAsync(out, b->obs, sizeof(lj_obs) * b->nboxes, hipMemcpyDeviceToHost, b->stream));
  LJ_HIP(hipStreamSynchronize(b->stream));
  return LJ_OK;
}

int lj_batch_set_tuning(lj_batch* b, const lj_batch_tuning* t)
{
  LJ_TRY(bsetdev(b));
  if (!t || (t->ipl != 1 && t->ipl != 2) || t->jchunk < 8 || t->jchunk > (1 << 20) ||
      t->blocks_per_cu < 0 || t->blocks_per_cu > 64 || (t->pair_once != 0 && t->pair_once != 1))
    return fail(LJ_ERR_ARG, "lj_batch_set_tuning: ipl in {1,2}, jchunk in [8, 2^20], blocks_per_cu in [0, 64], pair_once in {0,1}");
  const lj_batch_tuning old = b->tune;
  b->tune = *t;
  const int rc = build_tables(b);
  if (rc == LJ_OK) return LJ_OK;
  // no room for the new tables: the old ones again, if they find it
  const std::string msg = last_error();
  b->tune = old;
  (void)build_tables(b);
  return fail(rc, "%s", msg.c_str());
}

int lj_batch_get_tuning(lj_batch* b, lj_batch_tuning* t)
{
  if (!b || !t) return fail(LJ_ERR_ARG, "lj_batch_get_tuning: null argument");
  *t = b->tune;
  return LJ_OK;
}

int lj_batch_time_force(lj_batch* b, int reps, double* us)
{
  LJ_TRY(bready(b));
  if (reps <= 0 || !us) return fail(LJ_ERR_ARG, "lj_batch_time_force: bad arguments");
  hipStream_t st = b->stream;
  LJ_TRY(enqueue_batch_forces(b, st, false, true));  // warm
  LJ_HIP(hipEventRecord(b->e0, st));
  for (int k = 0; k < reps; ++k) LJ_TRY(enqueue_batch_forces(b, st, false, true));
  LJ_HIP(hipEventRecord(b->e1, st));
  LJ_HIP(hipEventSynchronize(b->e1));
  float ms = 0.f;
  LJ_HIP(hipEventElapsedTime(&ms, b->e0, b->e1));
  *us = 1000.0 * ms / reps;
  return LJ_OK;
}

int lj_batch_autotune(lj_batch* b, int reps, lj_batch_tuning* best_out, double* best_us)
{
  LJ_TRY(bsetdev(b));
  if (reps <= 0) reps = 3;
  const char* cache = std::getenv("LJ_AUTOTUNE_CACHE");
  const std::string key = tune_key(b);
  if (cache) {
    std::ifstream in(cache);
    std::string k;
    lj_batch_tuning t{};
    double us = 0.;
    while (in >> k >> t.ipl >> t.jchunk >> t.blocks_per_cu >> t.pair_once >> us)
      if (k == key) {
        LJ_TRY(lj_batch_set_tuning(b, &t));
        if (best_out) *best_out = t;
        if (best_us) *best_us = us;
        return LJ_OK;
      }
  }
  const int ipls[] = {1, 2};
  const int jcs[] = {256, 512, 1024, 2048};
  const int bpcs[] = {0, 4, 8};
  lj_batch_tuning best = b->tune;
  double best_t = 1e300;
  std::vector<lj_batch_tuning> cand;
  for (int ipl : ipls)
    for (int jc : jcs)
      for (int bpc : bpcs) cand.push_back(lj_batch_tuning{ipl, jc, bpc, 0});
  // the pair-once items, one workgroup each or drained by 4 or 8 resident
  // workgroups per CU (8: the kernel's occupancy limit)
  for (int bpc : bpcs) cand.push_back(lj_batch_tuning{1, 512, bpc, 1});
  // the fastest candidate; a persistent grid of pair-once items within 3% of
  // it is taken instead (one launch drains the whole ensemble; the pair-once
  // launch shapes measured within run-to-run noise of each other on MI355X)
  double best_p = 1e300;
  lj_batch_tuning best_pt{};
  for (const lj_batch_tuning& t : cand) {
    LJ_TRY(lj_batch_set_tuning(b, &t));
    double us = 0.;
    LJ_TRY(lj_batch_time_force(b, reps, &us));
    if (us < best_t) {
      best_t = us;
      best = t;
    }
    if (t.pair_once && t.blocks_per_cu > 0 && us < best_p) {
      best_p = us;
      best_pt = t;
    }
  }
  if (best_p <= 1.03 * best_t) {
    best = best_pt;
    best_t = best_p;
  }
  LJ_TRY(lj_batch_set_tuning(b, &best));
  // the one-launch step has no force pass of its own: whole steps decide (16 boxes
  // of 400, EVN: 9 us against 28 with the best tiling)
  double tiled = 0., one = 0.;  // no room for the copies: the best tiling stays
  if (small_steps(b->N) && time_steps(b, reps, &tiled) == LJ_OK) {
    LJ_TRY(lj_batch_set_tuning(b, &kDefaultTuning));
    if (time_steps(b, reps, &one) == LJ_OK && one <= tiled) {
      best = kDefaultTuning;
      best_t = one;
    } else {
      LJ_TRY(lj_batch_set_tuning(b, &best));
    }
  }
  if (cache) {
    std::ofstream o(cache, std::ios::app);
    o << key << " " << best.ipl << " " << best.jchunk << " " << best.blocks_per_cu << " "
      << best.pair_once << " " << best_t << "\n";
  }
  if (best_out) *best_out = best;
  if (best_us) *best_us = best_t;
  return LJ_OK;
}

int lj_batch_integrate(lj_batch* b, double dt, int nsteps)
{
  return lj_batch_integrate_hist(b, dt, nsteps, nullptr);
}

int lj_batch_integrate_hist(lj_batch* b, double dt, int nsteps, double* hist)
{
  LJ_TRY(bready(b));
  if (nsteps < 0 || !std::isfinite(dt)) return fail(LJ_ERR_ARG, "lj_batch_integrate: bad arguments");
  if (nsteps == 0) return LJ_OK;
  hipStream_t st = b->stream;
  if (hist && nsteps > b->hist_cap) {
    // the captured steps hold the history pointer: grow, then capture again
    LJ_HIP(hipStreamSynchronize(st));
    bdrop_graph(b);
    dev_free(b->hist);
    b->hist_cap = 0;
    const int cap = std::max(nsteps, 256);
    LJ_TRY(dev_alloc(&b->hist, (size_t)5 * cap * b->nboxes));
    if (!b->hist_base) LJ_TRY(dev_alloc(&b->hist_base, b->nboxes));
    b->hist_cap = cap;
  }
  if (b->hist_base) LJ_HIP(launch_batch_set_hist_base(st, bargs(b, dt), b->hist_base));
  if (!b->gexec || b->g_dt != dt) {
    bdrop_graph(b);
    LJ_HIP(hipStreamSynchronize(st));
    LJ_TRY(capture_batch_steps(b, dt, 1, &b->graph, &b->gexec));
    const int rc = capture_batch_steps(b, dt, kGraphSteps, &b->graph_run, &b->gexec_run);
    if (rc != LJ_OK) {
      bdrop_graph(b);
      return rc;
    }
    b->g_dt = dt;
  }
  int k = 0;
  for (; k + kGraphSteps <= nsteps; k += kGraphSteps) LJ_HIP(hipGraphLaunch(b->gexec_run, st));
  for (; k < nsteps; ++k) LJ_HIP(hipGraphLaunch(b->gexec, st));
  if (hist)
    LJ_HIP(hipMemcpyAsync(hist, b->hist, sizeof(double) * 5 * (size_t)nsteps * b->nboxes,
                          hipMemcpyDeviceToHost, st));
  LJ_HIP(hipStreamSynchronize(st));
  return LJ_OK;
}

int lj_batch_fl_configure(lj_batch* b, const lj_fl_ladder* ladders, int n)
{
  LJ_TRY(bsetdev(b));
  LJ_HIP(hipStreamSynchronize(b->stream));
  if (b->smp_fl) bdrop_graph(b);
  LJ_TRY(fl_configure(b->fl, b->stream, b->nboxes, b->L.data(), ladders, n));
  if (!b->fl.active()) b->smp_fl = 0;
  return LJ_OK;
}

int lj_batch_fl_num_entries(lj_batch* b, int* entries)
{
  if (!b || !entries) return fail(LJ_ERR_ARG, "lj_batch_fl_num_entries: null argument");
  *entries = b->fl.E;
  return LJ_OK;
}

int lj_batch_fl_sample(lj_batch* b)
{
  LJ_TRY(bsetdev(b));
  if (!b->fl.active()) return fail(LJ_ERR_STATE, "lj_batch_fl_sample: no counters configured");
  LJ_HIP(launch_fl_sample(b->stream, b->fl, b->pos, b->vel, 0, b->box, b->pblock, b->nblocks));
  LJ_HIP(hipStreamSynchronize(b->stream));
  return LJ_OK;
}

int lj_batch_fl_counts(lj_batch* b, int64_t* counts)
{
  LJ_TRY(bsetdev(b));
  if (!counts) return fail(LJ_ERR_ARG, "lj_batch_fl_counts: null output");
  if (!b->fl.active()) return fail(LJ_ERR_STATE, "lj_batch_fl_counts: no counters configured");
  LJ_HIP(hipMemcpyAsync(counts, b->fl.last, sizeof(int64_t) * b->nboxes * b->fl.E,
                        hipMemcpyDeviceToHost, b->stream));
  LJ_HIP(hipStreamSynchronize(b->stream));
  return LJ_OK;
}

int lj_batch_fl_stats(lj_batch* b, double* stats)
{
  LJ_TRY(bsetdev(b));
  if (!stats) return fail(LJ_ERR_ARG, "lj_batch_fl_stats: null output");
  if (!b->fl.active()) return fail(LJ_ERR_STATE, "lj_batch_fl_stats: no counters configured");
  LJ_HIP(hipMemcpyAsync(stats, b->fl.stats, sizeof(double) * kFlStat * b->nboxes * b->fl.E,
                        hipMemcpyDeviceToHost, b->stream));
  LJ_HIP(hipStreamSynchronize(b->stream));
  return LJ_OK;
}

int lj_batch_fl_reset(lj_batch* b)
{
  LJ_TRY(bsetdev(b));
  if (!b->fl.active()) return fail(LJ_ERR_STATE, "lj_batch_fl_reset: no counters configured");
  LJ_HIP(launch_fl_reset(b->stream, b->fl));
  LJ_HIP(hipStreamSynchronize(b->stream));
  return LJ_OK;
}

int lj_batch_set_step_sampling(lj_batch* b, int fluctuations)
{
  LJ_TRY(bsetdev(b));
  if (fluctuations && !b->fl.active())
    return fail(LJ_ERR_STATE, "lj_batch_set_step_sampling: configure the counters first");
  LJ_HIP(hipStreamSynchronize(b->stream));
  bdrop_graph(b);
  b->smp_fl = fluctuations ? 1 : 0;
  return LJ_OK;
}

}  // extern "C"
