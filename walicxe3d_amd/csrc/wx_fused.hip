// wx_fused.hip - the fused FP32 form of the Godunov update.
//
// One stage = one kernel launch over all blocks of all levels.  A workgroup
// of 256 threads owns a block, or a z slab of one on meshes of few blocks;
// thread (ti, tj) owns the column (i, j) and marches in k.  Per k-plane the
// primitives of the plane and its x/y face halo sit in LDS (x and y fluxes),
// the column's primitives of the planes around k sit in registers (z fluxes,
// Powell term).  Face halos are read straight from the neighbour blocks'
// interiors with the AMR exchange rules of wx_device.h - no ghost cells are
// stored in HBM.
//
// Precision: bulk flux/reconstruction arithmetic in FP32; conserved state U
// and its accumulation U + dt*dF in FP64; stage-1 pressure recovery from the
// FP64 state in FP64; the end of the step (viscosity, primitives, cooling,
// dt candidate) in FP64 on U^{n+1}; dt reduced as an exact min.
//
// Stage 1 (first order, dt/2): U^n (FP64) -> UP (FP32).
// Stage 2 (second order, dt): UP, U^n -> U^{n+1}.  Hydro and FP64 leave that
// state to k_end, which applies viscosity (its face neighbours are the
// half-step ghosts, as in the reference) and cooling and forms the next dt;
// FP32 MHD does so with viscosity or cooling only, else its stage 2 ends the
// step itself.
// k_flow (hydro, FP64 MHD; wx_hydro_kern.h), k_mhd (FP32 MHD;
// wx_mhd_kern.h), k_stage (MHD with plain FP32 fluxes, set_tuning kind 3).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>

#include "wx_fused.h"
#include "wx_hilbert.h"
#include "wx_fused_kern.h"
#include "wx_hydro_kern.h"

namespace wx {

// Workgroups below which the hydro kernels take thinner slabs (a slab of L
// planes solves L + 1 z faces and loads L + 3 planes per column).  us per step
// for HYDRO_WANT = 512, 1024, 2048, 4096: 64 blocks 51.2, 49.9, 50.5, 50.4; 904
// blocks on 4 levels 470, 424, 411, 423; 1728 blocks 618, 619, 615, 637.  The
// end of the step runs 4 planes per workgroup, fewer below END_WANT: 64 blocks
// 51.0, 50.5, 52.6 for 256, 512, 1024.  FP32 MHD (two workgroups per CU) takes
// slabs below MHD_WANT unless set_tuning chose: 64 blocks 83.4, 65.7, 76.3 for
// 256, 512, 1024; 32 blocks 56.2, 47.3, 46.9; whole blocks took 265 and 270.
// FP64 (hydro and MHD, two to three workgroups per CU) shares HYDRO_WANT, whole
// step for 512, 1024, 2048, 4096: HLLC without viscosity, 64 blocks 64.0, 70.6, 70.8,
// 71.1 us, 240 153, 163, 188, 185, 904 497, 478, 479, 508, 1728 871, 871, 863, 894;
// HLLD, 64 116, 133, 136, 131, 240 338, 350, 387, 384, 904 1199, 1174, 1151, 1213, 1728
// 2078, 2077, 2059, 2103: 2048 is the better line from 904 blocks on, and 10 to 19
// per cent behind 512 (planes enough to pay for a slab's extra ones) at 64 and 240.
constexpr int HYDRO_WANT = 2048, END_WANT = 512, MHD_WANT = 512;

static thread_local std::string f_err;
const char *fused_error() { return f_err.c_str(); }

// initial dt candidate from U (after an upload)
template <int NV>
__global__ void __launch_bounds__(256) k_dt_init(FusedArgs a) {
  const DevCfg &c = a.c;
  int b = blockIdx.x;
  int l = c.info[b].level - 1;
  double m = 1.0e30;
  for (int q = threadIdx.x; q < NINT; q += 256) {
    double u[MAXV], pd[MAXV];
    for (int v = 0; v < NV; v++) u[v] = a.U[((size_t)b * NV + v) * NINT + q];
    flow2prim(c.pd, u, pd);
    m = fmin(m, dt_cell<NV>(c, pd, c.dx[0][l], c.dx[1][l], c.dx[2][l]));
  }
  for (int off = 32; off > 0; off >>= 1) m = fmin(m, __shfl_xor(m, off));
  if ((threadIdx.x & 63) == 0) atomicMin(&a.step->dtmin_bits, (unsigned long long)__double_as_longlong(m));
}

// The scalars of a step: closes the step before it, then dt from the running
// minimum (the kernels' slots and the step record's own word) with the
// start-up ramp and the output clamp (source/hydro_solver.f90:183-207); both
// minima are cleared.  One wavefront.
__global__ void __launch_bounds__(64) k_begin(StepState *s, unsigned long long *slots, double cfl, int cooling) {
  double m = fold_slots(slots);
  if (threadIdx.x == 0) {
    m = fmin(m, __longlong_as_double((long long)s->dtmin_bits));
    step_close(s);
    step_open(s, m, cfl, cooling);
    s->dtmin_bits = ~0ull;
  }
}

// PRIM of the state in the same layout ([blk][nv][16^3]), for downloads
template <int NV>
__global__ void k_prims_int(const DevCfg c, int nblk, const double *src, double *dstP) {
  size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (size_t)nblk * NINT) return;
  int q = (int)(t % NINT);
  size_t b = t / NINT;
  double u[MAXV], p[MAXV];
  for (int v = 0; v < NV; v++) u[v] = src[(b * NV + v) * NINT + q];
  flow2prim(c.pd, u, p);
  for (int v = 0; v < NV; v++) dstP[(b * NV + v) * NINT + q] = p[v];
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
static int hip_fail(hipError_t e, const char *what) {
  if (e == hipSuccess) return 0;
  f_err = std::string(what) + ": " + hipGetErrorString(e);
  return 1;
}
#define FCHK(x) do { if (hip_fail((x), #x)) return 1; } while (0)

// Morton key of a block's position at the finest level: neighbours in space
// end up close in the processing order (shared L2 lines for halo reads)
static unsigned long long morton(const BlockInfo &B, int maxlev) {
  unsigned long long key = 0;
  int shift = maxlev - B.level;
  unsigned x = (unsigned)(B.coords[0] - 1) << shift, y = (unsigned)(B.coords[1] - 1) << shift,
           z = (unsigned)(B.coords[2] - 1) << shift;
  for (int bit = 0; bit < 20; bit++) {
    key |= (unsigned long long)((x >> bit) & 1) << (3 * bit);
    key |= (unsigned long long)((y >> bit) & 1) << (3 * bit + 1);
    key |= (unsigned long long)((z >> bit) & 1) << (3 * bit + 2);
  }
  return key;
}

// Block processing order: Morton (or Hilbert) order of the blocks'
// positions; with the XCD map, workgroup w runs on XCD w % 8, so each XCD
// gets a contiguous range of the curve (neighbour halos then hit that XCD's
// L2).
static int build_order(FusedState &f) {
  const int nb = f.nblk;
  std::vector<std::pair<unsigned long long, int>> keys(nb);
  if (f.curve == 1) {
    const int order = hilbert_order(f.nroot, f.maxlev);
    for (int b = 0; b < nb; b++)
      keys[b] = {block_hilbert_key(f.host_info[b].coords, f.host_info[b].level, f.maxlev, order), b};
  } else {
    for (int b = 0; b < nb; b++) keys[b] = {morton(f.host_info[b], f.maxlev), b};
  }
  std::sort(keys.begin(), keys.end());
  const int nx = 8;
  std::vector<int> ord(nb, -1);
  if (f.xcd_map && nb >= 64) {
    int full = (nb / nx) * nx;
    int perx = full / nx;
    for (int r = 0; r < full; r++) {
      int xcd = r / perx, within = r % perx;
      ord[within * nx + xcd] = keys[r].second;
    }
    for (int r = full; r < nb; r++) ord[r] = keys[r].second;
  } else {
    for (int r = 0; r < nb; r++) ord[r] = keys[r].second;
  }
  f.host_order = ord;
  FCHK(hipMemcpy(f.order, ord.data(), nb * sizeof(int), hipMemcpyHostToDevice));
  return 0;
}

int fused_alloc(FusedState &f, const DevCfg &c, const std::vector<BlockInfo> &info, bool adopt, hipStream_t st) {
  fused_free(f);
  f.nblk = c.nblk;
  f.nv = c.nv;
  f.two_u = !f.fp64 && c.nv == 8;
  size_t n = (size_t)c.nblk * c.nv * NINT;
  if (!adopt) FCHK(hipMalloc(&f.U, n * sizeof(double)));
  if (f.two_u) FCHK(hipMalloc(&f.U2, n * sizeof(double)));
  FCHK(hipMalloc(&f.UP, n * (f.fp64 ? sizeof(double) : sizeof(float))));
  FCHK(hipMalloc(&f.order, c.nblk * sizeof(int)));
  FCHK(hipMalloc(&f.rec, sizeof(StepRecord)));
  f.host_info = info;
  f.maxlev = c.maxlev;
  if (build_order(f)) return 1;
  for (int e = 0; e < 4; e++) FCHK(hipEventCreate(&f.ev[e]));
  (void)st;
  return 0;
}

static void drop_graphs(FusedState &f) {
  if (f.exec) hipGraphExecDestroy(f.exec);
  if (f.graph) hipGraphDestroy(f.graph);
  if (f.exec2) hipGraphExecDestroy(f.exec2);
  if (f.graph2) hipGraphDestroy(f.graph2);
  f.exec = f.exec2 = nullptr;
  f.graph = f.graph2 = nullptr;
  f.graph_u = f.graph2_u = nullptr;
}

void fused_drop_x(FusedState &f) {
  if (!f.X) return;
  drop_graphs(f);
  hipFree(f.X);
  f.X = nullptr;
}

// X comes with the first run: an upload's staging buffer and the two states of
// a mesh change, each as large, are gone by then, so the largest mesh that
// fits is the one that it was without X (hydro FP32: 20 bytes a variable and
// zone at most, in an upload, a mesh change and a run alike).
static int need_x(FusedState &f, const DevCfg &c) {
  if (f.X || (f.two_u && !ends_apart(c))) return 0;
  FCHK(hipMalloc(&f.X, (size_t)f.nblk * f.nv * NINT * sizeof(double)));
  return 0;
}

void fused_free(FusedState &f) {
  drop_graphs(f);
  hipFree(f.U);
  hipFree(f.U2);
  hipFree(f.UP);
  hipFree(f.order);
  hipFree(f.rec);
  hipFree(f.X);
  for (int e = 0; e < 4; e++)
    if (f.ev[e]) hipEventDestroy(f.ev[e]);
  for (int e = 0; e < 4; e++) f.ev[e] = nullptr;
  f.U = nullptr;
  f.U2 = nullptr;
  f.UP = nullptr;
  f.order = nullptr;
  f.rec = nullptr;
  f.X = nullptr;
}

static FusedArgs make_args(FusedState &f, const DevCfg &c) {
  FusedArgs a;
  a.c = c;
  a.U = f.U;
  a.Uout = f.U2 ? f.U2 : f.U;
  a.UPin = f.UP;
  a.UPout = f.UP;
  a.X = f.X;
  a.slots = f.rec->slots;
  a.order = f.order;
  a.step = &f.rec->s;
  a.nblk = f.nblk;
  a.nslab = 1;
  return a;
}

static void launch_dt_init(FusedState &f, const DevCfg &c, hipStream_t st) {
  FusedArgs a = make_args(f, c);
  if (c.nv == 8) hipLaunchKernelGGL(k_dt_init<8>, dim3(f.nblk), dim3(256), 0, st, a);
  else hipLaunchKernelGGL(k_dt_init<5>, dim3(f.nblk), dim3(256), 0, st, a);
}

int fused_upload(FusedState &f, const DevCfg &c, double *U, bool adopt, hipStream_t st) {
  if (adopt) {   // ownership first, so that no return path leaks U
    hipFree(f.U);
    f.U = U;
  } else {
    const size_t bytes = (size_t)f.nblk * f.nv * NINT * sizeof(double);
    if (!f.U) FCHK(hipMalloc(&f.U, bytes));   // an adoption that failed
    FCHK(hipMemcpyAsync(f.U, U, bytes, hipMemcpyDeviceToDevice, st));
  }
  StepRecord r{};
  r.s.dtmin_bits = ~0ull;
  std::memset(r.slots, 0xFF, sizeof(r.slots));
  FCHK(hipMemcpyAsync(f.rec, &r, sizeof(r), hipMemcpyHostToDevice, st));
  launch_dt_init(f, c, st);
  FCHK(hipGetLastError());
  FCHK(hipStreamSynchronize(st));
  return 0;
}

int fused_prims(FusedState &f, const DevCfg &c, double *P, hipStream_t st) {
  size_t n = (size_t)f.nblk * NINT;
  if (f.nv == 8)
    hipLaunchKernelGGL(k_prims_int<8>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, c, f.nblk, f.U, P);
  else
    hipLaunchKernelGGL(k_prims_int<5>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, c, f.nblk, f.U, P);
  FCHK(hipGetLastError());
  FCHK(hipStreamSynchronize(st));
  return 0;
}

int fused_timestep(FusedState &f, const DevCfg &c, hipStream_t st, double *dt_raw) {
  // one transfer: two took 37 us, one 25
  StepRecord r;
  FCHK(hipMemcpyAsync(&r, f.rec, sizeof(r), hipMemcpyDeviceToHost, st));
  FCHK(hipStreamSynchronize(st));
  // an untouched word reads as a NaN, which fmin drops
  double m, q;
  std::memcpy(&m, &r.s.dtmin_bits, sizeof(m));
  for (int n = 0; n < DT_SLOTS; n++) {
    std::memcpy(&q, &r.slots[n * DT_STRIDE], sizeof(q));
    m = std::fmin(m, q);
  }
  *dt_raw = c.cooling ? std::fmin(m, 1.0e30) * c.cfl : m * c.cfl;
  return 0;
}

// meshes without wind sources take kernels without the wind code; minmod, the
// default limiter, is fixed at compile time, the others are read at run time
template <int NV, typename RF, typename ST, int SOLVER, bool WINDS>
static void launch_flow_t(const FusedArgs &a, int grid, int stage, hipStream_t st) {
  constexpr int MM = 1;   // LIMITER_MINMOD (source/constants.f90)
  if (stage == 1)
    hipLaunchKernelGGL((k_flow<NV, false, RF, ST, SOLVER, MM, WINDS>), dim3(grid), dim3(256), 0, st, a);
  else if (a.c.pf.limiter == MM)
    hipLaunchKernelGGL((k_flow<NV, true, RF, ST, SOLVER, MM, WINDS>), dim3(grid), dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL((k_flow<NV, true, RF, ST, SOLVER, LIM_RUNTIME, WINDS>), dim3(grid), dim3(256), 0, st, a);
}

template <int NV, typename RF, typename ST, int SOLVER>
static void launch_flow(const FusedArgs &a, int grid, int stage, hipStream_t st) {
  if constexpr (NV == 5) {   // FP64 MHD has no wind sources (wx_init)
    if (a.c.nwind > 0) return launch_flow_t<NV, RF, ST, SOLVER, true>(a, grid, stage, st);
  }
  launch_flow_t<NV, RF, ST, SOLVER, false>(a, grid, stage, st);
}

template <int NV, typename RF, typename ST>
static void launch_end(const FusedArgs &a, hipStream_t st) {
  const int grid = a.nblk * a.nslab;
  if (a.c.visc_eta == 0.0) {
    hipLaunchKernelGGL((k_end<NV, RF, ST, false, false, false>), dim3(grid), dim3(256), 0, st, a);
    return;
  }
  if constexpr (NV == 5) {
    if (a.c.nwind > 0) {
      hipLaunchKernelGGL((k_end<NV, RF, ST, true, false, true>), dim3(grid), dim3(256), 0, st, a);
      return;
    }
  }
  hipLaunchKernelGGL((k_end<NV, RF, ST, true, false, false>), dim3(grid), dim3(256), 0, st, a);
}

// slabs per block that give `want` workgroups, at least `least`
static int slabs_for(int nblk, int want, int least) {
  int n = least;
  while (n < NC && nblk * n < want) n <<= 1;
  return n;
}

static void launch_stage(FusedState &f, const DevCfg &c, hipStream_t st, int stage) {
  FusedArgs a = make_args(f, c);
  const bool hllc = c.pd.solver == SOLVER_HLLC, hlld = c.pd.solver == SOLVER_HLLD;
  const bool mhd32 = c.nv == 8 && !f.fp64;
  if (!mhd32) a.nslab = slabs_for(f.nblk, HYDRO_WANT, 1);
  else if (!f.mhd_plain32) a.nslab = f.nslab > 0 ? f.nslab : slabs_for(f.nblk, MHD_WANT, 1);
  const int items = f.nblk * a.nslab;
  const int grid = f.grid > 0 ? std::min(f.grid, items) : items;
  if (mhd32) {
    launch_stage_mhd32(a, grid, c.pd.solver, c.visc_eta != 0.0, stage, f.mhd_plain32, st);
  } else if (c.nv == 8) {
    if (hlld) launch_flow<8, double, double, SOLVER_HLLD>(a, grid, stage, st);
    else launch_flow<8, double, double, SOLVER_HLLE>(a, grid, stage, st);
  } else if (f.fp64) {
    if (hllc) launch_flow<5, double, double, SOLVER_HLLC>(a, grid, stage, st);
    else launch_flow<5, double, double, SOLVER_HLL>(a, grid, stage, st);
  } else {
    if (hllc) launch_flow<5, float, float, SOLVER_HLLC>(a, grid, stage, st);
    else launch_flow<5, float, float, SOLVER_HLL>(a, grid, stage, st);
  }
}

// the end of the step, where the second stage's kernel leaves it
static void launch_rest(FusedState &f, const DevCfg &c, hipStream_t st) {
  const bool mhd32 = c.nv == 8 && !f.fp64;
  if (mhd32 && (f.mhd_plain32 || !ends_apart(c))) return;
  FusedArgs a = make_args(f, c);
  a.nslab = slabs_for(f.nblk, END_WANT, NC / END_PLANES);
  if (mhd32) launch_end_mhd32(a, st);
  else if (c.nv == 8) launch_end<8, double, double>(a, st);
  else if (f.fp64) launch_end<5, double, double>(a, st);
  else launch_end<5, float, float>(a, st);
}

static void enqueue_step(FusedState &f, const DevCfg &c, hipStream_t st) {
  hipLaunchKernelGGL(k_begin, dim3(1), dim3(64), 0, st, &f.rec->s, f.rec->slots, c.cfl, c.cooling);
  launch_stage(f, c, st, 1);
  launch_stage(f, c, st, 2);
  launch_rest(f, c, st);
}

// after a step of the two-buffer form the new state is in the other buffer
static void swap_u(FusedState &f) {
  if (f.U2) std::swap(f.U, f.U2);
}

static int capture_step(FusedState &f, const DevCfg &c, hipStream_t st, hipGraph_t *g, hipGraphExec_t *e) {
  FCHK(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
  enqueue_step(f, c, st);
  hipError_t err = hipStreamEndCapture(st, g);
  FCHK(err);
  FCHK(hipGraphInstantiate(e, *g, nullptr, nullptr, 0));
  return 0;
}

// The step graphs: ex[0] steps from the current U, ex[1] from the other
// buffer of the two-buffer form (the same graph otherwise).  Captured again
// whenever a buffer moved since the capture.
static int step_graphs(FusedState &f, const DevCfg &c, hipStream_t st, hipGraphExec_t ex[2]) {
  const bool ok = f.exec && f.graph_u == f.U && (!f.U2 || (f.exec2 && f.graph2_u == f.U2));
  if (!ok) {
    drop_graphs(f);
    if (capture_step(f, c, st, &f.graph, &f.exec)) return 1;
    f.graph_u = f.U;
    if (f.U2) {
      swap_u(f);
      const int rc = capture_step(f, c, st, &f.graph2, &f.exec2);
      swap_u(f);
      if (rc) return 1;
      f.graph2_u = f.U2;
    }
  }
  ex[0] = f.exec;
  ex[1] = f.U2 ? f.exec2 : f.exec;
  return 0;
}

int fused_run(FusedState &f, const DevCfg &c, hipStream_t st, int nsteps, int *it, double *dt, double *time,
              int *nextout, double dtout, double t_sc) {
  if (nsteps == 0) return 0;
  if (need_x(f, c)) return 1;
  // host scalars -> device (keeps the running dt minimum)
  StepState s;
  FCHK(hipMemcpyAsync(&s, &f.rec->s, sizeof(s), hipMemcpyDeviceToHost, st));
  FCHK(hipStreamSynchronize(st));
  s.it = *it;
  s.time = *time;
  s.nextout = *nextout;
  s.dtout = dtout;
  s.t_sc = t_sc;
  s.open = 0;
  FCHK(hipMemcpyAsync(&f.rec->s, &s, sizeof(s), hipMemcpyHostToDevice, st));
  hipGraphExec_t ex[2];
  if (step_graphs(f, c, st, ex)) return 1;
  FCHK(hipEventRecord(f.ev[0], st));
  for (int n = 0; n < nsteps; n++) {
    FCHK(hipGraphLaunch(ex[n & 1], st));
    swap_u(f);
  }
  FCHK(hipEventRecord(f.ev[1], st));
  FCHK(hipMemcpyAsync(&s, &f.rec->s, sizeof(s), hipMemcpyDeviceToHost, st));
  FCHK(hipStreamSynchronize(st));
  float ms = 0;
  hipEventElapsedTime(&ms, f.ev[0], f.ev[1]);
  f.t_tot = nsteps > 0 ? ms / nsteps : 0.0;
  step_close(&s);
  *it = s.it;
  *dt = s.dt;
  *time = s.time;
  *nextout = s.nextout;
  return 0;
}

// Times the two stage kernels separately (HIP events on the library stream)
// by replaying one step outside the graph; used by the benchmark.
int fused_time_stages(FusedState &f, const DevCfg &c, hipStream_t st, int reps) {
  float a1 = 0, a2 = 0;
  if (need_x(f, c)) return 1;
  for (int r = 0; r < reps; r++) {
    hipLaunchKernelGGL(k_begin, dim3(1), dim3(64), 0, st, &f.rec->s, f.rec->slots, c.cfl, c.cooling);
    FCHK(hipEventRecord(f.ev[0], st));
    launch_stage(f, c, st, 1);
    FCHK(hipEventRecord(f.ev[1], st));
    launch_stage(f, c, st, 2);
    launch_rest(f, c, st);
    FCHK(hipEventRecord(f.ev[2], st));
    swap_u(f);
    FCHK(hipEventSynchronize(f.ev[2]));
    float m1, m2;
    hipEventElapsedTime(&m1, f.ev[0], f.ev[1]);
    hipEventElapsedTime(&m2, f.ev[1], f.ev[2]);
    a1 += m1;
    a2 += m2;
  }
  f.t_s1 = a1 / reps;
  f.t_s2 = a2 / reps;
  f.timing_runs = reps;
  return 0;
}

// kind 0: stage-kernel grid (0 = one workgroup per block, else a persistent
//         grid of that many workgroups striding over the block list)
// kind 1: XCD-aware block order (1) or one range for all XCDs (0)
// kind 2: block order along the Morton (0) or the Hilbert (1) curve
// kind 3: FP32 MHD fluxes in delta form (0) or plain FP32 (1)
// kind 4: z slabs per block (1, 2, 4, 8, 16), one workgroup each, in the
//         delta-form MHD kernels; 0, the default, by mesh size (no effect elsewhere)
int fused_set_tuning(FusedState &f, int kind, int value) {
  if (kind < 0 || kind > 4) return 1;
  if ((kind == 2 || kind == 3) && (value < 0 || value > 1)) return 1;
  if (kind == 4 && (value < 0 || value > NC || (value & (value - 1)))) return 1;
  drop_graphs(f);
  if (kind == 3) {
    f.mhd_plain32 = value;
    return 0;
  }
  if (kind == 4) {
    f.nslab = value;
    return 0;
  }
  if (kind == 0) {
    if (value < 0) return 1;
    f.grid = value;
    return 0;
  }
  if (kind == 1)
    f.xcd_map = value != 0;
  else
    f.curve = value;
  return f.nblk > 0 ? build_order(f) : 0;
}

void fused_last_timing(const FusedState &f, double *s1, double *s2, double *tot) {
  if (s1) *s1 = f.t_s1;
  if (s2) *s2 = f.t_s2;
  if (tot) *tot = f.t_tot;
}

}  // namespace wx
