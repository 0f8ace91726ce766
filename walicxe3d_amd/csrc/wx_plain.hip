// wx_plain.hip - the plain FP64 form: one kernel per reference routine,
// arrays with two layers of face ghosts per block ([blk][nv][NSTORE], wx_common.h),
// arithmetic in the reference's order (built with -ffp-contract=off).
#include <hip/hip_runtime.h>

#include "wx_device.h"
#include "wx_kernels.h"

namespace wx {

// Workgroups below which the flux and update kernel splits blocks into slabs
// (a slab of L planes solves L + 1 z faces per column).  512 MHD blocks, whole
// step: 1053, 1008, 963, 978 us for 512, 1024, 2048, 4096; 512 hydro blocks:
// 610, 538, 533, 534 us; 64 hydro blocks: 85, 81, 82, 82 us.
constexpr int WX_UPDATE_WANT = 2048;
// The same for the timestep pass: one column of 16 planes per lane is a serial
// chain on a mesh of few blocks (getTimestep of 1 MHD block 39 us, in slabs 29).
// 256, 512, 1024, 2048: 64 MHD blocks 31.9, 31.0, 30.7, 30.6 us, 240: 42.8, 42.4,
// 41.9, 42.1, 1000: 75.4, 75.9, 72.6, 72.5.
constexpr int WX_TIMESTEP_WANT = 512;
// And for the end of the step.  Whole step for 512, 1024, 2048, 4096: 64 viscous
// hydro blocks 78.0, 82.6, 81.1, 81.5 us, 240: 215, 219, 225, 223, 904: 798, 797,
// 797, 805; viscous HLLD, 64: 154.6, 157.3, 157.1, 156.6, 240: 485, 479, 474, 477,
// 904: 1765, 1698, 1665, 1675, 1728: 3177, 3181, 3129, 3101.
constexpr int WX_FINISH_WANT = 2048;

// ---------------------------------------------------------------------------
// The device physics routines applied to arrays of records (one thread per
// record), for parity tests of single routines.  op (EVAL_*):
//   flow2prim   in nv -> out nv + 1 (primitives, istat)
//   prim2flow   in nv -> out nv
//   prim2fluxes in nv -> out nv, arg = direction 1..3
//   limiter     in 4 nv (pll, pl, pr, prr) -> out 2 nv (pl, pr), arg = limiter
//   riemann     in 2 nv (pl, pr) -> out nv, arg = solver (HLLD in the
//               reference's branch form)
//   riemann_sel in 2 nv -> out nv: HLLD in its select form (fused FP64 form)
//   speeds      in nv -> out 5 (sound, cfast x/y/z, cfastX)
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_eval(Phys<double> P, int op, int arg, int n, const double *in,
                                              double *out) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int nv = P.nv;
  double a[4 * MAXV], f[2 * MAXV];
  const int nin = op == EVAL_LIMITER ? 4 * nv : (op == EVAL_RIEMANN || op == EVAL_RIEMANN_SEL ? 2 * nv : nv);
  for (int q = 0; q < nin; q++) a[q] = in[(size_t)t * nin + q];
  int nout = nv;
  switch (op) {
    case EVAL_FLOW2PRIM:
      f[nv] = (double)flow2prim(P, a, f);
      nout = nv + 1;
      break;
    case EVAL_PRIM2FLOW:
      prim2flow(P, a, f);
      break;
    case EVAL_PRIM2FLUXES:
      swapdim(nv, arg - 1, a);
      xflux(P, a, f);
      swapdim(nv, arg - 1, f);
      break;
    case EVAL_LIMITER:
      for (int q = 0; q < nv; q++) {
        double pl = a[nv + q], pr = a[2 * nv + q];
        limit1(a[q], pl, pr, a[3 * nv + q], arg);
        f[q] = pl;
        f[nv + q] = pr;
      }
      nout = 2 * nv;
      break;
    case EVAL_RIEMANN:
      // P keeps the build's solver: primfhllc forms its contact speed only in
      // HLLC builds (source/hllc.f90:348-353)
      if (arg == SOLVER_HLLC) primfhllc(P, a, a + nv, f);
      else if (arg == SOLVER_HLLE) primfhlle(P, a, a + nv, f);
      else if (arg == SOLVER_HLLD) primfhlld(P, a, a + nv, f);
      else primfhll(P, a, a + nv, f);
      break;
    case EVAL_RIEMANN_SEL:
      primfhlld_sel<double>(P, a, a + nv, f);
      break;
    default:   // EVAL_SPEEDS
      f[0] = sound(P, a);
      f[1] = f[2] = f[3] = f[4] = 0.0;
      if (nv == 8) {
        f[1] = cfast1(P, a[4], a[0], a[5], a[6], a[7], a[5]);
        f[2] = cfast1(P, a[4], a[0], a[5], a[6], a[7], a[6]);
        f[3] = cfast1(P, a[4], a[0], a[5], a[6], a[7], a[7]);
        f[4] = cfastX(P, a);
      }
      nout = 5;
      break;
  }
  for (int q = 0; q < nout; q++) out[(size_t)t * nout + q] = f[q];
}

void plain_eval(const Phys<double> &P, int op, int arg, int n, const double *in, double *out, hipStream_t st) {
  hipLaunchKernelGGL(k_eval, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, P, op, arg, n, in, out);
}

// ---------------------------------------------------------------------------
// boundary (source/boundary.f90:46-64): face ghosts of depth `depth`.
// grid (6*depth, nblk), block 256 = transverse 16x16.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_boundary(DevCfg c, double *A, int depth) {
  int b = blockIdx.y;
  int f = blockIdx.x / depth;
  int g = blockIdx.x % depth + 1;
  int a1 = threadIdx.x % NC + 1, a2 = threadIdx.x / NC + 1;
  GhostSrc s;
  if (!ghost_source(c.info, c.bc, b, f, g, a1, a2, s)) return;
  int n, t1, t2;
  face_axes(f, n, t1, t2);
  int d[3];
  d[n] = (f & 1) ? NC + g : 1 - g;
  d[t1] = a1;
  d[t2] = a2;
  int q = cid(d[0], d[1], d[2]);
  int nv = c.nv;
  double val[MAXV];
  for (int v = 0; v < nv; v++) val[v] = ghost_value<double>(A, nv, s, v);
  for (int v = 0; v < nv; v++) A[((size_t)b * nv + v) * NSTORE + q] = val[v];
}

// Wind sources over interior and face-ghost cells (userBoundary).
// grid (28, nblk): 16 blocks of 256 interior cells, 12 of face ghosts.
// P, when given, takes the primitives of the covered interior cells.
__global__ void __launch_bounds__(256) k_winds(DevCfg c, double *A, PlaneWind pw, double *P) {
  int b = blockIdx.y;
  int i, j, k;
  if (blockIdx.x < 16) {
    int t = blockIdx.x * 256 + threadIdx.x;
    i = t % NC + 1; j = (t / NC) % NC + 1; k = t / (NC * NC) + 1;
  } else {
    int f = (blockIdx.x - 16) / 2, g = (blockIdx.x - 16) % 2 + 1;
    int n, t1, t2, d[3];
    face_axes(f, n, t1, t2);
    d[n] = (f & 1) ? NC + g : 1 - g;
    d[t1] = threadIdx.x % NC + 1;
    d[t2] = threadIdx.x / NC + 1;
    i = d[0]; j = d[1]; k = d[2];
  }
  double u[MAXV];
  bool hit = wind_state(c, b, i, j, k, u);
  if (plane_wind_state(c, pw, b, k, u)) hit = true;   // after the spherical sources
  if (hit) {
    int q = cid(i, j, k);
    for (int v = 0; v < c.nv; v++) A[((size_t)b * c.nv + v) * NSTORE + q] = u[v];
    if (P && blockIdx.x < 16) {
      double p[MAXV];
      flow2prim(c.pd, u, p);   // no passive scalars: refused with wind sources, unset by the plane wind
      for (int v = 0; v < c.pd.nv; v++) P[((size_t)b * c.nv + v) * NSTORE + q] = p[v];
      for (int v = c.pd.nv; v < c.nv; v++) P[((size_t)b * c.nv + v) * NSTORE + q] = u[v];
    }
  }
}

// ---------------------------------------------------------------------------
// calcPrimsAll (source/hydro_core.f90:67-223): interior (cells ALL/PHYS)
// and face ghosts with non-zero density (ALL/GHOST).  Edge and corner
// ghosts are never read by the update and are skipped.
// grid (28, nblk)
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_prims(DevCfg c, const double *A, double *P, int cells,
                                               unsigned long long *bad) {
  int b = blockIdx.y;
  int i, j, k;
  bool ghost = blockIdx.x >= 16;
  if (!ghost) {
    if (cells == 2) return;
    int t = blockIdx.x * 256 + threadIdx.x;
    i = t % NC + 1; j = (t / NC) % NC + 1; k = t / (NC * NC) + 1;
  } else {
    if (cells == 1) return;
    int f = (blockIdx.x - 16) / 2, g = (blockIdx.x - 16) % 2 + 1;
    int n, t1, t2, d[3];
    face_axes(f, n, t1, t2);
    d[n] = (f & 1) ? NC + g : 1 - g;
    d[t1] = threadIdx.x % NC + 1;
    d[t2] = threadIdx.x / NC + 1;
    i = d[0]; j = d[1]; k = d[2];
  }
  int nv = c.nv, q = cid(i, j, k);
  const double *Ab = A + (size_t)b * nv * NSTORE;
  double u[MAXV], p[MAXV];
  if (ghost && Ab[q] == 0.0) return;
  for (int v = 0; v < nv; v++) u[v] = Ab[v * NSTORE + q];
  int st = flow2prim(c.pd, u, p);
  for (int v = c.pd.nv; v < nv; v++) p[v] = u[v];   // passive scalars (hydro_core.f90:372-374)
  double *Pb = P + (size_t)b * nv * NSTORE;
  for (int v = 0; v < nv; v++) Pb[v * NSTORE + q] = p[v];
  if (st && bad && !ghost) atomicAdd(bad, 1ull);
}

// ---------------------------------------------------------------------------
// boundary(depth) and calcPrimsAll(CELLS_GHOST) in one pass: each face ghost
// of the first `exchange` layers is filled from its source, and the
// primitives of both layers are formed from the value in hand (a layer that
// was not exchanged is read; zero density is left alone, as calcPrimsAll
// does, and then keeps the primitives of Pold).  The source of a workgroup's
// cells is of one kind (one face of one block), so nothing diverges.  Bound:
// the lines of the x faces, whose sources lie a row (a 128-byte line) apart;
// both layers go to one workgroup so that it fetches each line once.
// grid (6, nblk).
// ---------------------------------------------------------------------------
template <int NV, int NF>
__global__ void __launch_bounds__(256) k_ghosts(DevCfg c, double *A, double *P, const double *Pold, int exchange) {
  const int b = blockIdx.y, f = blockIdx.x;
  const int a1 = threadIdx.x % NC + 1, a2 = threadIdx.x / NC + 1;
  const int n = f >> 1;
  Phys<double> ph = c.pd;
  ph.nv = NF;
#pragma unroll
  for (int g = 1; g <= 2; g++) {
    const int gn = (f & 1) ? NC + g : 1 - g;
    const int q = n == 0 ? cid(gn, a1, a2) : (n == 1 ? cid(a1, gn, a2) : cid(a1, a2, gn));
    double *Ab = A + (size_t)b * NV * NSTORE + q;
    double *Pb = P + (size_t)b * NV * NSTORE + q;
    double u[NV], p[NV];
    bool have = false;
    if (g <= exchange) {
      GhostSrc s;
      have = ghost_source(c.info, c.bc, b, f, g, a1, a2, s);
      if (have) {
#pragma unroll
        for (int v = 0; v < NV; v++) u[v] = ghost_value<double>(A, NV, s, v);
#pragma unroll
        for (int v = 0; v < NV; v++) Ab[v * NSTORE] = u[v];
      }
    }
    if (!have) u[0] = Ab[0];
    if (u[0] == 0.0) {
      if (Pold != P)
#pragma unroll
        for (int v = 0; v < NV; v++) Pb[v * NSTORE] = Pold[(size_t)b * NV * NSTORE + q + v * NSTORE];
      continue;
    }
    if (!have) {
#pragma unroll
      for (int v = 1; v < NV; v++) u[v] = Ab[v * NSTORE];
    }
    flow2prim(ph, u, p);
#pragma unroll
    for (int v = NF; v < NV; v++) p[v] = u[v];
#pragma unroll
    for (int v = 0; v < NV; v++) Pb[v * NSTORE] = p[v];
  }
}

// ---------------------------------------------------------------------------
// Passive scalars of the hydro solvers, variables pd.nv..nv-1, on states
// already turned to the x direction: a passive's physical flux is u*s
// (prim2fluxes, hydro_core.f90:429-431) and its conserved value s
// (prim2flow :307-309).  HLL and HLL1 take the HLL average
// (hll.f90:186-212); HLLC the star state rho* s_K / rho_K of the side the
// contact leaves (hllc.f90:232-296: 262-264, 283-285).  The wave speeds
// repeat those of the solver, with the same arithmetic.
// ---------------------------------------------------------------------------
__device__ inline void passive_fluxes(const Phys<double> &c, int nv, const double *pL, const double *pR,
                                      double *ff) {
  const double cl = sound(c, pL), cr = sound(c, pR);
  if (c.solver == SOLVER_HLLC) {
    const double dl1 = pL[0], dr1 = pR[0], ul1 = pL[1], ur1 = pR[1], pl1 = pL[4], pr1 = pR[4];
    const double sl = rfmin(ul1 - cl, ur1 - cr);
    const double sr = rfmax(ul1 + cl, ur1 + cr);
    const double sst =
        (pr1 - pl1 + dl1 * ul1 * (sl - ul1) - dr1 * ur1 * (sr - ur1)) / (dl1 * (sl - ul1) - dr1 * (sr - ur1));
    if (sl > 0.0) {
      for (int q = c.nv; q < nv; q++) ff[q] = pL[1] * pL[q];
      return;
    }
    if (sr < 0.0) {
      for (int q = c.nv; q < nv; q++) ff[q] = pR[1] * pR[q];
      return;
    }
    const double *pK;
    double sK;
    if (sst >= 0.0) { pK = pL; sK = sl; }
    else if (sst <= 0.0) { pK = pR; sK = sr; }
    else {
      for (int q = c.nv; q < nv; q++) ff[q] = NAN;
      return;
    }
    const double rhost = pK[0] * (sK - pK[1]) / (sK - sst);
    for (int q = c.nv; q < nv; q++) ff[q] = pK[1] * pK[q] + sK * (rhost * pK[q] / pK[0] - pK[q]);
    return;
  }
  const double sl = rfmin(pL[1] - cl, pR[1] - cr);
  const double sr = rfmax(pL[1] + cl, pR[1] + cr);
  if (sl >= 0.0) {
    for (int q = c.nv; q < nv; q++) ff[q] = pL[1] * pL[q];
    return;
  }
  if (sr <= 0.0) {
    for (int q = c.nv; q < nv; q++) ff[q] = pR[1] * pR[q];
    return;
  }
  for (int q = c.nv; q < nv; q++)
    ff[q] = (sr * (pL[1] * pL[q]) - sl * (pR[1] * pR[q]) + sl * sr * (pR[q] - pL[q])) / (sr - sl);
}

// ---------------------------------------------------------------------------
// HLL*fluxes (hll.f90:52-167, hllc.f90:55-201, hlle.f90:54-158,
// hlld.f90:54-158) and upwindStep (source/godunov.f90:199-277) with
// source_function (source/sources.f90:100-133: the user terms, then Powell's
// :38-95) in one pass.
// ---------------------------------------------------------------------------
// exchange of the x components of velocity and field with those along D
template <int NV, int D> struct Turn {
  __device__ __forceinline__ void operator()(double *v) const { swapdim(NV, D, v); }
};
// the same for y where d holds, per lane: selects, no branch
template <int NV> struct TurnIf {
  bool d;
  __device__ __forceinline__ void operator()(double *v) const {
    const double a = v[1], b = v[2];
    v[1] = d ? b : a;
    v[2] = d ? a : b;
    if (NV == 8) {
      const double e = v[5], f = v[6];
      v[5] = d ? f : e;
      v[6] = d ? e : f;
    }
  }
};

// cells around a face along one axis, as offsets into a block's variable
struct Cells {
  int ll, l, r, rr;
};

// flux between the cells l and r of one block's primitives
template <int NV, int NF, int SOLVER, int ORDER, typename T>
__device__ __forceinline__ void face(const Phys<double> &P, const double *Pb, const Cells &o, const T &turn,
                                     double *ff) {
  double pl[NV], pr[NV];
#pragma unroll
  for (int v = 0; v < NV; v++) {
    pl[v] = Pb[v * NSTORE + o.l];
    pr[v] = Pb[v * NSTORE + o.r];
  }
  if constexpr (ORDER == 2) {
    double pll[NV], prr[NV];
#pragma unroll
    for (int v = 0; v < NV; v++) {
      pll[v] = Pb[v * NSTORE + o.ll];
      prr[v] = Pb[v * NSTORE + o.rr];
    }
    limit_all<NV>(pll, pl, pr, prr, P.limiter);
  }
  turn(pl);
  turn(pr);
  if constexpr (SOLVER == SOLVER_HLLC) primfhllc_sel(P, pl, pr, ff);
  else if constexpr (SOLVER == SOLVER_HLLD) primfhlld_sel(P, pl, pr, ff);
  else if constexpr (SOLVER == SOLVER_HLLE) primfhlle(P, pl, pr, ff);
  else primfhll(P, pl, pr, ff);
  if constexpr (NV > NF) passive_fluxes(P, NV, pl, pr, ff);
  turn(ff);
}

// One workgroup updates L planes of a block; lane (i, j) owns a column.  Per
// plane each lane solves the x face and the y face below its cell and the z
// face above it, straight from the primitives with their ghost layers (the
// neighbours' loads hit the L1); the 32 faces at the far ends of the rows and
// columns go to the last 32 lanes.  x and y fluxes pass through LDS.
//
// Bound: FP64 issue and its latency at 3 waves per SIMD (IEEE divisions and
// square roots of the Riemann solver, 3.1 to 4.1 solves per cell, about 3200
// instructions per MHD cell).  512 MHD blocks (HLLD): 295 us the first stage,
// 348 us the second; with the fluxes through HBM in a pass of their own, and
// run-time variable counts that put the states into scratch, 1753 us each.
// The lower z flux waits in LDS and the upper one is solved last: held in
// registers through the x and y faces it costs a wave per SIMD.
// P2, when given, takes the primitives of the updated interior (the next
// stage's), so that they are not formed in a pass of their own.
template <int NV, int NF, int SOLVER, int ORDER>
__global__ void __launch_bounds__(256, 3)
    k_update(DevCfg c, const double *U, const double *P, double *UP, double *P2, const StepState *ss, double dt_host,
             int half, UserSource us, int L) {
  constexpr int NX = NC + 1;
  constexpr bool S2 = ORDER == 2;
  __shared__ double sfx[NV][NC * NX];   // [v][(j-1)*17 + s]
  __shared__ double sfy[NV][NX * NC];   // [v][s*16 + (i-1)]
  __shared__ double sfz[NV][256];       // z flux below the lane's cell
  const int b = blockIdx.y, k0 = blockIdx.x * L + 1, k1 = k0 + L - 1;
  const int tid = threadIdx.x, ti = tid % NC, tj = tid / NC, i = ti + 1, j = tj + 1;
  const int l = c.info[b].level - 1;
  const double dt = ss ? ss->dt : dt_host;
  const double dtp = half ? dt / 2.0 : dt;
  const double dx = c.dx[0][l], dy = c.dx[1][l], dz = c.dx[2][l];
  const double dtdx = dtp / dx, dtdy = dtp / dy, dtdz = dtp / dz;
  Phys<double> ph = c.pd;
  ph.nv = NF;
  const double *Pb = P + (size_t)b * NV * NSTORE;
  const double *Ub = U + (size_t)b * NV * NSTORE;
  double *UPb = UP + (size_t)b * NV * NSTORE;
  for (int k = k0 - 1; k <= k1; k++) {
    if (k >= k0) {
      {
        double ff[NV];
        face<NV, NF, SOLVER, ORDER>(
            ph, Pb, Cells{S2 ? cid(i - 2, j, k) : 0, cid(i - 1, j, k), cid(i, j, k), S2 ? cid(i + 1, j, k) : 0},
            Turn<NV, 0>{}, ff);
        if (k > k0) __syncthreads();   // the plane below has been read
#pragma unroll
        for (int v = 0; v < NV; v++) sfx[v][tj * NX + ti] = ff[v];
      }
      {
        double ff[NV];
        face<NV, NF, SOLVER, ORDER>(
            ph, Pb, Cells{S2 ? cid(i, j - 2, k) : 0, cid(i, j - 1, k), cid(i, j, k), S2 ? cid(i, j + 1, k) : 0},
            Turn<NV, 1>{}, ff);
#pragma unroll
        for (int v = 0; v < NV; v++) sfy[v][tj * NC + ti] = ff[v];
      }
      if (tid >= 256 - 2 * NC) {
        const bool d = tid >= 256 - NC;            // y face
        const int aa = tid & (NC - 1);             // row or column
        double ff[NV];
        const int one = d ? NC : 1, last = d ? cid(aa + 1, NC, k) : cid(NC, aa + 1, k);
        const int out = d ? cid(aa + 1, NC + 1, k) : cid(NC + 1, aa + 1, k);
        face<NV, NF, SOLVER, ORDER>(ph, Pb, Cells{last - one, last, out, out + NC * NC}, TurnIf<NV>{d}, ff);
#pragma unroll
        for (int v = 0; v < NV; v++) *(d ? &sfy[v][NC * NC + aa] : &sfx[v][aa * NX + NC]) = ff[v];
      }
    }
    // the z face last, so that its flux is not held through the others
    double fzc[NV];
    face<NV, NF, SOLVER, ORDER>(
        ph, Pb, Cells{S2 ? cid(i, j, k - 1) : 0, cid(i, j, k), cid(i, j, k + 1), S2 ? cid(i, j, k + 2) : 0},
        Turn<NV, 2>{}, fzc);
    if (k == k0 - 1) {
#pragma unroll
      for (int v = 0; v < NV; v++) sfz[v][tid] = fzc[v];
      continue;
    }
    __syncthreads();
    const int q = cid(i, j, k);
    double upv[NV];
#pragma unroll
    for (int v = 0; v < NV; v++) {
      upv[v] = Ub[v * NSTORE + q] + dtdx * (sfx[v][tj * NX + ti] - sfx[v][tj * NX + ti + 1]) +
               dtdy * (sfy[v][tj * NC + ti] - sfy[v][(tj + 1) * NC + ti]) + dtdz * (sfz[v][tid] - fzc[v]);
      sfz[v][tid] = fzc[v];
    }
    const bool powell = c.eight_wave && NV == 8;
    if (powell || us.on) {
      double pp[NV];
#pragma unroll
      for (int v = 0; v < NV; v++) pp[v] = Pb[v * NSTORE + q];
      double s[MAXV] = {0, 0, 0, 0, 0, 0, 0, 0};
      if (us.on) user_source(us, pp, s);
      if constexpr (NV == 8) {
        if (powell) {
          const double *Bx = Pb + 5 * NSTORE, *By = Pb + 6 * NSTORE, *Bz = Pb + 7 * NSTORE;
          double divB = (Bx[cid(i + 1, j, k)] - Bx[cid(i - 1, j, k)]) / (2.0 * dx) +
                        (By[cid(i, j + 1, k)] - By[cid(i, j - 1, k)]) / (2.0 * dy) +
                        (Bz[cid(i, j, k + 1)] - Bz[cid(i, j, k - 1)]) / (2.0 * dz);
          s[1] = s[1] - divB * pp[5];
          s[2] = s[2] - divB * pp[6];
          s[3] = s[3] - divB * pp[7];
          s[4] = s[4] - divB * (pp[1] * pp[5] + pp[2] * pp[6] + pp[3] * pp[7]);
          s[5] = s[5] - divB * pp[1];
          s[6] = s[6] - divB * pp[2];
          s[7] = s[7] - divB * pp[3];
        }
      }
#pragma unroll
      for (int v = 0; v < NV; v++) upv[v] = upv[v] + dtp * s[v];
    }
#pragma unroll
    for (int v = 0; v < NV; v++) UPb[v * NSTORE + q] = upv[v];
    if (P2) {
      double p[NV];
      flow2prim(ph, upv, p);
#pragma unroll
      for (int v = NF; v < NV; v++) p[v] = upv[v];   // passive scalars (hydro_core.f90:372-374)
      double *P2b = P2 + (size_t)b * NV * NSTORE;
#pragma unroll
      for (int v = 0; v < NV; v++) P2b[v * NSTORE + q] = p[v];
    }
  }
}

// ---------------------------------------------------------------------------
// doViscousStep (source/hydro_solver.f90:217-250).  grid (16, nblk).
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_viscous(DevCfg c, const double *UP, double *U) {
  int b = blockIdx.y;
  int t = blockIdx.x * 256 + threadIdx.x;
  int i = t % NC + 1, j = (t / NC) % NC + 1, k = t / (NC * NC) + 1;
  int q = cid(i, j, k);
  const int xp = cid(i + 1, j, k), xm = cid(i - 1, j, k), yp = cid(i, j + 1, k), ym = cid(i, j - 1, k),
            zp = cid(i, j, k + 1), zm = cid(i, j, k - 1);
  double eta = c.visc_eta;
  for (int v = 0; v < c.nv; v++) {
    const double *A = UP + ((size_t)b * c.nv + v) * NSTORE;
    U[((size_t)b * c.nv + v) * NSTORE + q] =
        A[q] + eta * (+A[xp] + A[xm] + A[yp] + A[ym] + A[zp] + A[zm] - 6.0 * A[q]);
  }
}

// ---------------------------------------------------------------------------
// getTimestep (source/hydro_solver.f90:129-211): min over interior cells.
// Positive doubles order like their bit patterns, so the global minimum is
// an unsigned 64-bit atomicMin on the bits.  One workgroup and one atomic per
// block, over DT_SLOTS words that the reader folds: atomics on one word are
// served one after the other, about 12 ns each, and one per wavefront of 64
// cells cost more than the pass itself (386 us for 512 MHD blocks).
// ---------------------------------------------------------------------------
template <int NV>
__device__ __forceinline__ double dt_of(const DevCfg &c, const double *p, double dx, double dy, double dz) {
  double dt = 1.0e30;
  if (NV == 8 && c.pd.mhd) {
    double cfx = cfast1(c.pd, p[4], p[0], p[5], p[6], p[7], p[5]);
    double cfy = cfast1(c.pd, p[4], p[0], p[5], p[6], p[7], p[6]);
    double cfz = cfast1(c.pd, p[4], p[0], p[5], p[6], p[7], p[7]);
    dt = fmin(dt, dx / (fabs(p[1]) + cfx));
    dt = fmin(dt, dy / (fabs(p[2]) + cfy));
    dt = fmin(dt, dz / (fabs(p[3]) + cfz));
  } else {
    double cs = sound(c.pd, p);
    dt = fmin(dt, dx / (fabs(p[1]) + cs));
    dt = fmin(dt, dy / (fabs(p[2]) + cs));
    dt = fmin(dt, dz / (fabs(p[3]) + cs));
  }
  return dt;
}

// the smallest dt of a workgroup of 256 lanes into a slot
__device__ __forceinline__ void dt_to_slot(double dt, int slot, unsigned long long *slots) {
  __shared__ double part[4];
  for (int off = 32; off > 0; off >>= 1) dt = fmin(dt, __shfl_xor(dt, off));
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = dt;
  __syncthreads();
  if (threadIdx.x == 0) {
    dt = fmin(fmin(part[0], part[1]), fmin(part[2], part[3]));
    atomicMin(&slots[(slot % DT_SLOTS) * DT_STRIDE], (unsigned long long)__double_as_longlong(dt));
  }
}

template <int NV>
__global__ void __launch_bounds__(256) k_timestep(DevCfg c, const double *P, unsigned long long *slots, int L) {
  const int ns = NC / L, b = blockIdx.x / ns, k0 = blockIdx.x % ns * L + 1;
  const int l = c.info[b].level - 1;
  const int i = threadIdx.x % NC + 1, j = threadIdx.x / NC + 1;
  const double dx = c.dx[0][l], dy = c.dx[1][l], dz = c.dx[2][l];
  constexpr int NP = NV == 8 ? 8 : 5;   // passive scalars don't enter
  const double *Pb = P + (size_t)b * NV * NSTORE;
  double dt = 1.0e30;
#pragma unroll 2
  for (int k = k0; k < k0 + L; k++) {
    const int q = cid(i, j, k);
    double p[MAXV];
#pragma unroll
    for (int v = 0; v < NP; v++) p[v] = Pb[v * NSTORE + q];
    dt = fmin(dt, dt_of<NV>(c, p, dx, dy, dz));
  }
  dt_to_slot(dt, blockIdx.x, slots);
}

// ---------------------------------------------------------------------------
// cooling (source/cooling.f90:37-118, apply_cooling :285-371).  grid (16, nblk)
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_cooling(DevCfg c, double *U, double *P, double dt, double mu0) {
  int b = blockIdx.y;
  int t = blockIdx.x * 256 + threadIdx.x;
  int i = t % NC + 1, j = (t / NC) % NC + 1, k = t / (NC * NC) + 1;
  int nv = c.nv, q = cid(i, j, k);
  double *Pb = P + (size_t)b * nv * NSTORE;
  double pr[5];
  for (int v = 0; v < 5; v++) pr[v] = Pb[v * NSTORE + q];
  // EOS_H_RATE (calcTemp, hydro_core.f90:258-264): P = (n_HI + n_HII) k T
  // with the neutral hydrogen density in the first passive scalar
  const bool hrate = c.eos == 3;
  double th = 0.0;
  if (hrate) th = pr[4] / (2.0 * pr[0] / mu0 - Pb[5 * NSTORE + q]) * c.p_sc / KB;
  double e;
  if (cool_cell(c, dt, pr, &e, hrate, th)) {
    Pb[4 * NSTORE + q] = pr[4];
    U[((size_t)b * nv + 4) * NSTORE + q] = e;
  }
}

// ---------------------------------------------------------------------------
// The end of a step in one pass: doViscousStep (source/hydro_solver.f90:
// 217-250), updatePrims (source/hydro_core.f90:43-59), cooling
// (source/cooling.f90:37-118) and, with slots, getTimestep of the new state.
// The lane of column (i, j) walks L planes and keeps the planes around k in
// registers, so a cell of UP is read once from its column and four times by
// its row and plane (L1).  The last 12 nblk workgroups form the primitives of
// the face ghosts, as updatePrims does; they come after all others, so that
// every chiplet (workgroups are dealt to them in turn) gets its share of the
// interior.  grid (16/L + 12) nblk.
// ---------------------------------------------------------------------------
template <int NV, int NF>
__global__ void __launch_bounds__(256) k_finish(DevCfg c, const double *UP, double *U, double *P,
                                                StepState *ss, double mu0, unsigned long long *slots, int L) {
  const int ns = NC / L, slab = blockIdx.x % ns;
  const bool inside = (int)blockIdx.x < c.nblk * ns;
  const int gw = (int)blockIdx.x - c.nblk * ns;
  const int b = inside ? blockIdx.x / ns : gw / 12;
  Phys<double> ph = c.pd;
  ph.nv = NF;
  double *Ub = U + (size_t)b * NV * NSTORE, *Pb = P + (size_t)b * NV * NSTORE;
  if (!inside) {
    const int e = gw % 12, f = e >> 1, g = (e & 1) + 1;
    const int a1 = threadIdx.x % NC + 1, a2 = threadIdx.x / NC + 1;
    const int n = f >> 1, gn = (f & 1) ? NC + g : 1 - g;
    const int q = n == 0 ? cid(gn, a1, a2) : (n == 1 ? cid(a1, gn, a2) : cid(a1, a2, gn));
    double u[NV], p[NV];
    u[0] = Ub[q];
    if (u[0] == 0.0) return;
#pragma unroll
    for (int v = 1; v < NV; v++) u[v] = Ub[v * NSTORE + q];
    flow2prim(ph, u, p);
#pragma unroll
    for (int v = NF; v < NV; v++) p[v] = u[v];
#pragma unroll
    for (int v = 0; v < NV; v++) Pb[v * NSTORE + q] = p[v];
    return;
  }
  const int l = c.info[b].level - 1;
  const double dx = c.dx[0][l], dy = c.dx[1][l], dz = c.dx[2][l];
  const int i = threadIdx.x % NC + 1, j = threadIdx.x / NC + 1, k0 = slab * L + 1;
  const double eta = c.visc_eta, dt = ss->dt;
  const double *A = UP + (size_t)b * NV * NSTORE;
  double below[NV], here[NV], dtmin = 1.0e30;
  int floors = 0;
#pragma unroll
  for (int v = 0; v < NV; v++) {
    below[v] = A[v * NSTORE + cid(i, j, k0 - 1)];
    here[v] = A[v * NSTORE + cid(i, j, k0)];
  }
  for (int k = k0; k < k0 + L; k++) {
    const int q = cid(i, j, k), xp = cid(i + 1, j, k), xm = cid(i - 1, j, k), yp = cid(i, j + 1, k),
              ym = cid(i, j - 1, k), zp = cid(i, j, k + 1);
    double u[NV], p[NV], above[NV];
#pragma unroll
    for (int v = 0; v < NV; v++) {
      const double *a = A + v * NSTORE;
      above[v] = a[zp];
      u[v] = here[v] + eta * (+a[xp] + a[xm] + a[yp] + a[ym] + above[v] + below[v] - 6.0 * here[v]);
    }
#pragma unroll
    for (int v = 0; v < NV; v++) {
      below[v] = here[v];
      here[v] = above[v];
    }
    if (flow2prim(ph, u, p)) floors++;
#pragma unroll
    for (int v = NF; v < NV; v++) p[v] = u[v];   // passive scalars (hydro_core.f90:372-374)
    if (c.cooling) {
      double e, th = 0.0;
      const bool hrate = NV > NF && c.eos == 3;
      if constexpr (NV > NF) {
        if (hrate) th = p[4] / (2.0 * p[0] / mu0 - p[5]) * c.p_sc / KB;   // see k_cooling
      }
      if (cool_cell(c, dt, p, &e, hrate, th)) u[4] = e;
    }
#pragma unroll
    for (int v = 0; v < NV; v++) {
      Ub[v * NSTORE + q] = u[v];
      Pb[v * NSTORE + q] = p[v];
    }
    if (slots) dtmin = fmin(dtmin, dt_of<NV>(c, p, dx, dy, dz));
  }
  if (floors) atomicAdd(&ss->floors, (unsigned long long)floors);
  if (slots) dt_to_slot(dtmin, blockIdx.x, slots);
}

// The scalars of a step: closes the step before it, then dt from the smallest
// of the slots with the start-up ramp and the output clamp
// (source/hydro_solver.f90:183-207).  One wavefront.
__global__ void __launch_bounds__(64) k_step_begin(StepState *s, unsigned long long *slots, double cfl, int cooling) {
  const double m = fold_slots(slots);
  if (threadIdx.x == 0) {
    step_close(s);
    step_open(s, m, cfl, cooling);
  }
}

// the smallest of the slots into *out, the slots cleared
__global__ void __launch_bounds__(64) k_dt_fold(unsigned long long *slots, unsigned long long *out) {
  const double m = fold_slots(slots);
  if (threadIdx.x == 0) *out = (unsigned long long)__double_as_longlong(m);
}

// ---------------------------------------------------------------------------
// markByPhysical (source/amr.f90:142-230), the per-block part: the largest
// |q(i+1) - q(i-1)| / q(i) / (2 dx) along x, y and z over the interior
// cells, for q = pressure and q = density, read from PRIM with its depth-1
// face ghosts.  dx is the level's x spacing in all three directions, as in
// the reference.  The reference returns at the first cell whose gradient
// reaches the refinement threshold; which flag it returns then depends only
// on the level, so the flag is a function of this maximum (set on the host).
// One variable at a time is staged in LDS as an 18^3 cube (its edges and
// corners are not read), every line of the block's interior and inner ghost
// planes loaded once; the division by the common 2 dx > 0, which keeps the
// order of the quotients, comes after the maximum.  grid nblk, block 1024.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(1024) k_mark(DevCfg c, const double *P, double *maxgrad) {
  constexpr int E = NC + 2;
  __shared__ double cube[E * E * E];
  __shared__ double part[16];
  const int b = blockIdx.x, t = threadIdx.x;
  const double two_dx = 2.0 * c.dx[0][c.info[b].level - 1];
  double m = 0.0;
  for (int s = 0; s < 2; s++) {
    const double *A = P + ((size_t)b * c.nv + (s == 0 ? 4 : 0)) * NSTORE;
    if (s) __syncthreads();
    for (int q = t; q < NINT; q += 1024)
      cube[((q / (NC * NC) + 1) * E + (q / NC) % NC + 1) * E + q % NC + 1] = A[q];
    for (int r = t; r < 6 * 256; r += 1024) {
      const int f = r >> 8, a1 = (r & 255) % NC + 1, a2 = (r & 255) / NC + 1, gn = (f & 1) ? NC + 1 : 0;
      const int i = f < 2 ? gn : a1, j = f < 2 ? a1 : (f < 4 ? gn : a2), k = f < 4 ? a2 : gn;
      cube[(k * E + j) * E + i] = A[cid(i, j, k)];
    }
    __syncthreads();
    for (int q = t; q < NINT; q += 1024) {
      const int o = ((q / (NC * NC) + 1) * E + (q / NC) % NC + 1) * E + q % NC + 1;
      const double a = cube[o];
      const double gx = fabs(cube[o + 1] - cube[o - 1]) / a;
      const double gy = fabs(cube[o + E] - cube[o - E]) / a;
      const double gz = fabs(cube[o + E * E] - cube[o - E * E]) / a;
      m = fmax(m, fmax(gx, fmax(gy, gz)));
    }
  }
  for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o));
  if ((t & 63) == 0) part[t >> 6] = m;
  __syncthreads();
  if (t == 0) {
    double r = part[0];
    for (int w = 1; w < 16; w++) r = fmax(r, part[w]);
    maxgrad[b] = r / two_dx;
  }
}

// ---------------------------------------------------------------------------
// The same for the fused form, whose state has no ghost layers
// ([blk][nv][16^3] FP64): density and pressure of the depth-1 face ghosts
// are formed from the sources the exchange reads (same-level copy,
// coarse->fine injection, fine->coarse 8-cell average, domain faces) and
// the wind sources, with the plain form's arithmetic, then flow2prim.
// ---------------------------------------------------------------------------
__device__ inline double ghost_value_int(const double *U, int nv, const GhostSrc &s, int v) {
  const double *S = U + ((size_t)s.blk * nv + v) * NINT;
  if (s.kind == 1) {
    double acc = 0.0;
    for (int dx = 0; dx < 2; dx++)
      for (int dy = 0; dy < 2; dy++)
        for (int dz = 0; dz < 2; dz++)
          acc = acc + S[((s.c[2] + dz - 1) * NC + (s.c[1] + dy - 1)) * NC + (s.c[0] + dx - 1)] / 8.0;
    return acc;
  }
  double val = S[((s.c[2] - 1) * NC + (s.c[1] - 1)) * NC + (s.c[0] - 1)];
  if (s.kind == 2 && v == s.flip) val = -1.0 * val;
  return val;
}

// density and pressure of ghost (a1, a2) of face f, layer 1, of block b
__device__ inline void ghost_rho_p(const DevCfg &c, const double *U, int b, int f, int a1, int a2, double &rho,
                                   double &pres) {
  GhostSrc s;
  double u[MAXV], p[MAXV];
  if (!ghost_source(c.info, c.bc, b, f, 1, a1, a2, s)) {
    rho = pres = 0.0;
    return;
  }
  for (int v = 0; v < c.nv; v++) u[v] = ghost_value_int(U, c.nv, s, v);
  int n, t1, t2, d[3];
  face_axes(f, n, t1, t2);
  d[n] = (f & 1) ? NC + 1 : 0;
  d[t1] = a1;
  d[t2] = a2;
  wind_state(c, b, d[0], d[1], d[2], u);
  flow2prim(c.pd, u, p);
  rho = p[0];
  pres = p[4];
}

// Recorded ghost layer: G[blk][2 (rho, p)][6 faces][256].  grid (6, nblk).
__global__ void __launch_bounds__(256) k_ghost_prims_fused(DevCfg c, const double *U, double *G) {
  const int b = blockIdx.y, f = blockIdx.x;
  double rho, pres;
  ghost_rho_p(c, U, b, f, threadIdx.x % NC + 1, threadIdx.x / NC + 1, rho, pres);
  G[(((size_t)b * 2 + 0) * 6 + f) * 256 + threadIdx.x] = rho;
  G[(((size_t)b * 2 + 1) * 6 + f) * 256 + threadIdx.x] = pres;
}

// markByPhysical on the fused state: density and pressure of the block and
// its depth-1 face ghosts (from G, or formed from U when G is null) staged
// in LDS as an 18^3 cube, then the maximum of k_mark.  grid nblk, 1024
// threads (93 KB of LDS: one workgroup of 16 waves per CU).
__global__ void __launch_bounds__(1024) k_mark_fused(DevCfg c, const double *U, const double *G, double *maxgrad) {
  constexpr int E = NC + 2;
  __shared__ double sr[E * E * E], sp[E * E * E];
  __shared__ double part[16];
  const int b = blockIdx.x, t = threadIdx.x, nv = c.nv;
  for (int q = t; q < NINT; q += 1024) {
    double u[MAXV], p[MAXV];
    for (int v = 0; v < nv; v++) u[v] = U[((size_t)b * nv + v) * NINT + q];
    flow2prim(c.pd, u, p);
    const int i = q % NC + 1, j = (q / NC) % NC + 1, k = q / (NC * NC) + 1;
    sr[(k * E + j) * E + i] = p[0];
    sp[(k * E + j) * E + i] = p[4];
  }
  for (int r = t; r < 6 * 256; r += 1024) {
    const int f = r >> 8, a1 = (r & 255) % NC + 1, a2 = (r & 255) / NC + 1;
    double rho, pres;
    if (G) {
      rho = G[(((size_t)b * 2 + 0) * 6 + f) * 256 + (r & 255)];
      pres = G[(((size_t)b * 2 + 1) * 6 + f) * 256 + (r & 255)];
    } else {
      ghost_rho_p(c, U, b, f, a1, a2, rho, pres);
    }
    int n, t1, t2, d[3];
    face_axes(f, n, t1, t2);
    d[n] = (f & 1) ? NC + 1 : 0;
    d[t1] = a1;
    d[t2] = a2;
    sr[(d[2] * E + d[1]) * E + d[0]] = rho;
    sp[(d[2] * E + d[1]) * E + d[0]] = pres;
  }
  __syncthreads();
  const double two_dx = 2.0 * c.dx[0][c.info[b].level - 1];
  double m = 0.0;
  for (int s2 = 0; s2 < 2; s2++) {
    const double *A = s2 == 0 ? sp : sr;
    for (int q = t; q < NINT; q += 1024) {
      const int o = ((q / (NC * NC) + 1) * E + (q / NC) % NC + 1) * E + q % NC + 1;
      const double a = A[o];
      const double gx = fabs(A[o + 1] - A[o - 1]) / a / two_dx;
      const double gy = fabs(A[o + E] - A[o - E]) / a / two_dx;
      const double gz = fabs(A[o + E * E] - A[o - E * E]) / a / two_dx;
      m = fmax(m, fmax(gx, fmax(gy, gz)));
    }
  }
  for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o));
  if ((t & 63) == 0) part[t >> 6] = m;
  __syncthreads();
  if (t == 0) {
    double r = part[0];
    for (int w = 1; w < 16; w++) r = fmax(r, part[w]);
    maxgrad[b] = r;
  }
}

// ---------------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------------
// planes per workgroup: whole columns once the mesh alone gives `want`
// workgroups, thinner slabs below that
static int planes_for(int nblk, int want) {
  int L = NC;
  while (L > 1 && nblk * (NC / L) < want) L >>= 1;
  return L;
}

// stored variables (with passive scalars) and flow variables as constants
#define WX_BY_NV(nv, CALL)                     \
  do {                                         \
    switch (nv) {                              \
      case 5: { CALL(5, 5); break; }           \
      case 6: { CALL(6, 5); break; }           \
      case 7: { CALL(7, 5); break; }           \
      default: { CALL(8, 8); break; }          \
    }                                          \
  } while (0)

void plain_boundary(const DevCfg &c, const PlaneWind &pw, double *A, int depth, hipStream_t st) {
  hipLaunchKernelGGL(k_boundary, dim3(6 * depth, c.nblk), dim3(256), 0, st, c, A, depth);
  double *none = nullptr;
  if (c.nwind > 0 || pw.plane != 0) hipLaunchKernelGGL(k_winds, dim3(28, c.nblk), dim3(256), 0, st, c, A, pw, none);
}
void plain_ghosts(const DevCfg &c, const PlaneWind &pw, double *A, double *P, const double *Pold, int depth,
                  double *Pcover, hipStream_t st) {
  int exchange = depth;
  if (c.nwind > 0 || pw.plane != 0) {
    // a source covers ghosts too: it comes between the exchange and the primitives
    hipLaunchKernelGGL(k_boundary, dim3(6 * depth, c.nblk), dim3(256), 0, st, c, A, depth);
    hipLaunchKernelGGL(k_winds, dim3(28, c.nblk), dim3(256), 0, st, c, A, pw, Pcover);
    exchange = 0;
  }
#define WX_CALL(NV, NF) \
  hipLaunchKernelGGL((k_ghosts<NV, NF>), dim3(6, c.nblk), dim3(256), 0, st, c, A, P, Pold, exchange)
  WX_BY_NV(c.nv, WX_CALL);
#undef WX_CALL
}
void plain_prims(const DevCfg &c, const double *A, double *P, int cells, unsigned long long *bad,
                 hipStream_t st) {
  hipLaunchKernelGGL(k_prims, dim3(28, c.nblk), dim3(256), 0, st, c, A, P, cells, bad);
}

template <int NV, int NF, int SOLVER>
static void launch_update(const DevCfg &c, const UserSource &us, const double *U, const double *P, double *UP,
                          double *P2, const StepState *ss, double dt, int half, int order, hipStream_t st) {
  const int L = planes_for(c.nblk, WX_UPDATE_WANT);
  const dim3 grid(NC / L, c.nblk);
  if (order == 2)
    hipLaunchKernelGGL((k_update<NV, NF, SOLVER, 2>), grid, dim3(256), 0, st, c, U, P, UP, P2, ss, dt, half, us, L);
  else
    hipLaunchKernelGGL((k_update<NV, NF, SOLVER, 1>), grid, dim3(256), 0, st, c, U, P, UP, P2, ss, dt, half, us, L);
}

void plain_update(const DevCfg &c, const UserSource &us, const double *U, const double *P, double *UP, double *P2,
                  const StepState *ss, double dt, int half, int order, hipStream_t st) {
  const int solver = c.pd.solver;
  if (c.nv == 8 && solver == SOLVER_HLLD)
    return launch_update<8, 8, SOLVER_HLLD>(c, us, U, P, UP, P2, ss, dt, half, order, st);
  if (c.nv == 8 && solver == SOLVER_HLLE)
    return launch_update<8, 8, SOLVER_HLLE>(c, us, U, P, UP, P2, ss, dt, half, order, st);
#define WX_CALL(NV, NF)                                                                            \
  if (solver == SOLVER_HLLC) launch_update<NV, NF, SOLVER_HLLC>(c, us, U, P, UP, P2, ss, dt, half, order, st); \
  else launch_update<NV, NF, SOLVER_HLL>(c, us, U, P, UP, P2, ss, dt, half, order, st)
  WX_BY_NV(c.nv, WX_CALL);
#undef WX_CALL
}
void plain_viscous(const DevCfg &c, const double *UP, double *U, hipStream_t st) {
  hipLaunchKernelGGL(k_viscous, dim3(16, c.nblk), dim3(256), 0, st, c, UP, U);
}
void plain_finish(const DevCfg &c, const double *UP, double *U, double *P, StepState *ss, double mu0,
                  unsigned long long *slots, hipStream_t st) {
  const int L = planes_for(c.nblk, WX_FINISH_WANT);
#define WX_CALL(NV, NF)                                                                                          \
  hipLaunchKernelGGL((k_finish<NV, NF>), dim3((NC / L + 12) * c.nblk), dim3(256), 0, st, c, UP, U, P, ss, mu0, slots, L)
  WX_BY_NV(c.nv, WX_CALL);
#undef WX_CALL
}
static void launch_timestep(const DevCfg &c, const double *P, unsigned long long *slots, hipStream_t st) {
  const int L = planes_for(c.nblk, WX_TIMESTEP_WANT);
#define WX_CALL(NV, NF) hipLaunchKernelGGL(k_timestep<NV>, dim3(NC / L * c.nblk), dim3(256), 0, st, c, P, slots, L)
  WX_BY_NV(c.nv, WX_CALL);
#undef WX_CALL
}
void plain_timestep(const DevCfg &c, const double *P, unsigned long long *slots, unsigned long long *dtbits,
                    hipStream_t st) {
  launch_timestep(c, P, slots, st);
  hipLaunchKernelGGL(k_dt_fold, dim3(1), dim3(64), 0, st, slots, dtbits);
}
void plain_step_begin(const DevCfg &c, const double *P, StepState *ss, unsigned long long *slots, hipStream_t st) {
  if (P) launch_timestep(c, P, slots, st);
  hipLaunchKernelGGL(k_step_begin, dim3(1), dim3(64), 0, st, ss, slots, c.cfl, c.cooling);
}
void plain_cooling(const DevCfg &c, double *U, double *P, double dt, double mu0, hipStream_t st) {
  hipLaunchKernelGGL(k_cooling, dim3(16, c.nblk), dim3(256), 0, st, c, U, P, dt, mu0);
}
void plain_mark(const DevCfg &c, const double *P, double *maxgrad, hipStream_t st) {
  hipLaunchKernelGGL(k_mark, dim3(c.nblk), dim3(1024), 0, st, c, P, maxgrad);
}
void fused_ghost_prims(const DevCfg &c, const double *U, double *G, hipStream_t st) {
  hipLaunchKernelGGL(k_ghost_prims_fused, dim3(6, c.nblk), dim3(256), 0, st, c, U, G);
}
void fused_mark(const DevCfg &c, const double *U, const double *G, double *maxgrad, hipStream_t st) {
  hipLaunchKernelGGL(k_mark_fused, dim3(c.nblk), dim3(1024), 0, st, c, U, G, maxgrad);
}

}  // namespace wx
