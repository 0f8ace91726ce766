// wx_hydro_kern.h - the stage kernels of the fused hydro form and of FP64 MHD,
// and the kernel that ends a step.
//
// One workgroup of 256 lanes updates L planes of a block; lane (i, j) owns a
// column.  Per plane the primitives of the plane and its x/y face halo sit in
// LDS (x and y faces), those of the column around it in registers (z faces).
// The end of the step (viscosity, primitives, cooling, dt) is a kernel of its
// own: it needs the updated neighbours of a cell, which inside the second
// stage means carrying two more planes of FP64 state, and the cooling's
// transcendentals, through the flux code, at a third of the registers spilled
// (162 VGPRs for HLLC).  Apart, the FP32 stages hold all their values (with wind
// sources and a run-time limiter 2 to 3 VGPRs go to scratch), and the end of the
// step all but 36 bytes a lane of a few instances; the FP64 MHD second stage
// still puts out 9 VGPRs (HLLE with minmod) to 25 (a run-time limiter).  Thin
// slabs need no recomputed planes.  The state in between costs 16 B per variable
// and zone, also where there is neither viscosity nor cooling (25 of 375 us for
// 240 FP64 MHD blocks).
//
// Bound: VALU issue at 4 waves per SIMD (FP32 stages, 128 VGPRs), memory and its
// latency at 3 (end of the step).  1728 blocks, HLLC with viscosity: first stage
// 450 -> 187 us, second 878 -> 238 + 210 us (end); 904 blocks on 4 levels with
// cooling 299 -> 121 and 784 -> 157 + 184 us; 64 blocks, where one workgroup per
// block left 192 of 256 CUs idle, 127 -> 14 and 221 -> 16 + 10 us.
#pragma once

#include <type_traits>

#include "wx_fused_kern.h"

namespace wx {

// Work item w of a grid over nblk blocks x nslab slabs: position in the block
// order and slab.  Workgroups are dealt to the 8 chiplets (XCDs) in turn; the
// slabs of a block go to one of them, so that the planes and halos they share
// come from one L2.
__device__ __forceinline__ void item_of(int w, int nblk, int nslab, int &bi, int &slab) {
  const int full = (nblk & ~7) * nslab;
  if (w < full) {
    const int r = w >> 3;
    bi = (r / nslab) * 8 + (w & 7);
    slab = r % nslab;
  } else {
    bi = (nblk & ~7) + (w - full) / nslab;
    slab = (w - full) % nslab;
  }
}

// State of cell (i, j, k) of block b in the storage type: load_cell without
// the round trip through FP64 (an average over finer cells is formed in FP64
// and rounded)
template <typename T, int NV, bool WIN, bool WINDS>
__device__ __forceinline__ void load_state(const FusedArgs &a, const T *W, int b, int i, int j, int k, T *u) {
  const bool in = (unsigned)(i - 1) < NC && (unsigned)(j - 1) < NC && (unsigned)(k - 1) < NC;
  if (in) {
    const T *Wb = W + (size_t)b * NV * NINT + lin(i, j, k);
#pragma unroll
    for (int v = 0; v < NV; v++) u[v] = Wb[v * NINT];
  } else {
    double d[NV];
    load_cell<T, NV, WIN, false, false>(a, W, b, i, j, k, d);
#pragma unroll
    for (int v = 0; v < NV; v++) u[v] = (T)d[v];
  }
  if constexpr (WINDS) {
    if (WIN || !in) {
      double w[MAXV];
      if (wind_state(a.c, b, i, j, k, w)) {
#pragma unroll
        for (int v = 0; v < NV; v++) u[v] = (T)w[v];
      }
    }
  }
}

// primitives in the flux precision: the first stage's pressure from the FP64
// state in FP64, the second's from the half-step state in its own type
template <int NV, typename RF, bool S2, typename T>
__device__ __forceinline__ void stage_prims(const Phys<double> &pd, const Phys<RF> &P, const T *u, RF *p) {
  if constexpr (S2) {
    RF ur[NV];
#pragma unroll
    for (int v = 0; v < NV; v++) ur[v] = (RF)u[v];
    flow2prim(P, ur, p);
  } else {
    double d[NV], q[NV];
#pragma unroll
    for (int v = 0; v < NV; v++) d[v] = (double)u[v];
    flow2prim(pd, d, q);
#pragma unroll
    for (int v = 0; v < NV; v++) p[v] = (RF)q[v];
  }
}

// rot for y where d holds, per lane
template <int NV, typename R> __device__ __forceinline__ void rot_y_if(bool d, R *v) {
  const R a = v[1], b = v[2];
  v[1] = d ? b : a;
  v[2] = d ? a : b;
  if constexpr (NV == 8) {
    const R e = v[5], f = v[6];
    v[5] = d ? f : e;
    v[6] = d ? e : f;
  }
}

// limited states and flux of one face in the x-aligned order
template <int NV, int SOLVER, int LIM, bool S2, typename RF>
__device__ __forceinline__ void flow_face(const Phys<RF> &P, const RF *pll, RF *pl, RF *pr, const RF *prr, RF *ff) {
  if constexpr (S2) {
    if constexpr (LIM == LIM_RUNTIME) {
      limit_all<NV>(pll, pl, pr, prr, P.limiter);
    } else {
#pragma unroll
      for (int v = 0; v < NV; v++) limit1(pll[v], pl[v], pr[v], prr[v], LIM);
    }
  }
  if constexpr (SOLVER == SOLVER_HLLC) primfhllc_sel(P, pl, pr, ff);
  else if constexpr (SOLVER == SOLVER_HLLD) primfhlld_sel(P, pl, pr, ff);
  else if constexpr (SOLVER == SOLVER_HLLE) primfhlle(P, pl, pr, ff);
  else primfhll(P, pl, pr, ff);
}

template <int NV, bool S2, typename RF, typename ST, int SOLVER, int LIM, bool WINDS>
__global__ void __launch_bounds__(256, sizeof(RF) == 4 ? 4 : 2) k_flow(FusedArgs a) {
  constexpr bool MHD = NV == 8;
  constexpr int H = S2 ? 2 : 1;            // halo depth of the stencil
  constexpr int W = NC + 2 * H;
  constexpr int WP = W | 1;                // LDS row pitch
  constexpr int NX = NC + 1;
  constexpr int NW = S2 ? 4 : (MHD ? 3 : 2);   // planes in the column window
  constexpr int C = NW - 1 - H;                // plane k in the window (with k-1 for the second order and Powell)
  using T = typename std::conditional<S2, ST, double>::type;
  __shared__ RF sp[NV][W * WP];            // primitives of the plane and its x/y halo
  __shared__ RF sfx[NV][NC * NX];          // x fluxes [v][(j-1)*17 + s]
  __shared__ RF sfy[NV][NX * NC];          // y fluxes [v][s*16 + (i-1)]
  // sources of the halo found once per block (1728 blocks 0.749 -> 0.683 ms a
  // step, 904 on four levels 466 -> 449 us); not with wind code (over 30 VGPRs
  // pushed out: 500 -> 536 us) nor in FP64 (343 -> 349 us)
  constexpr bool HREF = !WINDS && sizeof(RF) == 4;
  __shared__ HaloRef sref[HREF ? 4 * H * NC : 1];

  const DevCfg &c = a.c;
  Phys<RF> P = phys<RF>(c);
  Phys<double> pd = c.pd;
  P.nv = pd.nv = NV;
  P.mhd = pd.mhd = MHD;
  const T *in;
  if constexpr (S2) in = static_cast<const ST *>(a.UPin);
  else in = a.U;
  const int tid = threadIdx.x, ti = tid & 15, tj = tid >> 4, i = ti + 1, j = tj + 1;
  const double dt = a.step->dt;
  const double dtp = S2 ? dt : dt / 2.0;
  // halo cell of this lane: side, layer, position along the side
  const bool hth = tid < 4 * H * NC;
  int hi, hj;
  {
    const int part = tid / (2 * H * NC), r = tid % (2 * H * NC), side = r / (H * NC);
    const int g = (r % (H * NC)) / NC + 1, aa = r % NC + 1, at = side ? NC + g : 1 - g;
    hi = part == 0 ? at : aa;
    hj = part == 0 ? aa : at;
  }
  const int own = (j - 1 + H) * WP + (i - 1 + H);
  const int L = NC / a.nslab;

  for (int w = blockIdx.x; w < a.nblk * a.nslab; w += gridDim.x) {
    int bi, slab;
    item_of(w, a.nblk, a.nslab, bi, slab);
    const int b = a.order[bi];
    WX_EMU_CHECK(b >= 0 && b < a.nblk);
    const int k0 = slab * L + 1, k1 = k0 + L - 1;
    const int l = c.info[b].level - 1;
    const double dtdx = dtp / c.dx[0][l], dtdy = dtp / c.dx[1][l], dtdz = dtp / c.dx[2][l];
    // (RF)(1.0 / (2.0 * dx)): central differences of Powell's source
    const RF idx2 = (RF)(1.0 / (2.0 * c.dx[0][l])), idy2 = (RF)(1.0 / (2.0 * c.dx[1][l])),
             idz2 = (RF)(1.0 / (2.0 * c.dx[2][l]));
    if (HREF && hth) sref[tid] = halo_ref<false>(a, b, hi, hj);   // read back by the lane that wrote it
    RF win[NW][NV], fzp[NV];
    // Iteration k loads plane k + H of the column; the first iterations only
    // fill the window (one call site of the load, with its ghost paths).
    // The bottom face of a slab is solved by the slab below it as well, from
    // the same values at the same place.
    for (int k = k0 - 1 - (NW - 1); k <= k1; k++) {
#pragma unroll
      for (int q = 0; q < NW - 1; q++)
#pragma unroll
        for (int v = 0; v < NV; v++) win[q][v] = win[q + 1][v];
      {
        T u[NV];
        load_state<T, NV, S2, WINDS>(a, in, b, i, j, k + H, u);
        stage_prims<NV, RF, S2>(pd, P, u, win[NW - 1]);
      }
      if (k < k0 - 1) continue;
      T uh[NV];
      if (hth && k >= k0) {
        const HaloRef href = HREF ? sref[tid] : HaloRef{-1, 0};
        if (href.blk >= 0) {
          const T *S = in + (size_t)href.blk * NV * NINT + href.at(k);
#pragma unroll
          for (int v = 0; v < NV; v++) uh[v] = S[v * NINT];
        } else {
          load_state<T, NV, S2, WINDS>(a, in, b, hi, hj, k, uh);
        }
      }
      // z flux (k | k+1)
      RF fzc[NV];
      {
        RF pll[NV], pl[NV], pr[NV], prr[NV];
#pragma unroll
        for (int v = 0; v < NV; v++) {
          pl[v] = win[C][v];
          pr[v] = win[C + 1][v];
          if constexpr (S2) {
            pll[v] = win[0][v];
            prr[v] = win[NW - 1][v];
          }
        }
        rot<NV>(2, pl);
        rot<NV>(2, pr);
        if constexpr (S2) {
          rot<NV>(2, pll);
          rot<NV>(2, prr);
        }
        flow_face<NV, SOLVER, LIM, S2>(P, pll, pl, pr, prr, fzc);
        rot<NV>(2, fzc);
      }
      if (k >= k0) {
        // the faces of the plane below were solved before the last barrier
#pragma unroll
        for (int v = 0; v < NV; v++) sp[v][own] = win[C][v];
        if (hth) {
          RF ph[NV];
          stage_prims<NV, RF, S2>(pd, P, uh, ph);
#pragma unroll
          for (int v = 0; v < NV; v++) sp[v][(hj - 1 + H) * WP + (hi - 1 + H)] = ph[v];
        }
        __syncthreads();
        // x faces s = 0..15, one per lane
        {
          const int base = (tj + H) * WP + (ti - 1 + H);        // cell s
          RF pll[NV], pl[NV], pr[NV], prr[NV], ff[NV];
#pragma unroll
          for (int v = 0; v < NV; v++) {
            const RF *x = &sp[v][base];
            pl[v] = x[0];
            pr[v] = x[1];
            if constexpr (S2) {
              pll[v] = x[-1];
              prr[v] = x[2];
            }
          }
          flow_face<NV, SOLVER, LIM, S2>(P, pll, pl, pr, prr, ff);
#pragma unroll
          for (int v = 0; v < NV; v++) sfx[v][tj * NX + ti] = ff[v];
        }
        // y faces s = 0..15
        {
          const int base = (tj - 1 + H) * WP + (ti + H);
          RF pll[NV], pl[NV], pr[NV], prr[NV], ff[NV];
#pragma unroll
          for (int v = 0; v < NV; v++) {
            const RF *x = &sp[v][base];
            pl[v] = x[0];
            pr[v] = x[WP];
            if constexpr (S2) {
              pll[v] = x[-WP];
              prr[v] = x[2 * WP];
            }
          }
          rot<NV>(1, pl);
          rot<NV>(1, pr);
          if constexpr (S2) {
            rot<NV>(1, pll);
            rot<NV>(1, prr);
          }
          flow_face<NV, SOLVER, LIM, S2>(P, pll, pl, pr, prr, ff);
          rot<NV>(1, ff);
#pragma unroll
          for (int v = 0; v < NV; v++) sfy[v][tj * NC + ti] = ff[v];
        }
        // Powell's div B of the plane, while its primitives are in LDS
        RF divB = RF(0);
        if constexpr (MHD) {
          if (c.eight_wave)
            divB = (sp[5][own + 1] - sp[5][own - 1]) * idx2 + (sp[6][own + WP] - sp[6][own - WP]) * idy2 +
                   (win[C + 1][7] - win[C - 1][7]) * idz2;
        }
        // the 16 x and 16 y faces s = 16 on the last 32 lanes
        if (tid >= 256 - 2 * NC) {
          const bool d = tid >= 256 - NC;                        // y face
          const int aa = tid & (NC - 1), st = d ? WP : 1;
          const int base = d ? (NC - 1 + H) * WP + (aa + H) : (aa + H) * WP + (NC - 1 + H);
          RF pll[NV], pl[NV], pr[NV], prr[NV], ff[NV];
#pragma unroll
          for (int v = 0; v < NV; v++) {
            const RF *x = &sp[v][base];
            pl[v] = x[0];
            pr[v] = x[st];
            if constexpr (S2) {
              pll[v] = x[-st];
              prr[v] = x[2 * st];
            }
          }
          rot_y_if<NV>(d, pl);
          rot_y_if<NV>(d, pr);
          if constexpr (S2) {
            rot_y_if<NV>(d, pll);
            rot_y_if<NV>(d, prr);
          }
          flow_face<NV, SOLVER, LIM, S2>(P, pll, pl, pr, prr, ff);
          rot_y_if<NV>(d, ff);
#pragma unroll
          for (int v = 0; v < NV; v++) *(d ? &sfy[v][NC * NC + aa] : &sfx[v][aa * NX + NC]) = ff[v];
        }
        __syncthreads();
        // conservative update of cell (i, j, k) in FP64 (the flux differences
        // of FP32 operands are exact, so the sum over cells telescopes)
        const size_t at = (size_t)b * NV * NINT + lin(i, j, k);
        double ub[NV];
#pragma unroll
        for (int v = 0; v < NV; v++) ub[v] = a.U[at + v * NINT];
        if constexpr (WINDS) {
          double ws[MAXV];
          if (wind_state(c, b, i, j, k, ws))
#pragma unroll
            for (int v = 0; v < NV; v++) ub[v] = ws[v];
        }
        double un[NV];
#pragma unroll
        for (int v = 0; v < NV; v++)
          un[v] = ub[v] + dtdx * ((double)sfx[v][tj * NX + ti] - (double)sfx[v][tj * NX + ti + 1]) +
                  dtdy * ((double)sfy[v][tj * NC + ti] - (double)sfy[v][(tj + 1) * NC + ti]) +
                  dtdz * ((double)fzp[v] - (double)fzc[v]);
        if constexpr (MHD) {
          if (c.eight_wave) {
            // Powell source (source/sources.f90:38-95) from the stage primitives
            const RF *pp = win[C];
            un[1] += dtp * (double)(-divB * pp[5]);
            un[2] += dtp * (double)(-divB * pp[6]);
            un[3] += dtp * (double)(-divB * pp[7]);
            un[4] += dtp * (double)(-divB * (pp[1] * pp[5] + pp[2] * pp[6] + pp[3] * pp[7]));
            un[5] += dtp * (double)(-divB * pp[1]);
            un[6] += dtp * (double)(-divB * pp[2]);
            un[7] += dtp * (double)(-divB * pp[3]);
          }
        }
#pragma unroll
        for (int v = 0; v < NV; v++) {
          if constexpr (S2) a.X[at + v * NINT] = un[v];
          else static_cast<ST *>(a.UPout)[at + v * NINT] = (ST)un[v];
        }
      }
#pragma unroll
      for (int v = 0; v < NV; v++) fzp[v] = fzc[v];
    }
  }
}

// ---------------------------------------------------------------------------
// The end of a step from the state X that the second stage left: artificial
// viscosity (its face neighbours outside the block are the half-step ghosts,
// as in the reference), updatePrims, cooling and the CFL candidate
// (finish_cell).  In-plane neighbours enter rounded to RF, those along z in
// FP64.  L planes per workgroup, the column in registers; the ring of x/y
// ghosts of all L planes is gathered first.
// ---------------------------------------------------------------------------
constexpr int END_PLANES = 4;   // most planes per workgroup

// whether the delta-form MHD kernels leave the end of the step to k_end: with
// viscosity (neighbours) or cooling (its FP64 code, even unexecuted, spills)
inline bool ends_apart(const DevCfg &c) { return c.visc_eta != 0.0 || c.cooling; }

template <int NV, typename RF, typename ST, bool VISC, bool DEL, bool WINDS>
__global__ void __launch_bounds__(256, NV == 8 ? 2 : 3) k_end(FusedArgs a) {
  __shared__ RF ring[VISC ? NV : 1][END_PLANES * 4 * NC];   // [v][plane][side][position]
  __shared__ double sred[4];
  const DevCfg &c = a.c;
  const int tid = threadIdx.x, ti = tid & 15, tj = tid >> 4, i = ti + 1, j = tj + 1;
  int bi, slab;
  item_of(blockIdx.x, a.nblk, a.nslab, bi, slab);
  const int b = a.order[bi];
  WX_EMU_CHECK(b >= 0 && b < a.nblk);
  const int L = NC / a.nslab, k0 = slab * L + 1;
  WX_EMU_CHECK(L <= END_PLANES);
  const int l = c.info[b].level - 1;
  const double dx = c.dx[0][l], dy = c.dx[1][l], dz = c.dx[2][l], dt = a.step->dt;
  const double *Xb = a.X + (size_t)b * NV * NINT;
  const ST *half = static_cast<const ST *>(a.UPin);
  double here[NV], below[NV], dtmin = 1.0e30;
  if constexpr (VISC) {
    for (int t = tid; t < 4 * NC * L; t += 256) {
      const int side = (t >> 4) & 3, aa = (t & 15) + 1, k = k0 + (t >> 6);
      const int gi = side == 0 ? 0 : (side == 1 ? NC + 1 : aa), gj = side == 2 ? 0 : (side == 3 ? NC + 1 : aa);
      double u[NV];
      load_cell<ST, NV, true, DEL, WINDS>(a, half, b, gi, gj, k, u);
#pragma unroll
      for (int v = 0; v < NV; v++) ring[v][t] = (RF)u[v];
    }
    if (k0 == 1) {
      load_cell<ST, NV, true, DEL, WINDS>(a, half, b, i, j, 0, below);
    } else {
#pragma unroll
      for (int v = 0; v < NV; v++) below[v] = Xb[v * NINT + lin(i, j, k0 - 1)];
    }
  }
#pragma unroll
  for (int v = 0; v < NV; v++) here[v] = Xb[v * NINT + lin(i, j, k0)];
  if constexpr (VISC) __syncthreads();
  for (int k = k0; k < k0 + L; k++) {
    double u[NV], above[NV];
    if constexpr (VISC) {
      if (k == NC) {
        load_cell<ST, NV, true, DEL, WINDS>(a, half, b, i, j, NC + 1, above);
      } else {
#pragma unroll
        for (int v = 0; v < NV; v++) above[v] = Xb[v * NINT + lin(i, j, k + 1)];
      }
      // Both candidates of every neighbour are loaded, then one is chosen (at
      // the sides the cell itself stands in for the one outside): a load under a
      // condition is waited for at its join, 4 NV times a plane (1728 hydro
      // blocks 678 -> 615 us a step, 64 viscous HLLD blocks 107.5 -> 101.8).
      const int r = (k - k0) * 4 * NC;
      const bool re = ti == NC - 1, le = ti == 0, be = tj == NC - 1, fe = tj == 0;
      const double *x0 = Xb + lin(i, j, k);
      const double *xr = x0 + (re ? 0 : 1), *xl = x0 - (le ? 0 : 1), *xb = x0 + (be ? 0 : NC), *xf = x0 - (fe ? 0 : NC);
#pragma unroll
      for (int v = 0; v < NV; v++) {
        const double gr = xr[v * NINT], gl = xl[v * NINT], gb = xb[v * NINT], gf = xf[v * NINT];
        const RF rr = ring[v][r + NC + tj], rl = ring[v][r + tj], rb = ring[v][r + 3 * NC + ti],
                 rf = ring[v][r + 2 * NC + ti];
        const RF xp = re ? rr : (RF)gr, xm = le ? rl : (RF)gl, yp = be ? rb : (RF)gb, ym = fe ? rf : (RF)gf;
        const double lap = (double)xp + (double)xm + (double)yp + (double)ym + below[v] + above[v] - 6.0 * here[v];
        u[v] = here[v] + c.visc_eta * lap;
      }
    } else {
#pragma unroll
      for (int v = 0; v < NV; v++) {
        u[v] = here[v];
        if (k + 1 < k0 + L) above[v] = Xb[v * NINT + lin(i, j, k + 1)];
      }
    }
#pragma unroll
    for (int v = 0; v < NV; v++) {
      below[v] = here[v];
      here[v] = above[v];
    }
    finish_cell<NV, RF>(a, b, i, j, k, dt, u, dx, dy, dz, dtmin);
  }
  // exact min: wavefront shuffles, then one 64-bit atomic per workgroup on
  // the bit pattern (positive doubles order like their bits), spread over the
  // slots that the next step's first kernel folds
  for (int off = 32; off > 0; off >>= 1) dtmin = fmin(dtmin, __shfl_xor(dtmin, off));
  if ((tid & 63) == 0) sred[tid >> 6] = dtmin;
  __syncthreads();
  if (tid == 0) {
    const double m = fmin(fmin(sred[0], sred[1]), fmin(sred[2], sred[3]));
    atomicMin(&a.slots[(blockIdx.x % DT_SLOTS) * DT_STRIDE], (unsigned long long)__double_as_longlong(m));
  }
}

}  // namespace wx
