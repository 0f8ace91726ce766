// wx_mhd_kern.h - the stage kernel of the FP32 MHD form (HLLD, HLLE).
//
// Same block-per-workgroup structure as k_stage (wx_fused_kern.h): thread
// (i, j) owns a z-column and marches k; the column's cells sit in a
// register window, the plane k and its x/y face halo in LDS (the second
// stage, short of registers, keeps plane k only there).  The
// arithmetic is split so that FP32 rounding never touches an O(1) part of
// a face flux:
//   - primitives of every cell in FP64 (from the FP64 state, or in the
//     second stage from U^n plus the FP32 half-step increment);
//   - MUSCL slopes in FP32 from FP64 differences, face states in FP64;
//   - face flux = FP64 physical flux of the upwind state + the Riemann
//     correction in FP32 from jump-sized quantities (wx_delta.h), stored to
//     LDS in FP64;
//   - U + dt * (flux differences + Powell source) accumulated in FP64.
// Faces near the degenerate HLLD star state take the plain FP32 HLLD
// (wx_delta.h).
// Stage 1 writes the half-step state as FP32 increments over U^n; stage 2
// reads U^n of neighbour blocks for its halo and so writes U^{n+1} into the
// second state buffer (the two swap roles every step).
//
// Bound: memory and VALU issue alike, at the 2 waves per SIMD that 256 VGPRs
// and 67 KB of LDS leave: of the 1.29 ms of the second stage on 4096 HLLD blocks
// 0.89 are VALU issue, and its 5.3 GB read and 1.1 written are 5.0 TB/s (reads
// alone reach 5.9 on this card, a copy 4.75).  The x/y halo used to ask for its source cell in every
// plane, between two barriers; now the sources are found once per block
// (HaloRef, ColRef), the loads of the next plane are issued before the last
// barrier of this one, two barriers a plane remain of three, the waves take
// turns with the 32 outer faces, and the window fills in one go: 4096 HLLD
// blocks 2.54 -> 2.23 ms a step, HLLE 2.21 -> 1.98 ms, 64 HLLD blocks 66.5 -> 65.5 us.
// With viscosity or cooling the second stage leaves its state to k_end (TO_X):
// inside, that code held one workgroup per CU (82 KB of LDS) and spilled.
// 8 viscous HLLE blocks, whole blocks -> 16 slabs: first stage 81 -> 10 us,
// second 275 -> 22 + 7 us.
#pragma once

#include "wx_delta.h"
#include "wx_fused_kern.h"
#include "wx_hydro_kern.h"

namespace wx {

// FP64 primitives of one cell (flow2prim, source/hydro_core.f90:323-378,
// with its floors).  Every operation is written out (no contraction), so
// the two blocks that share a face derive the same values from a cell.
__device__ __forceinline__ void prims64(double icv, const double *u, double *w) {
#pragma clang fp contract(off)
  const double rho = u[0];
  // density reciprocal: hardware FP32 reciprocal and one Newton step
  double r = (double)rcp32((float)rho);
  r = __builtin_fma(r, __builtin_fma(-rho, r, 1.0), r);
  const double v1 = u[1] * r, v2 = u[2] * r, v3 = u[3] * r;
  const double ke = 0.5 * __builtin_fma(u[3], v3, __builtin_fma(u[2], v2, u[1] * v1));
  const double me = 0.5 * __builtin_fma(u[7], u[7], __builtin_fma(u[6], u[6], u[5] * u[5]));
  const double p = (u[4] - ke - me) * icv;
  w[0] = rho < 1.0e-40 ? 1.0e-40 : rho;
  w[1] = v1;
  w[2] = v2;
  w[3] = v3;
  w[4] = p < 1.0e-30 ? 1.0e-30 : p;
  w[5] = u[5];
  w[6] = u[6];
  w[7] = u[7];
}

// MUSCL face values of one variable (limiter, source/hydro_core.f90:613-697)
// from FP64 cell values: the slopes in FP32 (FP64 differences rounded), the
// face values cell +- slope / 2 in FP64
template <int LIM>
__device__ __forceinline__ void rec64(const Phys<float> &P, double xll, double xl, double xr, double xrr, double &l,
                                      double &r) {
  const float dl = (float)(xl - xll), dm = (float)(xr - xl), dr = (float)(xrr - xr);
  float al, ar;
  if constexpr (LIM == 1) {
    al = minmod32(dl, dm);
    ar = minmod32(dm, dr);
  } else {
    const int lim = LIM == LIM_RUNTIME ? P.limiter : LIM;
    al = average(dl, dm, lim);
    ar = average(dm, dr, lim);
  }
  l = xl + 0.5 * (double)al;
  r = xr - 0.5 * (double)ar;
}

// Exchange of the x components of velocity and field with those along D
// (swapxy / swapxz, source/hydro_core.f90:448-496)
template <int D> __device__ __forceinline__ void rot8(double *v) {
  if constexpr (D != 0) {
    double t = v[1];
    v[1] = v[1 + D];
    v[1 + D] = t;
    t = v[5];
    v[5] = v[5 + D];
    v[5 + D] = t;
  }
}

// rot8<1> where d holds (the y direction), per lane: selects, no branch
__device__ __forceinline__ void rot8_if(bool d, double *v) {
  const double v1 = v[1], v2 = v[2], v5 = v[5], v6 = v[6];
  v[1] = d ? v2 : v1;
  v[2] = d ? v1 : v2;
  v[5] = d ? v6 : v5;
  v[6] = d ? v5 : v6;
}

// Flux across one face along D from its two face states (unrotated) in the
// delta form of wx_delta.h; a face near the degenerate HLLD star state
// takes the one-code-path HLLD in FP32 (hlld_flux_ill)
template <int D, int SOLVER>
__device__ __forceinline__ void face_flux(const DevCfg &c, double *wl, double *wr, double *F) {
  rot8<D>(wl);
  rot8<D>(wr);
  if constexpr (SOLVER == SOLVER_HLLD) {
    if (!hlld_flux_delta(c.pd, c.pf, wl, wr, F)) hlld_flux_ill(c.pf, wl, wr, F);
  } else {
    hlle_flux_delta(c.pd, c.pf, wl, wr, F);
  }
  rot8<D>(F);
}

#ifndef WX_MHD_MIN_WAVES
#define WX_MHD_MIN_WAVES 2
#endif

template <bool S2, bool TO_X, int SOLVER, int LIM, bool WIND>
__global__ void __launch_bounds__(256, WX_MHD_MIN_WAVES) k_mhd(FusedArgs a) {
  constexpr int NV = 8;
  constexpr int H = S2 ? 2 : 1;            // halo depth of the stencil
  constexpr int W = NC + 2 * H;
  constexpr int WPD = W | 1;               // LDS row pitch (FP64 elements)
  constexpr int NW = S2 ? 4 : 3;           // planes in the column window
  constexpr int NXF = (NC + 1) * NC;       // x (or y) faces of a plane
  __shared__ double sw[NV][W * WPD];       // FP64 primitives of plane k (cross region)
  __shared__ double sfx[NV][NXF];          // x fluxes [v][row * 17 + s]
  __shared__ double sfy[NV][NXF];          // y fluxes [v][col * 17 + s]
  __shared__ double sred[4];
  __shared__ HaloRef sref[4 * H * NC];     // sources of the x/y halo of lanes tid < 4 H 16
  __shared__ ColRef scol[2][256];          // and of the column's ghosts; each read back by its lane

  const DevCfg &c = a.c;
  const Phys<float> &P = c.pf;
  const float *UPin = static_cast<const float *>(a.UPin);
  float *UPout = static_cast<float *>(a.UPout);
  const int tid = threadIdx.x;
  const int ti = tid & 15, tj = tid >> 4;
  const int i = ti + 1, j = tj + 1;
  const double dt = uni(a.step->dt);
  const double dtp = S2 ? dt : dt / 2.0;
  const double icv = uni(1.0 / c.pd.cv);
  double dtmin = 1.0e30;

  // x/y face halo of a plane, H layers on each of the 4 sides: lanes
  // tid < NH load one cell each.
  constexpr int NH = 4 * H * NC;
  // second stage: plane k of the column window lives in this lane's slot of
  // sw (where the x/y faces read it) rather than in registers, from the
  // point where it is stored until it is read back as plane k-1
  constexpr bool LW = S2;
  const int own = (j - 1 + H) * WPD + (i - 1 + H);
  // Loads one plane ahead, except where they push over 40 VGPRs out: with wind
  // code (8 viscous blocks 54.1 against 51.7 us a step) and in the HLLE second
  // stage (64 blocks 60 against 57.7 us, though 4096 blocks 1.94 against 1.98 ms)
  constexpr bool PIPE = !WIND && !(S2 && SOLVER == SOLVER_HLLE);
  const bool hth = tid < NH;
  // halo cell (hi, hj) of lane tid, layer g
  auto halo_cell = [&](int &hi, int &hj, int &g) {
    const int part = tid / (2 * H * NC);
    const int r = tid % (2 * H * NC);
    const int side = r / (H * NC);
    g = (r % (H * NC)) / NC + 1;
    const int aa = r % NC + 1;
    if (part == 0) { hi = side ? NC + g : 1 - g; hj = aa; }
    else { hj = side ? NC + g : 1 - g; hi = aa; }
  };

  // Work items: block bi of the order list, z slab of it (planes slab L + 1 ..
  // (slab + 1) L, L = NC / nslab).  A slab starts one plane early, at its
  // bottom z face, which the slab below computes too, with the same code and
  // inputs.
  const int nslab = uni(a.nslab);
  WX_EMU_CHECK(nslab >= 1 && NC % nslab == 0);
  const int L = NC / nslab;
  for (int item = blockIdx.x; item < a.nblk * nslab; item += gridDim.x) {
    int bi, slab;
    item_of(item, a.nblk, nslab, bi, slab);
    const int k0 = slab * L + 1, k1 = k0 + L - 1;
    // block, level and per-block constants are the same in every lane:
    // scalar registers
    const int b = uni(a.order[bi]);
    WX_EMU_CHECK(b >= 0 && b < a.nblk);
    const int l = uni(c.info[b].level - 1);
    const double dxl = c.dx[0][l], dyl = c.dx[1][l], dzl = c.dx[2][l];
    const double dtdx = uni(dtp / dxl), dtdy = uni(dtp / dyl), dtdz = uni(dtp / dzl);
    const double idx2 = uni(1.0 / (2.0 * dxl)), idy2 = uni(1.0 / (2.0 * dyl)), idz2 = uni(1.0 / (2.0 * dzl));

    const bool winds = WIND && a.c.nwind > 0;
    if (k0 - H < 1) scol[0][tid] = col_ref(a, b, BOTTOM, i, j);
    if (k1 + H > NC) scol[1][tid] = col_ref(a, b, TOP, i, j);
    if (hth) {
      int hi, hj, hg;
      halo_cell(hi, hj, hg);
      sref[tid] = halo_ref<true>(a, b, hi, hj);
    }
    // element 0 of the column's cell in plane kn; false: that takes load_cell
    auto col_at = [&](int kn, size_t &at) -> bool {
      WX_EMU_CHECK(kn >= k0 - H && kn <= k1 + H);
      if (winds) return false;
      const bool own = kn >= 1 && kn <= NC;
      int blk = b, cell = 0;
      if (own) cell = lin(i, j, kn);
      else {
        const ColRef r = scol[kn < 1 ? 0 : 1][tid];
        blk = uni(r.blk);
        cell = r.at(kn < 1 ? 1 - kn : kn - NC);
      }
      at = (size_t)blk * NV * NINT + cell;
      return blk >= 0;
    };
    // column window of FP64 primitives: at iteration k (after the shift)
    // S2: planes {k-1, k, k+1, k+2};  S1: planes {k-1, k, k+1}
    double wq[NW][NV];
    double fzp[NV];                        // z flux (k-1 | k)
#pragma unroll
    for (int w = 0; w < NW; w++)
#pragma unroll
      for (int v = 0; v < NV; v++) wq[w][v] = 0.0;

    // (a reflective face negates the normal momentum, where the value is used)
    auto col_flip = [&](int kn, double *u) {
      if (kn >= 1 && kn <= NC) return;
      if (!winds && scol[kn < 1 ? 0 : 1][tid].flip()) u[3] = -u[3];
    };

    // Loads of iteration kl: plane kl + NW - 2 of the column and plane kl of
    // the halo, with PIPE issued while iteration kl - 1 works.  In the second stage the
    // FP32 increments wait beside the state and are added where it is used
    // (-0 where the state is whole: it leaves every bit of a sum).
    double ucol[NV], uh[NV];
    float dcol[NV], dh[NV];
#pragma unroll
    for (int v = 0; v < NV; v++) { ucol[v] = uh[v] = 1.0; dcol[v] = dh[v] = -0.0f; }
    auto fetch = [&](int kl) {
      // (nothing of the consumed values stays alive)
#pragma unroll
      for (int v = 0; v < NV; v++) { ucol[v] = uh[v] = 1.0; dcol[v] = dh[v] = -0.0f; }
      if (kl > k1) return;
      const int kn = S2 ? kl + 2 : kl + 1;
      size_t at;
      if (col_at(kn, at)) {
#pragma unroll
        for (int v = 0; v < NV; v++) ucol[v] = a.U[at + v * NINT];
        if constexpr (S2)
#pragma unroll
          for (int v = 0; v < NV; v++) dcol[v] = UPin[at + v * NINT];
      } else {
        if constexpr (S2) load_cell<float, NV, true, true, WIND>(a, UPin, b, i, j, kn, ucol);
        else load_cell<double, NV, false, false, WIND>(a, a.U, b, i, j, kn, ucol);
        if constexpr (S2)
#pragma unroll
          for (int v = 0; v < NV; v++) dcol[v] = -0.0f;
      }
      if (hth && kl >= k0) {
        int hi, hj, hg;
        halo_cell(hi, hj, hg);
        const HaloRef href = sref[tid];
        if (href.blk >= 0) {
          const size_t at = (size_t)href.blk * NV * NINT + href.at(kl);
#pragma unroll
          for (int v = 0; v < NV; v++) uh[v] = a.U[at + v * NINT];
          if constexpr (S2)
#pragma unroll
            for (int v = 0; v < NV; v++) dh[v] = UPin[at + v * NINT];
        } else {
          if constexpr (S2) load_cell<float, NV, true, true, false>(a, UPin, b, hi, hj, kl, uh);
          else load_cell<double, NV, false, false, false>(a, a.U, b, hi, hj, kl, uh);
          if constexpr (S2)
#pragma unroll
            for (int v = 0; v < NV; v++) dh[v] = -0.0f;
        }
        if constexpr (WIND) {
          double w[MAXV];
          if (a.c.nwind > 0 && wind_state(a.c, b, hi, hj, kl, w)) {
#pragma unroll
            for (int v = 0; v < NV; v++) uh[v] = w[v];
            if (href.flip() == 1) uh[1] = -uh[1];   // negated again where it is used
            if (href.flip() == 2) uh[2] = -uh[2];
            if constexpr (S2)
#pragma unroll
              for (int v = 0; v < NV; v++) dh[v] = -0.0f;
          }
        }
      }
    };

    // The window's first planes (S2: k0-2 .. k0 and the loads of k0+1; S1:
    // k0-1 and the loads of k0) all at once, if none of them needs load_cell;
    // otherwise the first iterations fill it, one plane each (with PIPE the
    // very first only issues loads), so that one call site of load_cell serves
    // every plane: the kernel's code stays small.
    constexpr int BACK0 = (S2 ? 4 : 2) + PIPE;
    int kf = k0 - BACK0;
    {
      size_t at[S2 ? 4 : 2];
      bool all = true;
#pragma unroll
      for (int w = 0; w < (S2 ? 4 : 2); w++) all = col_at(k0 - H + w, at[w]) && all;
      if (all) {
        constexpr int NF = S2 ? 3 : 1;
        double uf[NF][NV];
        float df[NF][NV];
#pragma unroll
        for (int w = 0; w < NF; w++)
#pragma unroll
          for (int v = 0; v < NV; v++) {
            uf[w][v] = a.U[at[w] + v * NINT];
            if constexpr (S2) df[w][v] = UPin[at[w] + v * NINT];
          }
        if constexpr (PIPE)
#pragma unroll
          for (int v = 0; v < NV; v++) {
            ucol[v] = a.U[at[NF] + v * NINT];
            if constexpr (S2) dcol[v] = UPin[at[NF] + v * NINT];
          }
#pragma unroll
        for (int w = 0; w < NF; w++) {
          if constexpr (S2)
#pragma unroll
            for (int v = 0; v < NV; v++) uf[w][v] = uf[w][v] + (double)df[w][v];
          col_flip(k0 - H + w, uf[w]);
          prims64(icv, uf[w], wq[NW - NF + w]);
        }
        if constexpr (LW)
#pragma unroll
          for (int v = 0; v < NV; v++) sw[v][own] = wq[1][v];
        kf = k0 - 1;
      }
    }
    for (int k = kf; k <= k1; k++) {
      if constexpr (!PIPE) fetch(k);
      if constexpr (LW) {
        // plane k-1 from this lane's slot of the plane store, where the
        // previous iteration left it
#pragma unroll
        for (int v = 0; v < NV; v++) wq[0][v] = sw[v][own];
#pragma unroll
        for (int w = 1; w < NW - 1; w++)
#pragma unroll
          for (int v = 0; v < NV; v++) wq[w][v] = wq[w + 1][v];
      } else {
#pragma unroll
        for (int w = 0; w < NW - 1; w++)
#pragma unroll
          for (int v = 0; v < NV; v++) wq[w][v] = wq[w + 1][v];
      }
      if constexpr (S2)
#pragma unroll
        for (int v = 0; v < NV; v++) ucol[v] = ucol[v] + (double)dcol[v];
      if (!PIPE || k > k0 - BACK0) col_flip(k + NW - 2, ucol);
      prims64(icv, ucol, wq[NW - 1]);
      // own primitives of plane k and, by the halo lanes, its face halo into
      // LDS: the previous plane's readers were done at the last barrier
      if (LW || k >= k0)
#pragma unroll
        for (int v = 0; v < NV; v++) sw[v][own] = wq[1][v];
      if (hth && k >= k0) {
        int hi, hj, hg;
        halo_cell(hi, hj, hg);
        double wh[NV];
        if constexpr (S2)
#pragma unroll
          for (int v = 0; v < NV; v++) uh[v] = uh[v] + (double)dh[v];
        if (sref[tid].flip() == 1) uh[1] = -uh[1];
        if (sref[tid].flip() == 2) uh[2] = -uh[2];
        prims64(icv, uh, wh);
#pragma unroll
        for (int v = 0; v < NV; v++) sw[v][(hj - 1 + H) * WPD + (hi - 1 + H)] = wh[v];
      }
      // z flux (k | k+1): one code path for every plane, the bottom face included
      double fzc[NV];
      if (k >= k0 - 1) {
        double wl[NV], wr[NV];
#pragma unroll
        for (int v = 0; v < NV; v++) {
          if constexpr (S2) rec64<LIM>(P, wq[0][v], wq[1][v], wq[2][v], wq[3][v], wl[v], wr[v]);
          else { wl[v] = wq[1][v]; wr[v] = wq[2][v]; }
        }
        face_flux<2, SOLVER>(c, wl, wr, fzc);
      }
      if (k < k0) {
#pragma unroll
        for (int v = 0; v < NV; v++) fzp[v] = fzc[v];
        if constexpr (PIPE) fetch(k + 1);
        continue;
      }
      __syncthreads();
      // x faces s = 0..15 of plane k, one per lane (row tj, face ti)
      {
        const int base = (tj + H) * WPD + (ti - 1 + H);       // cell s = ti
        double wl[NV], wr[NV], ff[NV];
#pragma unroll
        for (int v = 0; v < NV; v++) {
          const double *x = &sw[v][base];
          if constexpr (S2) rec64<LIM>(P, x[-1], x[0], x[1], x[2], wl[v], wr[v]);
          else { wl[v] = x[0]; wr[v] = x[1]; }
        }
        face_flux<0, SOLVER>(c, wl, wr, ff);
#pragma unroll
        for (int v = 0; v < NV; v++) sfx[v][tj * (NC + 1) + ti] = ff[v];
      }
      // y faces s = 0..15, one per lane
      {
        const int t = (tid + 192) & 255;
        const int sy = t & 15, col = t >> 4;
        const int base = (sy - 1 + H) * WPD + (col + H);      // cell s
        double wl[NV], wr[NV], ff[NV];
#pragma unroll
        for (int v = 0; v < NV; v++) {
          const double *x = &sw[v][base];
          if constexpr (S2) rec64<LIM>(P, x[-WPD], x[0], x[WPD], x[2 * WPD], wl[v], wr[v]);
          else { wl[v] = x[0]; wr[v] = x[WPD]; }
        }
        face_flux<1, SOLVER>(c, wl, wr, ff);
#pragma unroll
        for (int v = 0; v < NV; v++) sfy[v][col * (NC + 1) + sy] = ff[v];
      }
      // the 16 x and the 16 y faces s = 16 together on 32 lanes of one wave (x
      // on the first 16, y on the others): one solve per lane, the states
      // rotated by lane (selects) into the x-aligned order of face_flux<0>.
      // The waves take turns, plane by plane: they sit on different SIMDs.
      const int e = tid - 64 * (k & 3);
      if ((unsigned)e < 2 * NC) {
        const bool d = e >= NC;                                // y face
        const int aa = d ? e - NC : e;                         // row or column
        const int st = d ? WPD : 1;
        const int base = d ? (NC - 1 + H) * WPD + (aa + H) : (aa + H) * WPD + (NC - 1 + H);
        double wl[NV], wr[NV], ff[NV];
#pragma unroll
        for (int v = 0; v < NV; v++) {
          const double *x = &sw[v][base];
          if constexpr (S2) rec64<LIM>(P, x[-st], x[0], x[st], x[2 * st], wl[v], wr[v]);
          else { wl[v] = x[0]; wr[v] = x[st]; }
        }
        rot8_if(d, wl);
        rot8_if(d, wr);
        face_flux<0, SOLVER>(c, wl, wr, ff);
        rot8_if(d, ff);
#pragma unroll
        for (int v = 0; v < NV; v++) (d ? sfy[v] : sfx[v])[aa * (NC + 1) + NC] = ff[v];
      }
      const double *Ub = a.U + (size_t)b * NV * NINT + lin(i, j, k);
      double ub[NV];
#pragma unroll
      for (int v = 0; v < NV; v++) ub[v] = Ub[v * NINT];
      double divB = 0.0;
      if (c.eight_wave)
        divB = (sw[5][own + 1] - sw[5][own - 1]) * idx2 + (sw[6][own + WPD] - sw[6][own - WPD]) * idy2 +
               (wq[2][7] - wq[0][7]) * idz2;
      if constexpr (PIPE) fetch(k + 1);
      __syncthreads();
      // conservative update of cell (i, j, k) in FP64
      double unew[NV];
      {
        // base of the update: U^n, or the wind state in a cell that a source
        // covers (each stage's boundary() imposes the sources through
        // userBoundary: source/godunov.f90:79,141, source/boundary.f90:61)
        double u0[NV];
#pragma unroll
        for (int v = 0; v < NV; v++) u0[v] = ub[v];
        if constexpr (WIND) {
          double w[MAXV];
          if (c.nwind > 0 && wind_state(c, b, i, j, k, w))
#pragma unroll
            for (int v = 0; v < NV; v++) u0[v] = w[v];
        }
#pragma unroll
        for (int v = 0; v < NV; v++)
          unew[v] = u0[v] + dtdx * (sfx[v][tj * (NC + 1) + ti] - sfx[v][tj * (NC + 1) + ti + 1]) +
                    dtdy * (sfy[v][ti * (NC + 1) + tj] - sfy[v][ti * (NC + 1) + tj + 1]) +
                    dtdz * (fzp[v] - fzc[v]);
        if (c.eight_wave) {
          // Powell source (source/sources.f90:38-95) from the stage primitives
          double ppl[NV];
          const double *pp = wq[1];
          if constexpr (LW) {
#pragma unroll
            for (int v = 0; v < NV; v++) ppl[v] = sw[v][own];
            pp = ppl;
          }
          unew[1] += dtp * (-divB * pp[5]);
          unew[2] += dtp * (-divB * pp[6]);
          unew[3] += dtp * (-divB * pp[7]);
          unew[4] += dtp * (-divB * (pp[1] * pp[5] + pp[2] * pp[6] + pp[3] * pp[7]));
          unew[5] += dtp * (-divB * pp[1]);
          unew[6] += dtp * (-divB * pp[2]);
          unew[7] += dtp * (-divB * pp[3]);
        }
        if constexpr (!S2) {
          // the half-step state as FP32 increments over U^n
          float *UPo = UPout + (size_t)b * NV * NINT + lin(i, j, k);
#pragma unroll
          for (int v = 0; v < NV; v++) UPo[v * NINT] = (float)(unew[v] - ub[v]);   // over the stored U^n
        }
      }
#pragma unroll
      for (int v = 0; v < NV; v++) fzp[v] = fzc[v];
      if constexpr (!S2) continue;

      // stage 2: the state for k_end, or the end of the step here
      if constexpr (TO_X) {
        double *Xo = a.X + (size_t)b * NV * NINT + lin(i, j, k);
#pragma unroll
        for (int v = 0; v < NV; v++) Xo[v * NINT] = unew[v];
      } else {
        finish_cell32<NV, false>(a, b, i, j, k, unew, dxl, dyl, dzl, dtmin);
      }
    }
    __syncthreads();
  }
  if constexpr (S2 && !TO_X) {
    // exact min: wavefront shuffles, then one 64-bit atomic per workgroup on
    // the bit pattern (positive doubles order like their bits)
    for (int off = 32; off > 0; off >>= 1) dtmin = fmin(dtmin, __shfl_xor(dtmin, off));
    if ((tid & 63) == 0) sred[tid >> 6] = dtmin;
    __syncthreads();
    if (tid == 0) {
      double m = fmin(fmin(sred[0], sred[1]), fmin(sred[2], sred[3]));
      atomicMin(&a.slots[(blockIdx.x % DT_SLOTS) * DT_STRIDE], (unsigned long long)__double_as_longlong(m));
    }
  }
}

// With viscosity or cooling the second stage leaves its state to k_end (to_x):
// one instance, with the wind code and the limiter read at run time, also for
// meshes without sources and for minmod.  Contraction fuses some sums of xflux
// from one side or the other as the code around them changes, and an instance
// without that code rounded them the other way; this one keeps the results that
// the kernel with viscosity inside gave.  It spills 13 VGPRs (HLLD; HLLE 5) and
// loads no plane ahead: 1728 viscous HLLD blocks 2.03 ms a step with k_end (1.43
// without viscosity; 3.04 with the viscosity inside), 64 blocks 105 us (451).
template <int SOLVER, bool WIND>
inline void launch_mhd_w(const FusedArgs &a, int grid, bool to_x, int stage, hipStream_t st) {
  constexpr int MM = 1;  // LIMITER_MINMOD (source/constants.f90)
  const bool mm = a.c.pf.limiter == MM && !WIND;
  if (stage == 1)
    hipLaunchKernelGGL((k_mhd<false, false, SOLVER, LIM_RUNTIME, WIND>), dim3(grid), dim3(256), 0, st, a);
  else if (to_x)
    hipLaunchKernelGGL((k_mhd<true, true, SOLVER, LIM_RUNTIME, true>), dim3(grid), dim3(256), 0, st, a);
  else if (mm)
    hipLaunchKernelGGL((k_mhd<true, false, SOLVER, MM, false>), dim3(grid), dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL((k_mhd<true, false, SOLVER, LIM_RUNTIME, WIND>), dim3(grid), dim3(256), 0, st, a);
}

inline void launch_mhd_end(const FusedArgs &a, hipStream_t st) {
  const int grid = a.nblk * a.nslab;
  if (a.c.visc_eta == 0.0)
    hipLaunchKernelGGL((k_end<8, float, float, false, true, false>), dim3(grid), dim3(256), 0, st, a);
  else if (a.c.nwind > 0)
    hipLaunchKernelGGL((k_end<8, float, float, true, true, true>), dim3(grid), dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL((k_end<8, float, float, true, true, false>), dim3(grid), dim3(256), 0, st, a);
}

// meshes with wind sources take the kernels that carry the wind code (every
// limiter at run time); the others leave it out
template <int SOLVER>
inline void launch_mhd(const FusedArgs &a, int grid, int stage, hipStream_t st) {
  const bool to_x = ends_apart(a.c);
  if (a.c.nwind > 0) launch_mhd_w<SOLVER, true>(a, grid, to_x, stage, st);
  else launch_mhd_w<SOLVER, false>(a, grid, to_x, stage, st);
}

}  // namespace wx
