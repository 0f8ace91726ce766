"""Launch-shape autotuner for the fused form.

Tunes, per workload (mesh size, variable count, solver), the choices the
fused stage kernels leave open:
  - grid: one workgroup per block, or a persistent grid of k x 256
    workgroups (256 CUs) striding over the block list;
  - block order: along the Morton or the Hilbert curve, as one range or as
    8 ranges mapped to XCDs (workgroup w runs on XCD w % 8, so each XCD's L2
    serves its own halo reads);
  - sub-block tiling of the FP32 MHD kernels: z slabs per block, one
    workgroup each, by the mesh size (the library's own rule) or a fixed
    count.  Every other kernel takes its slabs by the mesh size.
Each candidate runs a few timed steps (HIP events inside wx_run) on the live
state; the state advances, so tune on a scratch context.
"""
from __future__ import annotations

import itertools
import time

NUM_CUS = 256


def slab_choices(solver):
    """Fixed z-slab counts worth a measurement beside the library's rule: in
    the FP32 MHD form 1, 2, 4 and 8, with viscosity whole blocks only."""
    from walicxe3d_amd import hip
    w = solver.w
    if solver.form != hip.FUSED_FP32 or w.nv != 8 or w.visc_eta != 0.0:
        return (1,)
    return (1, 2, 4, 8)


def slab_counts(solver):
    """What tune() tries: 0, slabs by the mesh size, always; fixed counts
    only where the kernels take them (FP32 MHD)."""
    from walicxe3d_amd import hip
    if solver.form != hip.FUSED_FP32 or solver.w.nv != 8:
        return (0,)
    return (0,) + slab_choices(solver)


def candidates(nblk, slabs=(1,)):
    """(grid, xcd_map, curve, nslab) to try; nslab 0: by the mesh size, whose
    work items are at least the blocks."""
    out = []
    for nslab in slabs:
        items = nblk * max(nslab, 1)
        grids = [0] + [k * NUM_CUS for k in (2, 4, 8) if k * NUM_CUS < items]
        out += [(g, x, c, nslab) for g, x, c in itertools.product(grids, (1, 0), (0, 1))]
    return out


CONFIRM = 4   # candidates measured a second time, with 4x the steps


def tune(solver, steps=3, verbose=False):
    """Try every candidate on `solver` (a hip.Walicxe3D in a fused form),
    then the CONFIRM fastest again with 4x the steps; returns (best, table)
    with best = {"grid": g, "xcd_map": x, "curve": c (0 Morton, 1 Hilbert),
    "nslab": s (0 by the mesh size), "ms": t, "ms_confirm": t2}, chosen by ms_confirm."""
    table = []
    for grid, xcd, curve, nslab in candidates(solver.nblk, slab_counts(solver)):
        solver.set_tuning(0, grid)
        solver.set_tuning(1, xcd)
        solver.set_tuning(2, curve)
        solver.set_tuning(4, nslab)
        solver.run(1)                      # graph capture, warm caches
        t0 = time.perf_counter()
        solver.run(steps)
        ms = 1e3 * (time.perf_counter() - t0) / steps
        table.append({"grid": grid, "xcd_map": xcd, "curve": curve, "nslab": nslab, "ms": ms})
        if verbose:
            print("  grid %5d xcd %d curve %d slabs %d: %.3f ms/step" % (grid, xcd, curve, nslab, ms), flush=True)
    # the fastest few again, with more steps each: one short measurement
    # does not separate choices that differ by less than its own noise
    top = sorted(table, key=lambda r: r["ms"])[:CONFIRM]
    for r in top:
        solver.set_tuning(0, r["grid"])
        solver.set_tuning(1, r["xcd_map"])
        solver.set_tuning(2, r["curve"])
        solver.set_tuning(4, r["nslab"])
        solver.run(1)
        t0 = time.perf_counter()
        solver.run(4 * steps)
        r["ms_confirm"] = 1e3 * (time.perf_counter() - t0) / (4 * steps)
    best = min(top, key=lambda r: r["ms_confirm"])
    solver.set_tuning(0, best["grid"])
    solver.set_tuning(1, best["xcd_map"])
    solver.set_tuning(2, best["curve"])
    solver.set_tuning(4, best["nslab"])
    return best, table
