"""The fused hydro kernels in FP64 against the plain form: the same arithmetic
in another order of work (slabs of planes, halos read from the neighbours, the
end of the step in its own kernel), so without viscosity every state is the
same bit for bit.  The viscous sum takes the two z neighbours in the other
order (the column is walked upwards): 2 ulp of a term weighted by 5e-3, so a
cell's last bit changes now and then; 1e-13 of a variable's largest value is
over a hundred such flips per step.  The FP32 form is the same code in another type; its error is bounded in
test_gpu_parity.py."""
import dataclasses

import numpy as np
import pytest

from conftest import ic_in_order
from walicxe3d_amd import hip
from walicxe3d_amd import workloads as W

pytestmark = pytest.mark.gpu


def _both(w, steps):
    bids = np.asarray(w.blocks(), dtype=np.int32)
    U0 = ic_in_order(w, bids)
    out = []
    for form in (hip.PLAIN_FP64, hip.FUSED_FP64):
        s = hip.Walicxe3D(w, form=form, bids=bids)
        s.upload(U0)
        s.run(steps)
        out.append((s.download(prim=False), s.time.value, s.getTimestep()))
        s.close()
    return out


def _same(a, b, exact):
    (ua, ta, da), (ub, tb, db) = a, b
    if exact:
        return np.array_equal(ua, ub) and ta == tb and da == db
    top = np.abs(ua).max(axis=(0, 2, 3, 4))
    off = np.abs(ua - ub).max(axis=(0, 2, 3, 4))
    return np.all(off <= 1e-13 * top.max()) and abs(ta - tb) <= 1e-13 * ta and abs(da - db) <= 1e-13 * da


# walls, open sides, coarse-fine faces, wind sources; limiters fixed and read
# at run time
@pytest.mark.parametrize("name,visc,limiter", [
    ("sedov", 0.0, "minmod"), ("sedov", 0.0, "vanleer"), ("blast_reflect", 0.0, "minmod"), ("amr_small", 0.0, "superbee"),
    ("winds4", 0.0, "umist"), ("snr_amr4", 0.0, "minmod"), ("sedov", 5.0e-3, "minmod"),
    ("blast_reflect", 5.0e-3, "none"), ("amr_small", 5.0e-3, "woodward"), ("winds4", 5.0e-3, "minmod")])
def test_fused_fp64_hydro_equals_the_plain_form(name, visc, limiter):
    # without cooling, after which the plain form keeps the cooled pressure
    # and the fused form recovers it from the energy
    w = dataclasses.replace(W.get(name), visc_eta=visc, limiter=limiter, cooling=False)
    a, b = _both(w, 3)
    assert _same(a, b, visc == 0.0)


# 1 to 1024 blocks, and counts that are no multiple of 8: every slab count of
# the stages (16 to 1) and of the end of the step, and the tail of the dealing
@pytest.mark.parametrize("nroot", [(1, 1, 1), (3, 1, 1), (8, 2, 1), (5, 5, 1), (16, 3, 1), (16, 4, 1), (16, 8, 1)])
@pytest.mark.parametrize("base,visc", [(1, 0.0), (2, 0.0), (1, 5.0e-3), (2, 5.0e-3)])
def test_slab_counts(nroot, base, visc):
    w = dataclasses.replace(W.get("sedov"), nroot=nroot, maxlev=base, base_level=base, visc_eta=visc,
                            phys=tuple(float(n) for n in nroot))
    a, b = _both(w, 2)
    assert _same(a, b, visc == 0.0)
