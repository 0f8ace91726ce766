"""The plain form's step runs kernels of its own (ghosts with their
primitives, fluxes with the update, the end of the step in one pass); the
single routines of the C ABI run one kernel each.  Both are the reference's
arithmetic, so every stored array - interior and face ghosts of U, UP and PRIM
- has to come out the same bit for bit."""
import dataclasses

import numpy as np
import pytest

from conftest import ic_in_order
from walicxe3d_amd import hip
from walicxe3d_amd import workloads as W

pytestmark = pytest.mark.gpu


def _by_routine(s, w, steps):
    time = 0.0
    for it in range(1, steps + 1):
        dt = s.getTimestep() * 2.0 ** -(11 - it)
        first = w.solver == "hll1"
        s.boundary(1, hip.U)
        s.calcPrimsAll(hip.U, hip.CELLS_GHOST)
        s.fluxes_update(1, dt if first else dt / 2.0)
        if not first:
            s.boundary(2, hip.UP)
            s.calcPrimsAll(hip.UP, hip.CELLS_ALL)
            s.fluxes_update(2, dt)
        s.doViscousStep()
        s.updatePrims()
        s.cooling(dt)
        time += dt
    return time


# every stored-variable count, AMR faces of each kind, walls, both kinds of
# source, cooling with each temperature rule, the first-order scheme
@pytest.mark.parametrize("name", ["amr_small", "blast_reflect_passive", "mhd_hlle", "winds4", "plane_wind",
                                  "amr_small_hrate", "sedov_hll1", "ot64_gravity", "ot64_amr", "two_passives"])
def test_step_equals_the_single_routines(name):
    w = W.get("amr_small_passive" if name == "two_passives" else name)
    if name == "two_passives":
        w = dataclasses.replace(w, npassive=2)
    bids = np.asarray(w.blocks(), dtype=np.int32)
    U0 = ic_in_order(w, bids)
    a = hip.Walicxe3D(w, form=hip.PLAIN_FP64, bids=bids)
    b = hip.Walicxe3D(w, form=hip.PLAIN_FP64, bids=bids)
    a.upload(U0)
    b.upload(U0)
    a.run(2)
    a.step()
    t = _by_routine(b, w, 3)
    assert a.time.value == t and a.it.value == 3
    for which, what in ((0, "U"), (1, "UP"), (2, "PRIM")):
        x, y = a.raw(which), b.raw(which)
        assert np.array_equal(x, y, equal_nan=True), what
        # edge and corner ghosts are not stored
        assert not x[:, :, :2, :2, :].any() and not x[:, :, :, -2:, -2:].any()
    a.close()
    b.close()


# 8 to 1024 blocks: 1, 2, 4 and 8 planes per workgroup of the update
@pytest.mark.parametrize("nroot", [(1, 1, 1), (8, 2, 1), (16, 2, 1), (16, 4, 1), (16, 8, 1)])
def test_slab_counts_equal_the_fused_fp64_form(nroot):
    w = dataclasses.replace(W.get("ot64"), nroot=nroot, maxlev=2, base_level=2, phys=tuple(float(n) for n in nroot))
    bids = np.asarray(w.blocks(), dtype=np.int32)
    U0 = ic_in_order(w, bids)
    out = []
    for form in (hip.PLAIN_FP64, hip.FUSED_FP64):
        s = hip.Walicxe3D(w, form=form, bids=bids)
        s.upload(U0)
        s.run(2)
        out.append(s.download(prim=False))
        s.close()
    assert np.array_equal(out[0], out[1])
