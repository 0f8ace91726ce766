"""The FP32 MHD kernels' own halo tables: every kind of face (same level,
coarser, finer, open, reflective, periodic) on every side, first and second
stage.  Slab counts 1, 8 and the default (which reach the z ghosts as plane 0,
-1, 17, 18 of different slabs, by the parallel fill and plane by plane) give
the same bits; against the plain FP64 form a wrong or unnegated ghost is off by
the size of the state, the FP32 Riemann corrections by some 1e-7 of it a step:
the bar is the 1e-5 of test_gpu_parity.py, for each of density, momentum,
energy and field."""
import dataclasses

import numpy as np
import pytest

from conftest import ic_in_order
from walicxe3d_amd import hip
from walicxe3d_amd import workloads as W

pytestmark = pytest.mark.gpu

WALLS = ("reflective",) * 6
MIXED = ("reflective", "free", "free", "reflective", "reflective", "free")


@pytest.mark.parametrize("name,solver,bc", [
    ("mhd_hlle", "hlle", WALLS), ("mhd_hlle", "hlld", WALLS), ("mhd_hlle", "hlld", MIXED),
    ("ot64_amr", "hlld", WALLS), ("ot64_amr", "hlle", MIXED), ("ot64_amr", "hlld", None)])
@pytest.mark.parametrize("visc", [0.0, 2.0e-3])
def test_faces_and_slabs(name, solver, bc, visc):
    w = W.get(name)
    w = dataclasses.replace(w, solver=solver, visc_eta=visc, bc=bc or w.bc)
    bids = np.asarray(w.blocks(), dtype=np.int32)
    U0 = ic_in_order(w, bids)

    def go(form, slabs=None):
        s = hip.Walicxe3D(w, form=form, bids=bids)
        if slabs:
            s.set_tuning(4, slabs)
        s.upload(U0)
        s.run(3)
        out = s.download(prim=False)
        s.close()
        return out

    u = go(hip.FUSED_FP32)
    assert all(np.array_equal(u, go(hip.FUSED_FP32, n)) for n in (1, 8))
    r = go(hip.PLAIN_FP64)
    for g in (slice(0, 1), slice(1, 4), slice(4, 5), slice(5, 8)):
        assert np.abs(u[:, g] - r[:, g]).max() <= 1e-5 * np.abs(r[:, g]).max(), g
