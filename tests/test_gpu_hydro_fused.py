"""The fused hydro kernels in FP64 against the plain form: the same arithmetic
in another order of work (slabs of planes, halos read from the neighbours, the
end of the step in its own kernel), so without viscosity every state is the
same bit for bit.  The viscous sum takes the two z neighbours in the other
order (the column is walked upwards): 2 ulp of a term weighted by 5e-3, so a
cell's last bit changes now and then; 1e-13 of a variable's largest value is
over a hundred such flips per step.  The FP32 kernels are the same templates,
but only they keep their halo's sources in tables, checked at the end of this
file; their error is bounded in test_gpu_parity.py."""
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


# 1 to 1024 blocks, and counts that are no multiple of 8: slab counts 16 to 2 of
# the stages (whole blocks: test_whole_blocks) and every one of the end of the
# step, and the tail of the dealing
@pytest.mark.parametrize("nroot", [(1, 1, 1), (3, 1, 1), (8, 2, 1), (5, 5, 1), (16, 3, 1), (16, 4, 1), (16, 8, 1)])
@pytest.mark.parametrize("base,visc", [(1, 0.0), (2, 0.0), (1, 5.0e-3), (2, 5.0e-3)])
def test_slab_counts(nroot, base, visc):
    w = dataclasses.replace(W.get("sedov"), nroot=nroot, maxlev=base, base_level=base, visc_eta=visc,
                            phys=tuple(float(n) for n in nroot))
    a, b = _both(w, 2)
    assert _same(a, b, visc == 0.0)


def _per_variable(a, b):
    """off <= 1e-13 of each variable's own size.  Per cell and step the sums of
    the two forms differ by some ulp of a neighbour weighted by 5e-3 and by one
    rounding, 2e-16 of the largest value; in the next step a last bit of the
    energy moves momenta by sqrt(rho E) of that (dt/dx is about 1/c), which is
    their scale where the gas is at rest.  3 steps stay under 50 ulp, 1e-14;
    a wrong neighbour in the viscous sum moves a variable by 5e-3 of its own
    differences."""
    top = np.abs(b).max(axis=(0, 2, 3, 4))
    rest = np.sqrt(top[0] * top[4])
    speed = np.sqrt((b[:, 1:4] ** 2).sum(axis=1)).max()
    top[1:4] = max(speed, rest)
    off = np.abs(a - b).max(axis=(0, 2, 3, 4))
    assert np.all(off <= 1e-13 * top), off / top


@pytest.mark.parametrize("name,limiter", [("sedov", "minmod"), ("blast_reflect", "none"), ("amr_small", "woodward"),
                                          ("winds4", "minmod"), ("snr_amr4", "vanleer")])
def test_viscous_states_per_variable(name, limiter):
    w = dataclasses.replace(W.get(name), visc_eta=5.0e-3, limiter=limiter, cooling=False)
    a, b = _both(w, 3)
    _per_variable(a[0], b[0])


@pytest.mark.parametrize("visc", [0.0, 5.0e-3])
def test_whole_blocks(visc):
    """From 2048 blocks on a workgroup takes a block's 16 planes."""
    w = dataclasses.replace(W.get("sedov"), nroot=(16, 16, 8), maxlev=1, base_level=1, visc_eta=visc,
                            phys=(16.0, 16.0, 8.0))
    a, b = _both(w, 2)
    if visc:
        _per_variable(a[0], b[0])
    else:
        assert _same(a, b, True)


@pytest.mark.parametrize("solver,limiter,visc", [("hllc", "minmod", 0.0), ("hllc", "superbee", 5.0e-3),
                                                 ("hll", "minmod", 5.0e-3)])
def test_fp32_slab_counts(solver, limiter, visc):
    """A periodic box of 64 blocks, and boxes that repeat it 2 to 32 times: 16,
    16, 8, 4, 2 and 1 slabs a block by the number of blocks, the same numbers
    in every cell, so the same bits in every copy and the same timesteps."""
    w = W.get("sedov")
    rng = np.random.default_rng(8)
    box = rng.uniform(0.9, 1.1, (4, 4, 4, 5, 16, 16, 16))     # blocks z, y, x
    box[..., 1:4, :, :, :] -= 1.0
    box[..., 4, :, :, :] += 4.0
    first = None
    for reps in ((1, 1, 1), (1, 1, 2), (1, 2, 2), (2, 2, 2), (2, 2, 4), (4, 4, 2)):
        nroot = tuple(4 * r for r in reps)
        v = dataclasses.replace(w, solver=solver, limiter=limiter, visc_eta=visc, bc=("periodic",) * 6, nroot=nroot,
                                maxlev=1, base_level=1, phys=tuple(float(n) for n in nroot))
        bids = np.asarray(v.blocks(), dtype=np.int32)
        order = np.argsort(np.argsort(bids))                  # block IDs: x fastest, then y, then z
        U = np.tile(box, tuple(reps[::-1]) + (1, 1, 1, 1)).reshape(-1, 5, 16, 16, 16)[order]
        s = hip.Walicxe3D(v, form=hip.FUSED_FP32, bids=bids)
        s.upload(U)
        s.run(3)
        out = np.empty_like(U)
        out[order] = s.download(prim=False)
        out = out.reshape(nroot[::-1] + (5, 16, 16, 16))
        dt = (s.time.value, s.getTimestep())
        s.close()
        if first is None:
            first = out, dt
            assert not np.array_equal(out, box)
        assert dt == first[1]
        assert np.array_equal(out, np.tile(first[0], tuple(reps[::-1]) + (1, 1, 1, 1))), nroot


@pytest.mark.parametrize("name", ["sedov", "blast_reflect", "amr_small", "snr_amr4"])
@pytest.mark.parametrize("limiter", ["minmod", "vanleer"])
@pytest.mark.parametrize("visc", [0.0, 5.0e-3])
def test_fp32_halo_tables(monkeypatch, name, limiter, visc):
    """The FP32 kernels find the sources of a block's halo once and keep them
    in LDS; their instances for meshes with wind sources ask for every cell
    anew.  A source of radius 0 covers nothing, so it only picks the instance:
    the states are the same bit for bit (neither contracts), on every kind of
    face."""
    w = dataclasses.replace(W.get(name), visc_eta=visc, limiter=limiter)
    bids = np.asarray(w.blocks(), dtype=np.int32)
    U0 = ic_in_order(w, bids)
    out = []
    for winds in ([], [(0.0, 0.0, 0.0, 0.0, 1.0, 1.0, 1.0e4, 1.0)]):
        monkeypatch.setattr(W, "wind_params", lambda w, v=winds: v)
        s = hip.Walicxe3D(w, form=hip.FUSED_FP32, bids=bids)
        assert s.cfg.nwind == len(winds)
        s.upload(U0)
        s.run(3)
        out.append((s.download(prim=False), s.time.value, s.getTimestep()))
        s.close()
    assert np.array_equal(out[0][0], out[1][0]) and out[0][1:] == out[1][1:]
