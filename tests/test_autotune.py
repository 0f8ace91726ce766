"""The autotuner's search space (no GPU): launch grid, XCD ranges, curve and
z slabs per block, with slabs offered only where the kernels use them (the
FP32 MHD form without viscosity)."""
import types

from walicxe3d_amd import autotune, hip
from walicxe3d_amd import workloads as W


def fake(name, form):
    return types.SimpleNamespace(w=W.get(name), form=form)


def test_slab_choices_follow_the_kernels():
    assert autotune.slab_choices(fake("ot64", hip.FUSED_FP32)) == (1, 2, 4, 8)
    assert autotune.slab_choices(fake("briowu", hip.FUSED_FP32)) == (1, 2, 4, 8)
    assert autotune.slab_choices(fake("mhd_hlle", hip.FUSED_FP32)) == (1,)     # viscosity: whole columns
    assert autotune.slab_choices(fake("sedov", hip.FUSED_FP32)) == (1,)        # hydro kernels
    assert autotune.slab_choices(fake("ot64", hip.FUSED_FP64)) == (1,)
    assert autotune.slab_choices(fake("ot64", hip.PLAIN_FP64)) == (1,)


def test_candidates_cover_every_dimension():
    c = autotune.candidates(64, (1, 2, 4, 8))
    assert {n for *_, n in c} == {1, 2, 4, 8}
    # persistent grids only below the work-item count: 64 blocks x 8 slabs = 512 items
    assert {g for g, _, _, n in c if n == 8} == {0}
    assert {g for g, _, _, n in c if n == 1} == {0}
    c = autotune.candidates(4096, (1,))
    assert {g for g, *_ in c} == {0, 512, 1024, 2048}
    assert len(c) == 4 * 2 * 2


class Timed:
    """A solver whose steps take long for the fixed slab counts."""

    def __init__(self, name, form, nblk):
        self.w, self.form, self.nblk, self.slabs = W.get(name), form, nblk, 0

    def set_tuning(self, kind, value):
        if kind == 4:
            self.slabs = value

    def run(self, steps):
        import time
        time.sleep(steps * (2e-4 if self.slabs == 0 else 2e-3))


def test_tuning_keeps_the_choice_by_mesh_size_where_it_is_fastest():
    """A mesh whose fixed slab counts are all slower (8 viscous blocks: one
    slab 275 us a stage, the rule's 16 slabs 23) ends up with the rule, as
    before tuning; kernels without fixed counts are never given one."""
    for name, form in (("mhd_hlle", hip.FUSED_FP32), ("briowu", hip.FUSED_FP32)):
        s = Timed(name, form, 8)
        best, table = autotune.tune(s, steps=1)
        assert {r["nslab"] for r in table} == {0} | set(autotune.slab_choices(s))
        assert best["nslab"] == 0 and s.slabs == 0
    for name, form in (("sedov", hip.FUSED_FP32), ("ot64", hip.FUSED_FP64)):
        s = Timed(name, form, 8)
        _, table = autotune.tune(s, steps=1)
        assert {r["nslab"] for r in table} == {0}
