"""Downloads large enough for the threaded path give what the upload brought:
sizes around its limit, odd chunk counts, two threads at once (one of them
takes the runtime's path), and a context made after the last one gave the
buffers back."""
import dataclasses
import threading

import numpy as np
import pytest

from walicxe3d_amd import hip
from walicxe3d_amd import workloads as W

pytestmark = pytest.mark.gpu


def _state(nroot, seed):
    w = dataclasses.replace(W.get("sedov"), nroot=nroot, maxlev=1, base_level=1, phys=tuple(float(n) for n in nroot))
    rng = np.random.default_rng(seed)
    n = nroot[0] * nroot[1] * nroot[2]
    U = rng.uniform(0.5, 1.0, (n, 5, 16, 16, 16))
    U[:, 4] += 10.0
    return w, U


# 163840 bytes a block: 25 blocks below the limit of 4 MB, 26 above; chunks of
# 1, 2 and 4 MB with remainders
@pytest.mark.parametrize("nroot", [(25, 1, 1), (26, 1, 1), (13, 7, 1), (19, 11, 1), (17, 10, 10)])
@pytest.mark.parametrize("form", [hip.PLAIN_FP64, hip.FUSED_FP32])
def test_download_returns_the_upload(nroot, form):
    w, U = _state(nroot, 3)
    s = hip.Walicxe3D(w, form=form)
    s.upload(U)
    order = np.argsort(np.asarray(w.blocks()))   # identity here: one level, block IDs ascending
    assert np.array_equal(order, np.arange(len(U)))
    u, p = s.download()
    assert np.array_equal(u, U)
    assert np.array_equal(p[:, 0], U[:, 0])
    s.close()


def test_two_threads_and_a_new_context():
    states = [_state((20, 5, 1), 4), _state((10, 10, 2), 5)]
    sims = [hip.Walicxe3D(w, form=hip.FUSED_FP32) for w, _ in states]
    for s, (_, U) in zip(sims, states):
        s.upload(U)
    bad = []

    def loop(n):
        for _ in range(10):
            if not np.array_equal(sims[n].download(prim=False), states[n][1]):
                bad.append(n)

    th = [threading.Thread(target=loop, args=(n,)) for n in (0, 1)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad
    for s in sims:
        s.close()
    w, U = states[0]
    s = hip.Walicxe3D(w, form=hip.PLAIN_FP64)
    s.upload(U)
    assert np.array_equal(s.download(prim=False), U)
    assert np.array_equal(s.raw(0)[:, :, 2:18, 2:18, 2:18], U)
    s.close()


def test_download_into_pinned_memory():
    """Memory that the caller pinned takes the state directly (no chunks), at a
    size that ordinary memory takes in chunks; also from its middle on."""
    import ctypes as C
    w, U = _state((13, 7, 1), 6)
    s = hip.Walicxe3D(w, form=hip.FUSED_FP32)
    s.upload(U)
    L = hip.load()
    base = C.c_void_p()
    assert L.hipHostMalloc(C.byref(base), C.c_size_t(U.nbytes + 24), C.c_uint(0)) == 0   # of the runtime it links
    pin = np.ctypeslib.as_array(C.cast(base, hip._dp), (U.size + 3,))
    for off in (0, 3):
        pin[:] = 0.0
        at = C.cast(base.value + 8 * off, hip._dp)
        assert L.wx_download_state(s._h, at, None, hip.LAYOUT_BLOCKS, 0, None) == 0
        assert np.array_equal(pin[off:off + U.size].reshape(U.shape), U) and not pin[:off].any()
    s.close()
    assert L.hipHostFree(base) == 0
