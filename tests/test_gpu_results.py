"""Fields on their way out: results are written to pinned memory in pieces of
2^18 values, eight in flight, in the caller's numbering.  Meshes of many copies
of one strip, each copy with the same source, hold the strip's own field in
every copy, so piece boundaries, a second round, unreached vertices and labels
are checked against the field of one strip alone.  The device memory kept
between calls stays bounded."""
import ctypes

import numpy as np
import pytest

from gproshan_amd import _lib as L
from gproshan_amd import geodesics as P
from gproshan_amd import meshgen as G

pytestmark = pytest.mark.gpu

PIECE, ROUND = 1 << 18, 8


def copies(xyz, f, k):
    n = len(xyz)
    off = (np.arange(k, dtype=np.uint32) * n)[:, None, None]
    return np.tile(xyz, (k, 1)), (f[None].astype(np.uint32) + off).reshape(-1, 3)


@pytest.mark.parametrize("device_setup", [False, True], ids=["host", "device"])
@pytest.mark.parametrize("n", [(64, 1), (PIECE // 64, 0), (PIECE // 64, 1), (PIECE * ROUND // 64, 1)],
                         ids=["one", "piece", "piece+1", "round+1"])
def test_result_pieces(n, device_setup):
    k = n[0] + n[1]
    xyz, f = G.height_field(8, 3)
    kw = dict(precision=L.PREC_F64, device_setup=device_setup)
    if not device_setup:
        kw["clusters"] = True
    one = P.Plan(P.che(xyz, f), [9], **kw)
    one.run()
    ref = one.result()
    X, F = copies(xyz, f, k)
    C = P.che(X, F)
    unreached = 2                                           # the last copies have no source
    src = 9 + 64 * np.arange(k - unreached, dtype=np.uint32)
    want = np.full((k, 64), np.inf)
    want[:k - unreached] = ref
    plan = P.Plan(C, src, **kw)
    plan.run()
    assert np.array_equal(plan.result().reshape(k, 64), want)
    if not device_setup:
        cl = plan.clusters().reshape(k, 64)
        assert np.array_equal(cl[:k - unreached], np.repeat(np.arange(1, k - unreached + 1)[:, None], 64, 1))
        assert np.all(cl[k - unreached:] == P.NIL)
    plan.close()


def test_memory_kept_is_bounded():
    hip = ctypes.CDLL("libamdhip64.so")
    free, total = ctypes.c_size_t(), ctypes.c_size_t()

    def used():
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return total.value - free.value

    def solve(side):
        xyz, f = G.height_field(side, 1)
        P.ptp(P.che(xyz, f), [0], precision=L.PREC_F64, device_setup=True)

    solve(64)
    before = used()
    for side in range(100, 1000, 60):
        solve(side)
    assert used() - before <= (1 << 30) + (64 << 20)


def test_memory_kept_is_bounded_while_a_mesh_lives():
    """One mesh's device tables keep the lists from being emptied.  Growing meshes
    reuse hardly any block of the one before: together they drop over 2 GiB (more than 250
    bytes a vertex in FP64), of which 1 GiB may stay.  Blocks take up to 2 MiB
    more than asked for, at most a few dozen of them are kept: 128 MiB."""
    hip = ctypes.CDLL("libamdhip64.so")
    free, total = ctypes.c_size_t(), ctypes.c_size_t()

    def used():
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return total.value - free.value

    def solve(side):
        xyz, f = G.height_field(side, 1)
        P.ptp(P.che(xyz, f), [0], precision=L.PREC_F64, device_setup=True)

    solve(64)
    gone = used()
    hold = P.che(*G.height_field(8, 1))
    P.ptp(hold, [0], precision=L.PREC_F64, device_setup=True)
    before = used()
    sides = range(300, 1400, 90)
    assert 250 * sum(s * s for s in sides) > 2 << 30
    most = 0
    for side in sides:
        solve(side)
        most = max(most, used() - before)
    assert (1 << 29) < most <= (1 << 30) + (128 << 20), most
    del hold
    assert used() - gone <= 8 << 20
