"""FP64 sweeps on meshes in, at and past the coordinate range of the shared
reciprocal (edge components 0 or in [2^-100, 2^100]): in every one the field has
the oracle's bits, on host-built and device-built tables, with fans of six, of
other lengths and of mixed ones, and with a few vertices out of range in a mesh
that is otherwise in it."""
import numpy as np
import pytest

from gproshan_amd import _lib as L
from gproshan_amd import geodesics as P
from gproshan_amd import meshgen as G

pytestmark = pytest.mark.gpu


def _scaled(e):
    x, f = G.height_field(40, 2)
    return x * 2.0 ** e, f


def _flat():
    x, f = G.height_field(40, 2)
    x[:, 2] = 0
    return np.round(x * 39), f            # fronts along edges: the conditions are 0


def _mixed():
    x, f = G.height_field(40, 2)
    x = x.copy()
    x[820, 2] += 2.0 ** 120               # edges too long, in the midst of others
    x[300, :] = x[301, :] + 2.0 ** -110   # and one component too short
    return x, f


CASES = {"unit": lambda: _scaled(0), "low": lambda: _scaled(-88), "under": lambda: _scaled(-130),
         "high": lambda: _scaled(98), "over": lambda: _scaled(140), "flat": _flat, "mixed": _mixed,
         "fans5to8": lambda: G.polar_disk(12, 8, 1), "ico": lambda: G.icosphere(3, 0.02, 1)}


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("device_setup", [False, True], ids=["host", "device"])
def test_field_has_the_oracles_bits(oracle, case, device_setup):
    xyz, f = CASES[case]()
    src = np.array([17, len(xyz) // 2], np.uint32)
    ref, nsw = oracle.Mesh(xyz, f).ptp(src, oracle.GPU_COAL)
    C = P.che(xyz, f)
    d, _, st = P.ptp(C, src, precision=L.PREC_F64, device_setup=device_setup)
    assert st["sweeps"] == nsw
    assert np.array_equal(d, ref, equal_nan=True)
    smp, _, _ = P.farthest_point_sampling_ptp_gpu(C, [17], 3)
    assert len(smp) == 3
