"""The counting sort by level at the edges of its blocks (2,048 vertices a
workgroup up to 524,288 vertices, 8,192 above): the device's rings are the
host's, and a field on them has the bits of the host-built one."""
import numpy as np
import pytest

from gproshan_amd import _lib as L
from gproshan_amd import geodesics as P
from gproshan_amd import meshgen as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [(23, 89), (32, 64), (3, 683), (17, 241), (512, 512), (449, 584), (512, 528)])
def test_rings_at_the_edges_of_blocks(rows, cols):
    mesh = P.che(*G.height_field_rect(rows, cols, 3))
    src = [0, rows * cols // 2 + 1]
    for got, ref in zip(mesh.compute_toplesets(src, gpu=True), mesh.compute_toplesets(src)):
        assert np.array_equal(got, ref)
    if rows * cols < 5000:
        a = P.ptp(mesh, src, precision=L.PREC_F64, device_setup=True)[0]
        b = P.ptp(mesh, src, precision=L.PREC_F64)[0]
        assert np.array_equal(a, b)


@pytest.mark.parametrize("rows,cols", [(512, 1024), (509, 1031), (723, 724)])
def test_rings_about_the_larger_blocks(rows, cols):
    """524,288 vertices, a few more, a few less."""
    test_rings_at_the_edges_of_blocks(rows, cols)
