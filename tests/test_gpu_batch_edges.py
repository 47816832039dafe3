"""Batched fields where their BFS and their read-back change course: meshes to
262,144 vertices keep the visited bits in LDS, larger ones take the ordered BFS;
frontiers past 1,024 vertices are read back from memory; links past eight go on
in the fan table.  Each field equals the single-field solve bit for bit, in
whatever order the fields are read."""
import numpy as np
import pytest

from gproshan_amd import _lib as L
from gproshan_amd import geodesics as P
from gproshan_amd import meshgen as G

pytestmark = pytest.mark.gpu


def check(raw, jobs, block, order):
    meshes = [P.che(*r) for r in raw]
    b = P.Batch(meshes, jobs, block=block)
    for _ in range(2):
        b.run()
        for q in order:
            m, s = jobs[q]
            d, sw = b.result(q)
            ref, _, st = P.ptp(meshes[m], [s], precision=L.PREC_F32, fp32_geometry=L.GEO_FP32)
            assert sw == st["sweeps"], (q, jobs[q])
            assert np.array_equal(d, ref), (q, jobs[q])
    b.close()


@pytest.mark.parametrize("block", [256, 1024])
def test_small_and_long_links(block):
    raw = [(np.eye(3), np.array([[0, 1, 2]], np.uint32)), G.polar_disk(12, 9, 1), G.polar_disk(4, 65, 2),
           G.polar_disk(3, 1000, 3), G.icosphere(3, 0.01, 0)]
    jobs = [(0, 2), (1, 0), (1, 60), (2, 0), (2, 200), (3, 0), (3, 5), (3, 2500), (4, 100)]
    check(raw, jobs, block, [0, 1, 2, 3, 4, 5, 6, 7, 8, 8, 3, 0, 6])


@pytest.mark.parametrize("rows,cols", [(512, 512), (512, 513)], ids=["bits", "ordered"])
def test_wide_rings(rows, cols):
    """Rings of 1,500 vertices; fields longer than half the read-back window."""
    mid = rows // 2 * cols + cols // 2
    check([G.height_field_rect(rows, cols, 5), G.icosphere(4, 0.01, 1)], [(0, mid), (0, 3), (1, 9), (0, mid + 77)],
          1024, [3, 0, 1, 2, 3])
