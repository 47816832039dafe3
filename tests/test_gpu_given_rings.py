"""The ring drivers on rings of the caller's own making, plain and coalesced,
against the oracle's drivers on the same rings, bit for bit: rings that are
swept from device-built tables and rings that are laid out on the host (partial
ones, a vertex listed twice, a long fan, a mesh that is not manifold)."""
import numpy as np
import pytest

from gproshan_amd import _lib as L
from gproshan_amd import geodesics as P
from gproshan_amd import meshgen as G

pytestmark = pytest.mark.gpu


def _bfs(M, src):
    _, srt, lim = M.toplesets(np.array(src, np.uint32))
    return np.array(srt, np.uint32), np.array(lim, np.uint32)


def _as_is(srt, lim):
    return srt, lim


def _shuffled(srt, lim):
    rng = np.random.default_rng(1)
    return np.concatenate([rng.permutation(srt[a:b]) for a, b in zip(lim[:-1], lim[1:])]), lim


def _empty_rings(srt, lim):
    return srt, np.concatenate([lim[:3], lim[2:3], lim[3:], lim[-1:], lim[-1:]])


def _merged(srt, lim):
    return srt, np.unique(np.append(lim[::3], lim[-1]))


def _cut(srt, lim):
    return srt, lim[:len(lim) // 2]


def _twice(srt, lim):
    srt = srt.copy()
    srt[lim[3]] = srt[lim[3] + 1]
    return srt, lim


def _parts():
    x, f = G.height_field(21, 2)
    y, g = G.icosphere(2, 0.02, 1)
    return np.vstack([x, y + 5.0]), np.vstack([f, g + len(x)]).astype(np.uint32)


def _bowtie_strip():
    x, f = G.height_field(12, 2)
    return np.vstack([x, [[-1, 0, 0.5], [-1, 1, 0.5]]]), np.vstack([f, [[0, 144, 145]]]).astype(np.uint32)


MESHES = {
    "hf": (lambda: G.height_field_rect(37, 53, 3), [700, 5, 1900]),
    "ico": (lambda: G.icosphere(3, 0.01, 0), [9]),
    "parts": (_parts, [40, 300]),          # the second part is in no ring
    "hub40": (lambda: G.polar_disk(9, 40, 1), [70]),
    "bowtie": (_bowtie_strip, [60]),
}
RINGS = [_as_is, _shuffled, _empty_rings, _merged, _cut, _twice]
CASES = [(m, r) for m in ("hf", "ico", "parts") for r in RINGS] + [("hub40", _as_is), ("bowtie", _as_is)]


@pytest.mark.parametrize("mesh,rings", CASES, ids=[f"{m}{r.__name__}" for m, r in CASES])
def test_rings_of_the_callers(oracle, mesh, rings):
    gen, src = MESHES[mesh]
    xyz, f = gen()
    M, C = oracle.Mesh(xyz, f), P.che(xyz, f)
    srt, lim = rings(*_bfs(M, src))
    ts = (None, np.ascontiguousarray(srt), np.ascontiguousarray(lim, np.uint32))
    forms = [(P.parallel_toplesets_propagation_gpu, oracle.GPU_PLAIN)]
    if rings is not _twice:                # renumbering needs each vertex once
        forms.append((P.parallel_toplesets_propagation_coalescence_gpu, oracle.GPU_COAL))
    for drv, variant in forms:
        ref, _ = M.ptp(src, variant, toplesets=ts)
        d, _ = drv(C, src, ts)
        assert np.array_equal(d, ref)
        d, _, cl = drv(C, src, ts, clusters=True)
        assert np.array_equal(d, ref)
        if rings in (_as_is, _shuffled):
            _, cref, _ = M.ptp_clusters(src, variant)
            assert np.array_equal(cl, cref)


def test_labels_follow_the_sources_given():
    """Sources out of order, in one ring with other vertices, one twice."""
    xyz, f = G.height_field_rect(40, 30, 3)
    C = P.che(xyz, f)
    src = np.array([900, 17, 400], np.uint32)
    ts = C.compute_toplesets(src)
    _, _, ref = P.parallel_toplesets_propagation_gpu(C, src, ts, clusters=True)
    for order in ([2, 0, 1], [1, 2, 0]):
        _, _, cl = P.parallel_toplesets_propagation_gpu(C, src[order], ts, clusters=True)
        assert np.array_equal(src[order][cl - 1], src[ref - 1])
    d0, _ = P.parallel_toplesets_propagation_gpu(C, src, ts)
    d1, _ = P.parallel_toplesets_propagation_gpu(C, np.append(src, src[:1]), ts)
    assert np.array_equal(d0, d1)
    with pytest.raises(L.GPError):
        P.parallel_toplesets_propagation_coalescence_gpu(C, [5000], ts)
