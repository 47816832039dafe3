"""FP32 plans replay graphs from their second run on, their first is launched on the
stream: results, labels, traces and counts of replayed runs against the first run's
and against a plan that is always launched, bit for bit, for every kind of plan
that can replay, windows of one chunk and of hundreds, and changed launch shapes."""
import numpy as np
import pytest

from gproshan_amd import _lib as L
from gproshan_amd import geodesics as P
from gproshan_amd import meshgen as G

pytestmark = pytest.mark.gpu

MESHES = {
    "hf": (lambda: G.height_field_rect(150, 131, 3), [7000, 40]),
    "ico": (lambda: G.icosphere(3, 0.01, 0), [9]),
    "disk24": (lambda: G.polar_disk(40, 24, 4), [500]),            # a fan past the register-held slots
    "grid": (lambda: G.anisotropic_grid(96), [96 * 48 + 48]),      # flagged triangles
    "hf512": (lambda: G.height_field(512, 5), [512 * 256 + 256]),
}
PLANS = {
    "rings": dict(),
    "plain": dict(coalesce=False),
    "device": dict(device_setup=True),
    "labels": dict(clusters=True),
    "labels_plain": dict(clusters=True, coalesce=False),
    "geo64": dict(fp32_geometry=L.GEO_FP64),
    "geo32": dict(fp32_geometry=L.GEO_FP32),
    "last_read": dict(result_buffer=L.RESULT_LAST_READ),
    "uncapped": dict(uncapped=True, tol=1e-6),
    "cut": dict(max_sweeps=11),
    "bands": dict(schedule=L.SCHED_EUCLID_BAND, band_width=0.5, tol=1e-6),
    "ring_bands": dict(schedule=L.SCHED_RING_BAND, tol=1e-6),
}
CASES = [(m, k) for m in ("hf", "ico") for k in PLANS] + [
    ("disk24", "rings"), ("disk24", "labels"), ("grid", "rings"), ("grid", "labels"), ("grid", "geo64"),
    ("hf512", "device"), ("hf512", "uncapped"), ("hf512", "bands")]


def _outputs(plan, kw):
    st = plan.run()
    out = [plan.result(), plan.trace()]
    if kw.get("clusters"):
        out.append(plan.clusters())
    return out, {k: st[k] for k in ("sweeps", "relaxations", "cond_checks", "f64_updates", "precision", "capped",
                                    "kernel", "check_sweeps")}


def _same(a, b):
    assert a[1] == b[1]
    for x, y in zip(a[0], b[0]):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("mesh,kind", CASES, ids=[f"{m}-{k}" for m, k in CASES])
def test_replayed_runs(mesh, kind):
    gen, src = MESHES[mesh]
    C, kw = P.che(*gen()), PLANS[kind]
    launched = P.Plan(C, src, launch_mode=L.LAUNCH_STREAM, **kw)
    want = _outputs(launched, kw)
    plan = P.Plan(C, src, **kw)
    for _ in range(4):                       # launched, then replayed three times
        _same(_outputs(plan, kw), want)
        _same(_outputs(launched, kw), want)  # other work between the replays
    plan.close()
    launched.close()


@pytest.mark.parametrize("kind", ["device", "labels", "bands"])
def test_replayed_runs_of_another_shape(kind):
    """After autotune: other grids and other numbers of sweeps a graph."""
    gen, src = MESHES["hf"]
    C, kw = P.che(*gen()), PLANS[kind]
    launched = P.Plan(C, src, launch_mode=L.LAUNCH_STREAM, **kw)
    want = _outputs(launched, kw)
    for warm in (0, 2):                      # tuned before its first run; with graphs of the old shape
        plan = P.Plan(C, src, **kw)
        for _ in range(warm):
            plan.run()
        plan.autotune()
        for _ in range(3):
            _same(_outputs(plan, kw), want)
        plan.close()
    for grid in (8, 40, 1000):
        plan = P.Plan(C, src, grid=grid, **kw)
        for _ in range(3):
            _same(_outputs(plan, kw), want)
        plan.close()
    launched.close()
