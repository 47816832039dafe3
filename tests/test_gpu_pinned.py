"""Results where no pinned memory is to be had (hipHostMalloc refused past the
size of the schedule's records, in a process of its own): the same fields, labels
and orders by way of pageable copies."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
HERE = os.path.dirname(os.path.abspath(__file__))

PROGRAM = """
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
limit = ctypes.c_size_t.in_dll(shim, "pinned_limit")
refused = ctypes.c_size_t.in_dll(shim, "pinned_refused")
import numpy as np
from gproshan_amd import _lib as L
from gproshan_amd import geodesics as P
from gproshan_amd import meshgen as G


def results(side):
    xyz, f = G.height_field(side, 1)
    C = P.che(xyz, f)
    out = list(P.ptp(C, [5], precision=L.PREC_F64, device_setup=True)[:2])
    plan = P.Plan(C, [5, 60], precision=L.PREC_F32, clusters=True)
    plan.run()
    out += [plan.result(), plan.clusters()]
    return out


def batch():
    meshes = [P.che(*G.height_field(n, n)) for n in (20, 40)]
    b = P.Batch(meshes, [(0, 3), (1, 9), (0, 7)], block=256)
    b.run()
    return [v for q in (1, 0, 2) for v in b.result(q)]


# 2^18 values a piece: one piece, and more than two
for make in (lambda: results(100), lambda: results(730), batch):
    limit.value = 8192
    before = refused.value
    got = make()
    assert refused.value > before, "nothing was refused"
    limit.value = 2 ** 62
    want = make()
    assert len(got) == len(want)
    for a, b in zip(got, want):
        assert np.array_equal(a, b)
    print("same", flush=True)
"""


def test_results_without_pinned_memory(tmp_path):
    shim = str(tmp_path / "libpinned_limit.so")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-o", shim, os.path.join(HERE, "cpp", "pinned_limit.cpp"),
                    f"-L{rocm}/lib", "-Wl,--no-as-needed", "-lamdhip64", f"-Wl,-rpath,{rocm}/lib", "-ldl"], check=True)
    env = dict(os.environ, PYTHONPATH=os.path.dirname(HERE))
    r = subprocess.run([sys.executable, "-c", PROGRAM, shim], capture_output=True, text=True, timeout=100, env=env)
    print(r.stdout, r.stderr)
    assert r.returncode == 0 and r.stdout.count("same") == 3
