"""The memory kept between calls, its source compiled for the CPU on a stand-in of
the HIP runtime: the bounds with a mesh alive, the order in which blocks go back,
and failed allocations."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    path = str(tmp_path_factory.mktemp("pool") / "pool_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(HERE, "cpp", "fake_hip"), "-o", path,
                    os.path.join(HERE, "cpp", "pool_check.cpp")], check=True)
    return path


@pytest.mark.parametrize("what", ["device_bound", "pinned_bound", "device_fails", "pinned_fails"])
def test_pool(exe, what):
    r = subprocess.run([exe, what], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
