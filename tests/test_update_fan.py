"""The sweeps' FP64 update (one reciprocal for three quotients, certain signs)
against the reference's expressions, bit for bit, over random triangles: the
shared source compiled for the CPU."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    path = str(tmp_path_factory.mktemp("fan") / "update_fan_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-o", path,
                    os.path.join(HERE, "cpp", "update_fan_check.cpp")], check=True)
    return path


@pytest.mark.parametrize("seed", [1, 2])
def test_update_fan_has_the_references_bits(exe, seed):
    r = subprocess.run([exe, "300000", str(seed)], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0 and " 0 differ" in r.stdout
