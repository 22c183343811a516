"""CPU: the rounding bound that widens the raytracer's bins holds for poses whose
linear part makes rays longer or shorter than 1 (tests/hit_rounding_check.cc, compiled
here with g++ and the kernels' own header ugu_amd/csrc/rt_math.h)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("hit") / "hit_rounding_check")
    subprocess.run(["g++", "-O2", "-std=gnu++17", "-ffp-contract=off", "-o", exe,
                    os.path.join(ROOT, "tests", "hit_rounding_check.cc")], check=True)
    return exe


@pytest.mark.parametrize("scale", [1.0, 0.01, 30.0, 570.0])
@pytest.mark.parametrize("shear", [0.0, 0.5])
def test_bound_holds(check, scale, shear):
    r = subprocess.run([check, "1", "200000", str(scale), str(shear)], capture_output=True,
                       text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
