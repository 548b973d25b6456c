"""foo::Model on the CPU: the host library over a device layer that counts (tests/model_check.cpp)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe, lib = str(tmp_path_factory.mktemp("model") / "model_check"), os.path.join(ROOT, "gpreempt_amd")
    subprocess.run(["g++", "-O1", "-std=c++17", "-rdynamic", "-I" + os.path.join(ROOT, "include"), "-o", exe, os.path.join(ROOT, "tests", "model_check.cpp"),
                    "-L" + lib, "-lgpreempt_exec", "-lgpreempt_hip", "-Wl,-rpath," + lib, "-lpthread"], check=True)

    def run(*args):
        r = subprocess.run([exe, *args], capture_output=True, text=True, timeout=60)
        assert r.returncode == 0 and r.stdout.startswith("ok "), r.stdout + r.stderr
    return run


def test_two_first_inputs_make_one_ring(check):
    check()


def test_sweeps_allocate_when_the_first_of_them_runs(check):
    check("sweeps")
