"""Model::set from several threads before any input has been set (tests/first_input_check.cpp over the host library)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_two_first_inputs_make_one_ring(tmp_path):
    exe, lib = str(tmp_path / "first_input_check"), os.path.join(ROOT, "gpreempt_amd")
    subprocess.run(["g++", "-O1", "-std=c++17", "-rdynamic", "-I" + os.path.join(ROOT, "include"), "-o", exe, os.path.join(ROOT, "tests", "first_input_check.cpp"),
                    "-L" + lib, "-lgpreempt_exec", "-lgpreempt_hip", "-Wl,-rpath," + lib, "-lpthread"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.startswith("ok "), r.stdout + r.stderr
