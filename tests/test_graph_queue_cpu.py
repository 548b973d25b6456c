"""The host loop that queues the graph workloads' iterations, on the CPU: host/graphcompute.cpp compiled against a device
made of threads (tests/graph_queue_check.cpp)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("queue") / "graph_queue_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(ROOT, "gpreempt_amd", "host"), "-o", exe,
                    os.path.join(ROOT, "tests", "graph_queue_check.cpp"), os.path.join(ROOT, "gpreempt_amd", "host", "graphcompute.cpp"), "-lpthread"], check=True)

    def run(what):
        r = subprocess.run([exe, what], capture_output=True, text=True, timeout=100)
        assert r.returncode == 0 and r.stdout.startswith("ok "), r.stdout[-2000:] + r.stderr[-2000:]
    return run


def test_a_run_leaves_nothing_in_its_stream(check):
    check("blocking")


def test_a_long_run_keeps_nothing_per_launch(check):
    check("memory")


def test_a_stop_waits_for_few_launches(check):
    check("stops")


def test_what_connected_components_clears(check):
    check("clears")
