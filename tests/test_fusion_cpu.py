"""What a caller sees of a model that merges launches, beside one that does not (tests/fusion_check.cpp; no GPU)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe, lib = str(tmp_path_factory.mktemp("fusion") / "fusion_check"), os.path.join(ROOT, "gpreempt_amd")
    subprocess.run(["g++", "-O1", "-std=c++17", "-rdynamic", "-I" + os.path.join(ROOT, "include"), "-o", exe, os.path.join(ROOT, "tests", "fusion_check.cpp"),
                    "-L" + lib, "-lgpreempt_exec", "-lgpreempt_hip", "-Wl,-rpath," + lib, "-lpthread"], check=True)

    def run(*args):
        r = subprocess.run([exe, *args], capture_output=True, text=True, timeout=60)
        assert r.returncode == 0 and r.stdout.startswith("ok "), r.stdout + r.stderr
    return run


def test_a_layer_whose_operand_is_overwritten_later_in_the_pass_is_launched(check):
    check("writers")


def test_storages_show_what_they_would_if_every_kernel_were_launched(check):
    """values set before, between and behind the launches, and pointers handed out"""
    check("storages")


def test_a_recorded_pass_writes_every_storage(check):
    check("recorded")


def test_a_kernel_launched_again_keeps_the_form_of_its_first_launch(check):
    check("stopped")


def test_members_of_a_group_launched_alone_set_and_injected_into(check):
    check("groups")
