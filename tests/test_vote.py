"""The agreement between the workgroups of one launch (csrc/vote.h), on the CPU."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("vote") / "vote_check")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-I", os.path.join(HERE, "..", "ps-lite_amd", "csrc"),
                    os.path.join(HERE, "vote_check.cc"), "-o", exe], check=True)
    return exe


def test_all_workgroups_go_on_or_none(program):
    out = subprocess.run([program], stdout=subprocess.PIPE, text=True, timeout=100)
    assert out.returncode == 0 and out.stdout.startswith("ok"), out.stdout


def test_a_workgroup_that_leaves_unmarked_is_noticed(program):
    """The program has to find what it is there to find: a workgroup that gives up and tells nobody."""
    out = subprocess.run([program, "--leave-unmarked"], stdout=subprocess.PIPE, text=True, timeout=100)
    assert out.returncode == 1 and "workgroups go on" in out.stdout, out.stdout
