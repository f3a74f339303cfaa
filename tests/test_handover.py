"""How a workgroup leaves its share to the last one of its launch (csrc/handover.h), on the CPU."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("handover") / "handover_check")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-I", os.path.join(HERE, "..", "ps-lite_amd", "csrc"),
                    os.path.join(HERE, "handover_check.cc"), "-o", exe], check=True)
    return exe


def test_every_share_is_worked_on_once(program):
    out = subprocess.run([program], stdout=subprocess.PIPE, text=True, timeout=100)
    assert out.returncode == 0 and out.stdout.startswith("ok"), out.stdout


def test_a_share_worked_on_twice_is_noticed(program):
    """The program has to find what it is there to find: a workgroup that does not ask whether its share has been taken."""
    out = subprocess.run([program, "--keep"], stdout=subprocess.PIPE, text=True, timeout=100)
    assert out.returncode == 1 and "worked on 2 times" in out.stdout, out.stdout
