"""How far the row kernels read in a request's values (csrc/quads.h), on the CPU."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("quads") / "quads_check")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-I", os.path.join(HERE, "..", "ps-lite_amd", "csrc"),
                    os.path.join(HERE, "quads_check.cc"), "-o", exe], check=True)
    return exe


def test_nothing_is_read_past_the_values(program):
    out = subprocess.run([program], stdout=subprocess.PIPE, text=True, timeout=100)
    assert out.returncode == 0 and out.stdout == "ok\n", out.stdout


def test_a_read_past_the_values_is_noticed(program):
    """The program has to find what it is there to find: a row that follows may be shorter than what a quad is short of."""
    out = subprocess.run([program, "--any-row"], stdout=subprocess.PIPE, text=True, timeout=100)
    assert out.returncode == 1 and "of 2 (k 1, n 2)" in out.stdout, out.stdout
