"""Tables that grow together when a launch fails (csrc/growths.h), on the CPU."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("growths") / "growths_check")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-I", os.path.join(HERE, "..", "ps-lite_amd", "csrc"),
                    os.path.join(HERE, "growths_check.cc"), "-o", exe], check=True)
    return exe


def test_a_table_keeps_the_array_that_has_its_keys(program):
    out = subprocess.run([program], stdout=subprocess.PIPE, text=True, timeout=100)
    assert out.returncode == 0 and out.stdout == "ok\n", out.stdout


def test_a_table_without_its_keys_is_noticed(program):
    """The program has to find what it is there to find: a table that keeps an array that nothing was moved to."""
    out = subprocess.run([program, "--forget"], stdout=subprocess.PIPE, text=True, timeout=100)
    assert out.returncode == 1 and "no keys" in out.stdout, out.stdout
