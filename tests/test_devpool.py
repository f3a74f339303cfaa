"""The lists of device arrays (csrc/devpool.hip), on the CPU: the file is compiled against a stand-in for the runtime."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("devpool") / "devpool_check")
    csrc = os.path.join(REPO, "ps-lite_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-Wall", "-pthread", "-I", os.path.join(HERE, "include", "host_hip"),
                    "-I", os.path.join(REPO, "include"), "-I", csrc, os.path.join(HERE, "devpool_check.cc"), "-x", "c++",
                    os.path.join(csrc, "devpool.hip"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("what", ["settle", "linger", "bound", "unkept"])
def test_arrays_change_hands_and_go_back(program, what):
    env = dict(os.environ)
    env.pop("PSKV_NO_ASYNC_ALLOC", None)
    if what == "unkept":
        env["PSKV_NO_ASYNC_ALLOC"] = "1"
    out = subprocess.run([program, what], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60, env=env)
    assert out.returncode == 0 and out.stdout.endswith("ok\n"), out.stdout
