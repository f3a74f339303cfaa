"""Which pushes stream through the slot array, and in which shape (csrc/stream_rule.h), on the CPU."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_what_is_accepted_fits_the_kernels_and_the_figures_of_the_rule(tmp_path):
    exe = str(tmp_path / "stream_rule_check")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-I", os.path.join(HERE, "..", "ps-lite_amd", "csrc"),
                    os.path.join(HERE, "stream_rule_check.cc"), "-o", exe], check=True)
    out = subprocess.run([exe], stdout=subprocess.PIPE, text=True, timeout=100)
    assert out.returncode == 0 and out.stdout == "ok\n", out.stdout
