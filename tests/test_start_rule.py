"""Which var-len requests start with one launch (csrc/start_rule.h), on the CPU."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_a_push_keeps_the_shortcut_of_the_request_that_it_repeats(tmp_path):
    exe = str(tmp_path / "start_rule_check")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-I", os.path.join(HERE, "..", "ps-lite_amd", "csrc"),
                    os.path.join(HERE, "start_rule_check.cc"), "-o", exe], check=True)
    out = subprocess.run([exe], stdout=subprocess.PIPE, text=True, timeout=100)
    assert out.returncode == 0 and out.stdout == "ok\n", out.stdout
