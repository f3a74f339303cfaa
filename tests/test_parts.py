"""What the host makes of the words of a slice with lens (csrc/parts.h), on the CPU."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_words_are_joined_and_not_waited_for_one_by_one(tmp_path):
    exe = str(tmp_path / "parts_check")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-I", os.path.join(HERE, "..", "ps-lite_amd", "csrc"),
                    os.path.join(HERE, "parts_check.cc"), "-o", exe], check=True)
    out = subprocess.run([exe], stdout=subprocess.PIPE, text=True, timeout=100)
    assert out.returncode == 0 and out.stdout == "ok\n", out.stdout
