"""Which stream a slice takes (csrc/stream_choice.h), on the CPU."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_calls_of_any_size_stay_on_a_quiet_gpu_and_find_the_free_stream_of_a_busy_one(tmp_path):
    exe = str(tmp_path / "stream_choice_check")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-I", os.path.join(HERE, "..", "ps-lite_amd", "csrc"),
                    os.path.join(HERE, "stream_choice_check.cc"), "-o", exe], check=True)
    out = subprocess.run([exe], stdout=subprocess.PIPE, text=True, timeout=100)
    assert out.returncode == 0 and out.stdout == "ok\n", out.stdout
