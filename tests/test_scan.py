"""What the wavefronts of the var-len kernels do to each other between barriers (csrc/scan.h, csrc/table_kernels.h), on
the CPU: the kernels are compiled against a stand-in that runs them wavefront by wavefront, in every order."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)
CLANG = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "clang++")


@pytest.mark.skipif(not os.path.exists(CLANG), reason="needs the compiler that builds the kernels")
def test_offsets_whichever_wavefront_is_ahead(tmp_path):
    exe = str(tmp_path / "scan_check")
    subprocess.run([CLANG, "-std=c++17", "-O1", "-fno-strict-aliasing", "-I", os.path.join(HERE, "include", "host_wave"),
                    "-I", os.path.join(REPO, "include"), "-I", os.path.join(REPO, "ps-lite_amd", "csrc"),
                    os.path.join(HERE, "scan_check.cc"), "-o", exe], check=True)
    out = subprocess.run([exe], stdout=subprocess.PIPE, text=True, timeout=100)
    assert out.returncode == 0 and out.stdout == "ok\n", out.stdout
