"""The deal of the W4A16 grouped GEMMs' row tiles to workgroups and XCDs
(csrc/gemm_items.hpp), checked on the host by a small C++ program built here
with g++ (tests/cpp/gemm_items_check.cpp)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "moe-ascend-opt_amd", "csrc")


def test_every_block_once_and_no_xcd_overloaded(tmp_path):
    exe = str(tmp_path / "gemm_items_check")
    build = subprocess.run(["g++", "-O2", "-std=c++17", f"-I{CSRC}", os.path.join(HERE, "cpp", "gemm_items_check.cpp"),
                            "-o", exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert build.returncode == 0, build.stdout
    run = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert run.returncode == 0 and run.stdout.strip() == "ok", run.stdout
