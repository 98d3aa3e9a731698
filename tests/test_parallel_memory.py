"""Memory that runs out while host ranges are put on threads
(gagp_amd/csrc/parallel.hpp) is an error of the call, or none: the ranges no
thread was started for run on the caller's. It never ends the process."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_no_allocation_ends_the_process(tmp_path):
    exe = str(tmp_path / "parallel_memory")
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-I" + os.path.join(ROOT, "gagp_amd", "csrc"),
                    os.path.join(ROOT, "tests", "parallel_memory.cpp"), "-o", exe], check=True)
    run = subprocess.run([exe], capture_output=True, text=True)
    assert run.returncode == 0, run.stderr
    wrong, threw, covered = map(int, run.stdout.split())
    assert wrong == 0 and threw > 0 and covered > 0
