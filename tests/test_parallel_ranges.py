"""Host work over index ranges on several threads (gagp_amd/csrc/parallel.hpp)
touches every index once and fails as one thread would."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_ranges_cover_and_throw_the_first(tmp_path):
    exe = str(tmp_path / "parallel_ranges")
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-I" + os.path.join(ROOT, "gagp_amd", "csrc"),
                    os.path.join(ROOT, "tests", "parallel_ranges.cpp"), "-o", exe], check=True)
    assert subprocess.run([exe], check=True, capture_output=True, text=True).stdout.strip() == "0"
