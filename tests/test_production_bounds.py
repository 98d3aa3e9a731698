"""The bounds by which a derivation on the device chooses among all of a
nonterminal's productions (gagp_amd/csrc/grammar.cpp: production_bounds) give
the production the in-order scan of the rounded weights does: equality, on the
host, for random weights and for choices at and around every bound."""
import json
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BUILD = os.path.join(ROOT, "gagp_amd", "_build")


def test_bounds_choose_as_the_scan_does(tmp_path):
    objs = [os.path.join(BUILD, n) for n in ("grammar.o", "identity.o")]
    missing = [p for p in objs if not os.path.exists(p)]
    assert not missing, "build the engine first (__graft_entry__.build()): missing %s" % missing
    exe = str(tmp_path / "production_bounds")
    subprocess.run(["g++", "-O1", "-std=c++17", "-ffp-contract=off", "-I" + os.path.join(ROOT, "gagp_amd", "csrc"),
                    os.path.join(ROOT, "tests", "production_bounds.cpp")] + objs + ["-o", exe], check=True)
    r = json.loads(subprocess.run([exe], check=True, capture_output=True, text=True).stdout)
    assert r["compared"] > 500000
    assert r["wrong"] == 0
