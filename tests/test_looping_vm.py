"""The looping path's VM on the host (CPU): tests/looping_vm.cpp compiles
vm_steps itself for one lane and compares value, error and charged fuel with
the C oracle VM on the bytecode, for seeded random programs whose steps
were packed and unpacked, with every subset
of the inputs unset, at the task's fuel and at small ones; and its division
with the host's at the edges of the 32-bit path, with the reciprocal off by
2^-23 either way. Integers and error codes: equality."""
import json
import os
import subprocess

import pytest

from _util import GOLDEN

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BUILD = os.path.join(ROOT, "gagp_amd", "_build")
ORACLE = os.path.join(ROOT, "oracle", "liboracle.so")


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    objs = [os.path.join(BUILD, n) for n in ("grammar.o", "task.o", "export.o", "identity.o")]
    missing = [p for p in objs + [ORACLE] if not os.path.exists(p)]
    assert not missing, "build the engine and the oracle first (__graft_entry__.build()): missing %s" % missing
    exe = str(tmp_path_factory.mktemp("driver") / "looping_vm")
    subprocess.run(["g++", "-O1", "-std=c++17", "-ffp-contract=off", "-D__HIPCC__", "-I" + os.path.join(ROOT, "tests", "one_lane"),
                    "-I" + os.path.join(ROOT, "gagp_amd", "csrc"), os.path.join(ROOT, "tests", "looping_vm.cpp")] + objs +
                   [ORACLE, "-Wl,-rpath," + os.path.dirname(ORACLE), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("task,n", [("stmt_input", 600), ("stmt_sum_even", 60), ("list_sum_even", 60), ("let-sum", 60)])
def test_unset_inputs_match_the_bytecode(driver, task, n):
    out = subprocess.run([driver, os.path.join(GOLDEN, "tasks", task, "task.json"), str(n)], check=True, capture_output=True, text=True)
    r = json.loads(out.stdout)
    assert r["programs"] >= 50 and r["compared"] > 10000
    assert r["errors"][0] > 1000  # cases that read an unset input
    assert r["mismatches"] == 0 and r["repacked"] == 0


def test_division_at_its_edges(driver):
    out = subprocess.run([driver, "division"], check=True, capture_output=True, text=True)
    r = json.loads(out.stdout)
    assert r["compared"] > 500000 and r["mismatches"] == 0
