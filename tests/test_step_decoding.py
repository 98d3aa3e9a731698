"""The looping path's decoded steps on the host (CPU): tests/step_decoding.cpp
decodes seeded random programs of the list, let and statement tasks
(gagp_amd/csrc/steps.hpp, the decoder the device kernels share), runs the
steps case by case and compares value, error and remaining fuel of every case
with the C oracle VM on the bytecode -- at the task's fuel and, on a sixteenth
of the cases, at every fuel from 1 to 120, so every instruction of a joined
step is the one that runs out somewhere. Integers and error codes: equality."""
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
    exe = str(tmp_path_factory.mktemp("driver") / "step_decoding")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I" + os.path.join(ROOT, "gagp_amd", "csrc"),
                    os.path.join(ROOT, "tests", "step_decoding.cpp")] + objs +
                   [ORACLE, "-Wl,-rpath," + os.path.dirname(ORACLE), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("task", ["list-sum", "let-sum", "list_sum_even", "list_max_range", "list_count_gt_rev", "stmt_sum_even",
                                  "stmt_lowfuel", "stmt_input"])
def test_steps_match_the_bytecode(driver, task):
    out = subprocess.run([driver, os.path.join(GOLDEN, "tasks", task, "task.json"), "60"], check=True, capture_output=True, text=True)
    r = json.loads(out.stdout)
    assert r["programs"] >= 50 and r["compared"] > 10000
    assert r["mismatches"] == 0
    assert r["errors"][4] > 100  # cases that ran out inside a step
    assert r["steps"] < r["instructions"] * 3 // 5  # operand loads, stores and branches joined their operators
