"""A search prepares the looping path when its grammar's programs may leave the
straight-line one (CPU): no program may be lowered to a path the search does
not have. Grammars with branches and loops, with len and index as their only
list operations, and straight-line ones at and past the limits of rows and depth."""
import json
import os
import subprocess

import pytest

from _util import GOLDEN
from gagp_amd import workloads

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BUILD = os.path.join(ROOT, "gagp_amd", "_build")


def reads_only(max_nodes=31, max_depth=9):
    """Arithmetic over the length and the elements of a list: no jumps."""
    ref = {"ref": "Read.Int"}
    alternatives = [("len", workloads._op("len(IntList)->Int", {"input": "xs"})),
                    ("at", workloads._op("index(IntList,Int)->Int", {"input": "xs"}, ref)),
                    ("clamped", workloads._op("index_clamped_or_zero(IntList,Int)->Int", {"input": "xs"}, ref)),
                    ("const", workloads._const([0, 1, 2, -1])),
                    ("add", workloads._op("add(Int,Int)->Int", ref, ref)), ("sub", workloads._op("sub(Int,Int)->Int", ref, ref))]
    return {"format_version": "grammar-definition-v2", "entry": {"nonterminal": "Read.Int", "type": "Int"},
            "inputs": [{"name": "xs", "type": "IntList"}], "search_limits": {"max_nodes": max_nodes, "max_depth": max_depth},
            "execution_limits": {"fuel": 1000}, "nonterminals": [{"id": "Read.Int", "type": "Int", "scope": [], "alternatives": [
                {"id": name, "weight": 1, "expression": e} for name, e in alternatives]}]}


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    objs = [os.path.join(BUILD, n) for n in ("grammar.o", "task.o", "identity.o")]
    missing = [p for p in objs if not os.path.exists(p)]
    assert not missing, "build the engine first (__graft_entry__.build()): missing %s" % missing
    exe = str(tmp_path_factory.mktemp("driver") / "looping_grammar")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I" + os.path.join(ROOT, "gagp_amd", "csrc"),
                    os.path.join(ROOT, "tests", "looping_grammar.cpp")] + objs + ["-o", exe], check=True)
    return exe


def ask(driver, task):
    return json.loads(subprocess.run([driver, task, "60"], check=True, capture_output=True, text=True).stdout)


@pytest.mark.parametrize("task", ["list_sum_even", "stmt_sum_even", "let-sum", "list_count_gt_rev"])
def test_loops_and_branches_are_known(driver, task):
    r = ask(driver, os.path.join(GOLDEN, "tasks", task, "task.json"))
    assert r["looping"] > 0 and r["leaves"]


def test_list_reads_without_a_jump_are_known(driver, tmp_path):
    cases = json.load(open(os.path.join(GOLDEN, "tasks", "list_sum_even", "train.cases.json")))["cases"]
    r = ask(driver, workloads.write_task(str(tmp_path), "reads", reads_only(), cases, cases))
    assert r["looping"] > 10 and r["leaves"]


@pytest.mark.parametrize("nodes,depth", [(63, 12), (126, 17), (131, 17), (132, 17), (400, 17), (60, 18), (60, 19), (120, 30)])
def test_straight_line_limits_are_known(driver, nodes, depth, tmp_path):
    grammar = workloads.polynomial_grammar(range(10), nodes, depth)
    cases = [workloads._int_case(x, x) for x in range(3)]
    r = ask(driver, workloads.write_task(str(tmp_path), "line", grammar, cases, cases))
    assert r["lowered"] > 10
    assert r["leaves"] or not r["looping"]
