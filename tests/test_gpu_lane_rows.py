"""Rows of at most 64 nodes over grammars of at most 64 expressions are varied
and lowered with one node per lane, others in memory and node by node. A
task's grammar padded past 64 expressions (test_gpu_wide_grammar) takes the
second form and draws the same, so a search must publish the same result in
both, to the last bit: at the edges of the row, for code over the straight-line
and looping limits, and for every kind of node."""
import os

import pytest

import gagp_amd
from _util import GOLDEN, strip_timing
from test_gpu_wide_grammar import padded

pytestmark = pytest.mark.gpu


def logic(grammar):
    """Conditions may be joined: and/or, whose constants the lowering adds."""
    for nt in grammar["nonterminals"]:
        if nt["type"] == "Bool":
            nt["alternatives"] += [{"id": "lane." + op, "weight": 1, "expression": {
                "signature": "%s(Bool,Bool)->Bool" % op, "args": [{"ref": nt["id"]}, {"ref": nt["id"]}]}} for op in ("and", "or")]


@pytest.mark.parametrize("task,nodes,depth", [
    ("polynomial", 63, 24), ("polynomial", 64, 40), ("polynomial", 65, 24), ("quintic", 5, 4), ("list_sum_even", 64, 13),
    ("list_sum_even", 24, 9), ("list_range_nested", 64, 12), ("list_count_gt_rev", 63, 12), ("stmt_sum_even", 64, 12),
    ("stmt_input", 64, 12), ("stmt_count_gt", 40, 12), ("let-sum", 64, 30)])
def test_lane_rows_match_rows_in_memory(task, nodes, depth, tmp_path):
    print("lane rows", task, nodes, depth, flush=True)
    results = []
    for wide in (False, True):
        out = tmp_path / str(wide)
        out.mkdir()

        def edit(grammar):
            grammar["search_limits"].update(max_nodes=nodes, max_depth=depth)
            logic(grammar)
            if not wide:
                grammar["nonterminals"].pop(next(i for i, nt in enumerate(grammar["nonterminals"]) if nt["id"] == "Pad"))
        path = padded(os.path.join(GOLDEN, "tasks", task, "task.json"), str(out), edit)
        b = gagp_amd.Batch()
        b.add(path, None, 300, 6, 3)
        b.run()
        results.append(strip_timing(b.result(0)))
    assert results[0] == results[1]
