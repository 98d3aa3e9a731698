"""Grammars with more than 64 expressions take the general derivation (the
lane-register form holds one expression per lane). An unreachable nonterminal
of 70 constants widens a task's grammar past that without touching any draw,
so the search must publish the reference's golden result of the narrow task,
and stepping both from one seed must agree for a constant range of 2^20 and
more values, which only the general form draws."""
import json
import os

import pytest

import gagp_amd
from _util import GOLDEN, strip_timing

pytestmark = pytest.mark.gpu
MANIFEST = json.load(open(os.path.join(GOLDEN, "runs", "manifest.json")))


def padded(task, out, edit=None):
    doc = json.load(open(task))
    base = os.path.dirname(task)
    grammar = json.load(open(os.path.join(base, doc["grammar"])))
    grammar["nonterminals"].append({"id": "Pad", "type": "Int", "scope": [], "alternatives": [
        {"id": "p%d" % k, "weight": 1, "expression": {"constant": {"type": "Int", "values": [str(k)]}}} for k in range(70)]})
    if edit:
        edit(grammar)
    with open(os.path.join(out, "grammar.json"), "w") as f:
        json.dump(grammar, f)
    doc.update(grammar="grammar.json", train=os.path.join(base, doc["train"]), test=os.path.join(base, doc["test"]))
    with open(os.path.join(out, "task.json"), "w") as f:
        json.dump(doc, f)
    return os.path.join(out, "task.json")


@pytest.mark.parametrize("name", ["polynomial_p512_g32_s7", "list_sum_even_p512_g10_s5", "stmt_sum_even_p512_g10_s5",
                                  "quintic_wide_p512_g16_s5"])
def test_wide_grammar_matches_the_narrow_golden(name, tmp_path):
    m = MANIFEST[name]
    task = padded(os.path.join(GOLDEN, m["task"]), str(tmp_path))
    b = gagp_amd.Batch()
    b.add(task, None, m["population"], m["generations"], m["seed"])
    b.run()
    want = strip_timing(json.load(open(os.path.join(GOLDEN, "runs", name, "result.json"))))
    assert strip_timing(b.result(0)) == want


@pytest.mark.parametrize("top", [2 ** 20 - 2, 2 ** 20 - 1, 2 ** 40])
def test_constant_ranges_draw_alike_in_both_forms(top, tmp_path):
    # The narrow grammar draws small ranges in lane registers and leaves 2^20
    # values or more to the general form; the padded one always takes the latter.
    def ranged(grammar):
        for a in grammar["nonterminals"][0]["alternatives"]:
            if a["id"] == "small":
                a["expression"] = {"constant": {"type": "Int", "range": ["-1", str(top - 1)]}}
    results = []
    for pad in (False, True):
        out = tmp_path / str(pad)
        out.mkdir()

        def edit(grammar):
            ranged(grammar)
            if not pad:
                grammar["nonterminals"].pop()
        task = padded(os.path.join(GOLDEN, "tasks", "polynomial", "task.json"), str(out), edit)
        b = gagp_amd.Batch()
        b.add(task, None, 300, 6, 3)
        b.run()
        results.append(strip_timing(b.result(0)))
    assert results[0] == results[1]
